"""The C-ABI library: it loads, exports every symbol include/tyr_hip.h declares, and its host-side
validation rejects bad arguments before touching a GPU (so these run without one)."""
import ctypes
import os
import re
import subprocess
import sys

import pytest

from tyr_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_symbols():
    text = open(os.path.join(ROOT, "include", "tyr_hip.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(tyr_hip_[a-z0-9_]+)\s*\(", text)))


def test_header_and_binding_agree():
    assert declared_symbols() == sorted(_lib.SYMBOLS)


def test_library_exports_every_declared_symbol():
    L = ctypes.CDLL(_lib.LIB_PATH)
    for name in declared_symbols():
        assert hasattr(L, name), name


def test_strerror_and_version():
    L = _lib.load()
    assert L.tyr_hip_version() >= 100
    assert L.tyr_hip_strerror(0) == b"ok"
    for code in range(-8, 0):
        assert L.tyr_hip_strerror(code) not in (b"", b"unknown tyr_hip status")
    assert b"CUDA tensor" in L.tyr_hip_strerror(-8)      # the reference launcher's wording
    assert L.tyr_hip_strerror(-99) == b"unknown tyr_hip status"


def test_host_validation_needs_no_gpu():
    L = _lib.load()
    p = 0x1000  # never dereferenced: every call below must fail validation first
    OK, NULL, SHAPE, UNSUP, MISAL, WS = 0, -1, -2, -3, -4, -5
    assert L.tyr_hip_gemm_bf16(None, p, p, 8, 8, 8, 0, None) == NULL
    assert L.tyr_hip_gemm_bf16(p, p, p, 0, 8, 8, 0, None) == SHAPE
    assert L.tyr_hip_gemm_bf16(p, p, p, 8, 8, 12, 0, None) == UNSUP
    assert L.tyr_hip_gemm_bf16(p + 2, p, p, 8, 8, 8, 0, None) == MISAL
    assert L.tyr_hip_gemm_bf16(p, p, p, 2 ** 40, 8, 8, 0, None) == SHAPE
    assert L.tyr_hip_gemm_bf16_batched(p, p, p, 0, 8, 8, 8, 64, 64, 64, 0, None) == SHAPE
    assert L.tyr_hip_gemm_bf16_batched(p, p, p, 2, 8, 8, 8, 64, 64, 32, 0, None) == SHAPE      # outputs would overlap
    assert L.tyr_hip_gemm_bf16_batched(p, p, p, 2, 8, 8, 8, 68, 64, 64, 0, None) == MISAL
    assert L.tyr_hip_gemm_bf16_batched(p, p, p, 70000, 8, 8, 8, 64, 64, 64, 0, None) == SHAPE
    prev = L.tyr_hip_gemm_force_general(1)
    assert L.tyr_hip_gemm_force_general(prev) == 1 and L.tyr_hip_gemm_force_general(prev) == prev
    prev = L.tyr_hip_flash_attn_fwd_persistent(1)
    assert L.tyr_hip_flash_attn_fwd_persistent(prev) == 1 and L.tyr_hip_flash_attn_fwd_persistent(prev) == prev
    # the calibration loop writes 256 floats per workgroup: a smaller sink is refused before any launch
    assert L.tyr_hip_mfma_sustain(p, 1 << 20, 0, 256, 10, p, 256 * 256 * 4 - 1, None, None) == WS
    assert L.tyr_hip_gemm_fp8(p, p, None, 16, 16, 16, 1.0, 1.0, 0, None) == NULL
    assert L.tyr_hip_gemm_fp8(p, p, p, 16, 8, 16, 1.0, 1.0, 0, None) == UNSUP
    assert L.tyr_hip_gemm_fp8_ex(p, p, p, 16, 16, 16, 1.0, None, None, 7, 0, None) == UNSUP           # unknown output type
    assert L.tyr_hip_gemm_fp8_ex(p, p, p, 16, 16, 16, 1.0, None, p + 4, 1, 0, None) == MISAL          # column scales: 16-byte rows
    assert L.tyr_hip_flash_attn_fwd(p, p, None, p, None, 1, 1, 16, 128, 1, 0.1, None) == NULL
    assert L.tyr_hip_flash_attn_fwd(p, p, p, p, None, 1, 1, 0, 128, 1, 0.1, None) == SHAPE
    assert L.tyr_hip_flash_attn_fwd(p, p, p, p, None, 1, 1, 16, 96, 1, 0.1, None) == UNSUP
    assert L.tyr_hip_flash_attn_fwd(p, p, p, p, None, 1, 1, 16, 128, 1, -1.0, None) == UNSUP
    assert L.tyr_hip_flash_attn_fwd(p, p, p + 8, p, None, 1, 1, 16, 128, 1, 0.1, None) == MISAL
    assert L.tyr_hip_gqa_decode(p, p, p, p, None, 1, 6, 4, 16, 128, 16, 0.1, 1, p, 1 << 20, None) == SHAPE   # Hq % Hkv
    assert L.tyr_hip_gqa_decode(p, p, p, p, None, 1, 8, 2, 16, 128, 8, 0.1, 1, p, 1 << 20, None) == SHAPE   # stride < L
    assert L.tyr_hip_gqa_decode(p, p, p, p, None, 1, 8, 2, 16, 96, 16, 0.1, 1, p, 1 << 20, None) == UNSUP
    assert L.tyr_hip_gqa_decode(p, p, p, p, None, 1, 8, 2, 16, 128, 16, 0.1, 1, None, 0, None) == WS
    assert L.tyr_hip_gqa_decode(p, p, p, p, None, 1, 8, 2, 16, 128, 16, 0.1, 1, p, 64, None) == WS
    assert L.tyr_hip_gqa_decode_workspace_bytes(2, 8, 2, 1000, 128, 4) == 2 * 8 * 4 * 130 * 4
    assert 1 <= L.tyr_hip_gqa_decode_auto_splits(32, 8, 8192) <= 64
    assert L.tyr_hip_gqa_decode_auto_splits(1, 1, 10) == 1
    assert OK == 0


def test_automatic_decode_splits_all_hold_rows():
    """The count the library reports, sizes the workspace for and launches is one count: chunks are whole 32-row steps, and
    every one of them holds rows."""
    L = _lib.load()
    for B in (1, 2, 3, 5, 8, 13, 20, 33, 40, 64):
        for Hkv in (1, 2, 4, 8, 15, 32):
            for rows in (1, 64, 383, 385, 416, 417, 700, 1023, 1500, 2000, 2049, 3001, 8191, 32768, 100001):
                s = L.tyr_hip_gqa_decode_auto_splits(B, Hkv, rows)
                chunk = -(-(-(-rows // s)) // 32) * 32
                assert 1 <= s <= 64 and -(-rows // chunk) == s, (B, Hkv, rows, s, chunk)
                assert L.tyr_hip_gqa_decode_workspace_bytes(B, Hkv, Hkv, rows, 128, 0) == B * Hkv * s * 130 * 4


@pytest.mark.parametrize("B,Hq,Hkv,N,D,cut", [
    (9, 16, 4, 1944, 128, True),       # 36 kv heads: whole key tiles 832 us, in parts 573
    (5, 32, 8, 1325, 128, True),       # 331, 296
    (2, 32, 8, 4601, 64, False),       # with a key mask 507 whole, 607 in parts
    (4, 16, 4, 3000, 128, False),      # whole 534, in parts 555: the long first tiles run while other CUs are idle
    (16, 16, 16, 4096, 128, False),    # 8192 key tiles fill the device
    (1, 32, 8, 2000, 128, True)])      # 254, 149
def test_backward_cuts_key_tiles_where_that_is_faster(B, Hq, Hkv, N, D, cut):
    """The workspace of the parts says whether dK / dV of a causal backward are cut into them; the times are of an MI355X."""
    L = _lib.load()
    least = L.tyr_hip_flash_attn_bwd_workspace_bytes(B, Hq, N, D)
    assert (L.tyr_hip_flash_attn_bwd_parts_workspace_bytes(B, Hq, Hkv, N, D, 1, 0) > least) == cut


@pytest.mark.parametrize("bh,N,D,causal,window,rows", [
    (96, 382, 128, 0, 0, 128),         # whole backward 60.6 us with 128-row tiles for dQ, 67.6 with 64
    (40, 8160, 128, 1, 103, 128),      # 261, 285
    (384, 810, 128, 1, 613, 128),      # 392, 416
    (12, 3472, 128, 1, 0, 64),         # 181, 170
    (8, 3545, 128, 1, 763, 64),        # 66.2, 64.4: few jobs under a window
    (192, 150, 64, 0, 0, 128)])        # 23.8, 25.1
def test_dq_takes_the_form_that_is_faster_for_it(bh, N, D, causal, window, rows):
    """The dQ kernel's tiles are chosen by its own step times (internal function; the times are of an MI355X)."""
    class Shape(ctypes.Structure):
        _fields_ = [("rows", ctypes.c_int), ("pair", ctypes.c_int), ("single", ctypes.c_int)]
    shape = ctypes.CDLL(_lib.LIB_PATH)["_ZN3tyr10attn_shapeEliibib"]
    shape.restype, shape.argtypes = Shape, [ctypes.c_int64, ctypes.c_int, ctypes.c_int, ctypes.c_bool, ctypes.c_int, ctypes.c_bool]
    assert shape(bh, N, D, bool(causal), window, True).rows == rows


def test_nothing_throws_when_the_heap_is_exhausted(tmp_path):
    """The header promises that no entry point throws.  Host-side planning runs here with an operator new that fails: an
    exception would leave a C function and end the process."""
    src = tmp_path / "no_heap.cpp"
    src.write_text(r"""
#include <dlfcn.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <new>
static bool fail;
void* operator new(size_t n) { if (fail) throw std::bad_alloc(); return malloc(n); }
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }
int main(int, char** argv) {
    void* h = dlopen(argv[1], RTLD_NOW);
    if (!h) { puts(dlerror()); return 2; }
    auto bwd = (size_t(*)(uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, int, uint64_t))dlsym(h, "tyr_hip_flash_attn_bwd_full_workspace_bytes");
    auto gemm = (size_t(*)(uint64_t, uint64_t, uint64_t, uint64_t, int, int))dlsym(h, "tyr_hip_gemm_workspace_bytes");
    auto dec = (size_t(*)(uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t))dlsym(h, "tyr_hip_gqa_decode_workspace_bytes");
    fail = true;
    size_t sum = 0;
    for (uint64_t n = 1; n <= 8192; n = n * 3 / 2 + 1)
        for (uint64_t hkv = 1; hkv <= 32; hkv *= 2)
            for (int causal = 0; causal < 2; ++causal)
                sum += bwd(1, 32, hkv, n, 128, causal, 0) + bwd(3, 32, hkv, n, 64, 1, 100) + gemm(1, n, 8 * n, 16 * n, 2, 1) + dec(2, 32, hkv, n, 128, 0);
    fail = false;
    printf("ok %d\n", sum != 0);
}
""")
    exe = tmp_path / "no_heap"
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-rdynamic", str(src), "-o", str(exe), "-ldl"])
    r = subprocess.run([str(exe), _lib.LIB_PATH], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout == "ok 1\n", (r.returncode, r.stdout, r.stderr[-500:])


def test_import_opens_no_kernel_library(tmp_path):
    """Importing the package opens nothing; the library is opened by the first call, and one that lacks functions (an older
    build) is no error before a call needs them."""
    src = tmp_path / "few.c"
    src.write_text('const char* tyr_hip_strerror(int s) { return s ? "bad" : "ok"; }\n')
    few = tmp_path / "libfew.so"
    subprocess.check_call(["gcc", "-shared", "-fPIC", str(src), "-o", str(few)])
    code = ("import tyr_amd, torch\nfrom tyr_amd import gpu\nmaps = open('/proc/self/maps').read()\n"
            "assert '_tyr_torch' in maps and 'libfew' not in maps and 'libtyr_hip' not in maps\n"
            "try: tyr_amd.copy(torch.zeros(4))\nexcept tyr_amd.TyrGpuError as e: assert 'CUDA tensor' in str(e), e\n"
            "assert 'libfew' not in open('/proc/self/maps').read()\nprint('ok')\n")
    for lib in (str(few), str(tmp_path / "absent.so"), _lib.LIB_PATH):
        r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, cwd=ROOT, env=dict(os.environ, TYR_HIP_LIBRARY=lib))
        assert r.returncode == 0 and r.stdout == "ok\n", (lib, r.stdout, r.stderr[-800:])


def test_python_mirror_refuses_cpu_tensors_without_a_gpu():
    import torch
    import tyr_amd
    a = torch.zeros(16, 16, dtype=torch.bfloat16)
    with pytest.raises(tyr_amd.TyrGpuError, match="a must be a CUDA tensor"):
        tyr_amd.gemm_bf16(a, a)
    with pytest.raises(tyr_amd.TyrGpuError, match="q must be a CUDA tensor"):
        tyr_amd.flash_attn_fwd(a.view(1, 1, 16, 16), a.view(1, 1, 16, 16), a.view(1, 1, 16, 16))
