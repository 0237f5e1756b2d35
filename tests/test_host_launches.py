"""What the C ABI's host code decides, on the CPU: the kernel files are compiled for the host alone, with every signed overflow
an abort, and linked with a HIP runtime that records the launches instead of making them (tests/host_launches)."""
import os
import re
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

from tests.test_gpu_attention_bwd_wide import TWO_A_CU, WIDE

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CHECKED = ["-Xarch_host", "-fsanitize=signed-integer-overflow", "-Xarch_host", "-fsanitize-minimal-runtime", "-Xarch_host",
           "-fno-sanitize-recover=signed-integer-overflow"]


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("host")
    hipcc = "/opt/rocm/bin/hipcc"

    def compile_(name):
        obj = str(tmp / (os.path.basename(name) + ".o"))
        subprocess.check_call([hipcc, "--offload-arch=gfx950", "--offload-host-only", "-O1", "-std=c++17", "-w", *CHECKED, "-c",
                               os.path.join(ROOT, name), "-o", obj])
        return obj
    with ThreadPoolExecutor() as pool:
        objs = list(pool.map(compile_, [f"tyr_amd/csrc/{n}.hip" for n in ("capi", "flash_attn_fwd", "flash_attn_bwd", "gemm_bf16", "gemm_fp8")]))
    main, exe = str(tmp / "recorder.o"), str(tmp / "recorder")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__=1", "-isystem", "/opt/rocm/include", "-c",
                           os.path.join(ROOT, "tests", "host_launches", "recorder.cpp"), "-o", main])
    # what the other kernel files and the fat binaries would define is never reached
    subprocess.check_call(["/opt/rocm/llvm/bin/clang++", main, *objs, "-fsanitize=signed-integer-overflow", "-fsanitize-minimal-runtime",
                           "-Wl,--unresolved-symbols=ignore-all", "-o", exe])

    def run(lines):
        r = subprocess.run([exe], input="\n".join(lines) + "\n", capture_output=True, text=True)
        got = r.stdout.splitlines()
        assert r.returncode == 0 and len(got) == len(lines), (lines[min(len(got), len(lines) - 1)], r.returncode, r.stderr[-300:])
        return got
    return run


def test_a_window_of_any_size_is_one_of_all_rows(ask):
    """The sums that the plan and the places of dS make with a window stay in 32 bits: the last 126 values below 2^31 did not."""
    for B, Hq, Hkv, N in ((1, 32, 8, 2000), (4, 16, 16, 769), (9, 16, 4, 200), (2, 4, 4, 100), (16, 16, 16, 4096)):
        whole = None
        for window in (N, N + 1, 2 ** 30, 2 ** 31 - 127, 2 ** 31 - 126, 2 ** 31 - 1, 2 ** 31, 2 ** 64 - 1):
            size, = ask([f"bytes {B} {Hq} {Hkv} {N} 128 1 {window}"])
            got = [size] + ask([f"bwd {B} {Hq} {Hkv} {N} 128 1 {window} {mask} {ws}" for mask in ("none", "lens") for ws in size.split()])
            whole = whole or got
            assert got == whole and got[1].startswith("0 flash_attn_bwd"), (window, got, whole)


def test_scratch_queries_take_any_length(ask):
    """Beyond the lengths a call accepts, the largest scratch is 0 (nothing uses it); no query overflows."""
    for N in (2 ** 22, 2 ** 23 - 1, 2 ** 23, 2 ** 25, 2 ** 30, 2 ** 31 - 129, 2 ** 31 - 127, 2 ** 31 - 1, 2 ** 31, 2 ** 40):
        for window in (0, 1, 2 ** 31 - 1, 2 ** 40):
            for D in (64, 128):
                got, = ask([f"bytes 1 1 1 {N} {D} 1 {window}"])
                least, parts, full = map(int, got.split())
                assert least == (0 if N >= 2 ** 31 else (N + 127) // 128 * 1024)
                assert (full == parts == 0) if N * D * 2 >= 2 ** 31 else full >= parts >= least
                call, = ask([f"bwd 1 1 1 {N} {D} 1 {window} none {least}"])
                assert (call == "-3" if N < 2 ** 31 else call == "-2") if full == 0 else call.startswith("0 flash_attn_bwd")


@pytest.mark.parametrize("B,Hq,Hkv,N,D,causal,window", [(1, 32, 8, 2000, 128, 1, 0), (2, 16, 4, 1500, 128, 0, 0), (1, 8, 8, 3000, 128, 1, 1500),
                                                        (1, 4, 4, 700, 128, 1, 0), (1, 8, 2, 2049, 64, 1, 0), (2, 4, 4, 100, 64, 0, 0),
                                                        (16, 16, 16, 4096, 128, 1, 0)])
@pytest.mark.parametrize("mask", ["none", "lens", "keys"])
def test_backward_runs_the_largest_form_that_its_scratch_holds(ask, B, Hq, Hkv, N, D, causal, window, mask):
    """dS kept, else key tiles cut into parts, else whole key tiles: one byte less than a form needs gives the next one."""
    window = 0 if mask == "keys" else window
    shape = f"{B} {Hq} {Hkv} {N} {D} {causal} {window}"
    least, parts, full = map(int, ask([f"bytes {shape}"])[0].split())
    sizes = [least - 1, least, parts - 1, parts, full - 1, full, 1 << 40]
    got = dict(zip(sizes, ask([f"bwd {shape} {mask} {n}" for n in sizes])))
    assert got[least - 1] == "-5" and got[full] == got[1 << 40]
    assert not any(k in got[least] for k in ("_sum_", "_product_"))
    if parts > least:
        assert got[parts - 1] == got[least] and "_sum_kernel" in got[parts] and "_product_" not in got[parts]
    if full > parts:
        assert got[full - 1] == got[parts] and "_stats_kernel" in got[full] and "_product_kernel" in got[full]
    kept, cut = {2000: (True, True), 1500: (True, True), 3000: (True, not window), 700: (False, True), 2049: (False, True),
                 100: (False, False), 4096: (False, False)}[N]
    assert (full > parts, parts > least) == (kept, cut)


def test_every_backward_kernel_is_reached(ask):
    built = {k for k in ask(["kernels"])[0].split() if k.startswith("flash_attn_bwd")}
    shapes = [f"{B} {Hq} {Hkv} {N} {D} {opt}" for B in (1, 2, 4, 16) for Hq, Hkv in ((1, 1), (8, 2), (4, 4), (32, 8)) for N in (64, 300, 700, 1500, 4096)
              for D in (64, 128) for opt in ("0 0", "1 0", "1 50", "1 600")]
    calls = [f"bwd {shape} {mask} {ws}" for shape, sizes in zip(shapes, ask([f"bytes {s}" for s in shapes])) for ws in sizes.split()
             for mask in ("none", "lens", "keys") if mask != "keys" or shape.endswith(" 0")]
    got = ask(calls)
    assert all(g.startswith("0 ") for g in got)
    assert built == {k.rsplit(":", 1)[0] for g in got for k in g.split()[1:]}


@pytest.mark.parametrize("M,N,K,trans_b,size", [(256, 4096, 4096, 0, 2), (1, 4096, 4096, 1, 2), (3, 512, 8192, 1, 2), (200, 16, 8192, 1, 2),
                                                (4096, 4096, 4096, 0, 2), (333, 4096, 4096, 1, 1), (120, 1024, 8192, 0, 1)])
def test_sums_in_any_order_need_no_memory(ask, M, N, K, trans_b, size):
    """Without memory for partials, or with less than they take, K is not split, but still summed by as many waves as is fastest;
    without a workspace in the order that a batch has.  The scratch of what is not split is none."""
    def call(ws):
        rc, need, *kernels = ask([f"gemm {M} {N} {K} {trans_b} {size} {ws}"])[0].split()
        assert rc == "0"
        return int(need), " ".join(kernels)
    need, alone = call("any")
    assert "_reduce_" not in alone and call(16)[1] == alone
    if need:
        assert "_reduce_" in call(need)[1] and call(need - 1)[1] == alone
    else:
        assert call(1 << 40)[1] == alone
    assert (need > 0) == ((M, N) in ((3, 512), (200, 16), (120, 1024)))
    assert (call(0)[1] == alone) == (size == 1 or M == 4096), (call(0), alone)


@pytest.mark.parametrize("M,N,K,trans_b,size,rows,cols,groups,split", [
    (2719, 448, 1280, 0, 2, 96, 64, 2, False),      # 8.2 us; 64x128 over two k-groups 8.7
    (1105, 1344, 832, 0, 2, 96, 64, 2, False),      # 6.9, 7.2
    (173, 352, 4456, 1, 2, 16, 16, 4, False),       # 5.2; over eight k-groups 5.9
    (401, 296, 3488, 1, 2, 32, 32, 4, False),       # 5.7; 16x16 over eight 7.0
    (549, 736, 7936, 0, 1, 64, 128, 1, True),       # 13.3; 32x64 over four in one piece 17.9
    (1, 4096, 4096, 1, 2, 16, 16, 8, False),        # 4.4; over four 4.9
    (333, 4096, 4096, 1, 1, 64, 128, 2, False),     # 10.9; over one 12.4
    (256, 4096, 4096, 0, 2, 64, 64, 2, False)])     # 14.6; over one 17.5
def test_tiles_of_twice_the_waves_where_they_are_faster(ask, M, N, K, trans_b, size, rows, cols, groups, split):
    """The tile of a product, the k-groups of its workgroups and whether K is split; the times are of an MI355X."""
    got, = ask([f"gemm {M} {N} {K} {trans_b} {size} {1 << 40}"])
    m = re.fullmatch(r"0 \d+ gemm_tile_kernel<gt::Cfg<(1|2),(true|false),(\d+),(\d+),\d+,\d+,(\d+),\d+>>:\d+( gemm_tile_reduce_kernel<\d>:\d+)?", got)
    assert m and (int(m[1]), m[2] == "true", int(m[3]), int(m[4]), int(m[5]), bool(m[6])) == (size, bool(trans_b), rows, cols, groups, split), got


@pytest.mark.parametrize("B,Hq,Hkv,N,D,opt,form", [
    (1, 32, 32, 315, 64, "0 0", "half"),        # two launches 16.9, one 14.0, 64-key tiles 11.3 us, two workgroups of which share a CU
    (10, 32, 8, 222, 64, "0 0", "half"),        # 41.7, -, 35.3
    (9, 8, 8, 66, 64, "0 0", "half"),           # 11.5, 8.3, 8.0
    (1, 16, 4, 1042, 64, "0 0", "two"),         # 45.8, 55.8, 67.7
    (2, 4, 4, 2129, 64, "0 0", "two"),          # 68.6, 81.1, 74.2: too many rows for two workgroups on a CU
    (7, 8, 8, 143, 64, "0 0", "half"),          # 13.8, 11.4, 9.1: shared CUs in a launch of few more workgroups than CUs
    (1, 2, 2, 2001, 64, "1 0", "one"),          # 39.8, 31.3, 37.3
    (4, 8, 8, 310, 64, "1 0", "half"),          # 20.2, 16.1, 11.3
    (1, 1, 1, 128, 64, "0 0", "half"),          # the train step of one head
    (2, 8, 8, 685, 128, "0 0", "one"),          # 40.3, 34.5, 41.0; dS kept 38.6
    (5, 8, 8, 217, 128, "0 0", "one"),          # 24.6, 17.5, 19.8; 22.5
    (2, 8, 8, 685, 128, "1 0", "half"),         # 40.4, 38.1, 26.6; 31.9
    (2, 16, 16, 764, 128, "1 0", "one"),        # 45.4, 40.7, 47.3; 46.0
    (4, 16, 4, 544, 128, "1 0", "ds"),          # 52.5, 60.2, 68.3; 45.4
    (1, 32, 8, 2000, 128, "1 0", "ds"),         # 148, -, -; 136
    (16, 16, 16, 4096, 128, "1 0", "two")])     # dS would take 4.4 GB
def test_the_form_of_a_backward_is_the_fastest(ask, B, Hq, Hkv, N, D, opt, form):
    """By the launches of a call with all the scratch it can use; the times are of an MI355X, whole backward."""
    got, = ask([f"bwd {B} {Hq} {Hkv} {N} {D} {opt} none {1 << 40}"])
    first = got.split()[1]
    kind = {"flash_attn_bwd_dq_kernel": "two", "flash_attn_bwd_stats_kernel": "ds", "flash_attn_bwd_both_kernel": "half" if first.split(":")[0].endswith("true>") else "one"}
    assert kind[first.split("<")[0]] == form, got


def test_the_shapes_of_the_wide_tests_take_their_kernels(ask):
    """dK / dV by key tiles of 256, or one launch of 64-key tiles that leaves a CU (160 KB of LDS, 256 CUs) room for two of more workgroups
    than CUs: what tests/test_gpu_attention_bwd_wide.py compares has to run them."""
    def launches(B, Hq, Hkv, N, D, causal, mask, window):
        got, = ask([f"bwd_lds {B} {Hq} {Hkv} {N} {D} {int(causal)} {window} {mask or 'none'} {1 << 40}"])
        return [k.rsplit(":", 2) for k in got.split()[1:]]
    for row in WIDE:
        (first, _, _), (second, grid, _) = launches(*row)
        assert first.startswith("flash_attn_bwd_dq_kernel<") and second.startswith("flash_attn_bwd_dkv_wide_kernel<"), row
        assert int(grid) == row[0] * row[2] * -(-row[3] // 256), row
    for row in TWO_A_CU:
        (only, grid, lds), = launches(*row)
        assert re.fullmatch(r"flash_attn_bwd_both_kernel<64,.*,true>", only) and int(grid) > 256 and 2 * int(lds) <= 160 * 1024, (row, only, lds)
