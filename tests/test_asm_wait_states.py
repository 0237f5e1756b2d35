"""What the gfx950 assembly of the attention backward has to show (compiled here, no GPU needed).

Wait states around the matrix products that flash_attn_bwd_dkv_wide_kernel issues in asm, where the compiler, which puts
them in for its own products, does not see any.  Every product of those kernels is checked against the instructions around it,
with the body of every loop entered twice:
  * no operand is written by an ordinary vector instruction less than 2 wait states before the product,
  * no result is read or written by another kind of instruction less than 8 (16x16x32) or 12 (32x32x16) wait states behind it,
  * no accumulator operand of a product in flight is written.
An instruction is one wait state, s_nop n is n + 1.

Scalar offsets of the requests of query tiles: at most the size of the buffer, which is what their range check is known for.

Registers of the dQ kernels: as many waves a SIMD as each form is launched for, and no more in scratch memory than is stated beside them."""
import os
import re
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tyr_amd", "csrc")
HIPCC = "/opt/rocm/bin/hipcc"


def registers(text):
    """(class, index) of every vector register that a list of operands names."""
    out = set()
    for c, lo, hi, one in re.findall(r"\b([va])(?:\[(\d+):(\d+)\]|(\d+)\b)", text):
        out |= {(c, i) for i in (range(int(lo), int(hi) + 1) if lo else (int(one),))}
    return out


def operands(line):
    name, _, rest = line.partition(" ")
    ops, depth, cur = [], 0, ""
    for ch in rest:
        depth += (ch == "[") - (ch == "]")
        if ch == "," and depth == 0:
            ops.append(cur.strip())
            cur = ""
        else:
            cur += ch
    return name, [o for o in ops + [cur.strip()] if o]


def straight(lines):
    """Instructions with every backward branch taken once more."""
    at = {m.group(1): i for i, l in enumerate(lines) if (m := re.match(r"(\.L\w+):", l))}
    out = []
    for i, l in enumerate(lines):
        if not l.endswith(":"):
            out.append(l)
        m = re.match(r"s_c?branch\S*\s+(\.L\w+)", l)
        if m and at.get(m.group(1), i + 1) <= i:
            out += [x for x in lines[at[m.group(1)]:i + 1] if not x.endswith(":")]
    return out


def violations(code):
    bad, now = [], 0
    vector_write, result, source = {}, {}, {}     # register -> wait state of its last write; (wait state, needed) of a product's result, operand
    for line in code:
        name, ops = operands(line)
        if name == "s_nop":
            now += int(ops[0], 0) + 1
            continue
        now += 1
        if name.startswith("v_mfma"):
            need = 12 if "32x32" in name else 8
            dst, a, b, c = (registers(o) for o in ops[:4])
            bad += [line for r in a | b | c if now - vector_write.get(r, -99) <= 2]
            bad += [line for r in (a | b) & result.keys() if now - result[r][0] <= result[r][1]]
            for r in dst:
                result[r] = (now, need)
            for r in c:
                source[r] = (now, need)
            continue
        used = registers(" ".join(ops))
        bad += [line for r in used & result.keys() if now - result[r][0] <= result[r][1]]
        stores = name.startswith(("global_store", "buffer_", "ds_write", "scratch_store", "s_"))
        written = set() if stores or not ops else registers(ops[0]) | (registers(ops[1]) if "swap" in name else set())
        bad += [line for r in written & source.keys() if now - source[r][0] <= source[r][1]]
        for r in written:
            result.pop(r, None)
            if name.startswith("v_"):
                vector_write[r] = now
            else:
                vector_write.pop(r, None)
    return bad


def wide_kernels(path):
    with open(path) as f:
        text = f.read()
    for m in re.finditer(r"^(_ZN3tyr30flash_attn_bwd_dkv_wide_kernel\w+):(.*?)^\.Lfunc_end", text, re.S | re.M):
        lines = [l.split(";")[0].split("//")[0].strip() for l in m.group(2).split("\n")]
        yield m.group(1), [l for l in lines if l and (l.endswith(":") or not l.startswith("."))]


@pytest.fixture(scope="module")
def listing(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not installed")
    out = str(tmp_path_factory.mktemp("asm") / "bwd.s")
    subprocess.check_call([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                           "--cuda-device-only", "-S", os.path.join(CSRC, "flash_attn_bwd.hip"), "-o", out], stderr=subprocess.DEVNULL)
    return out


def test_products_in_asm_keep_their_distance(listing):
    kernels = dict(wide_kernels(listing))
    assert kernels
    for name, lines in kernels.items():
        assert sum(l.startswith("v_mfma") for l in lines) >= 96, name
        assert violations(straight(lines)) == [], name


def unbounded_requests(code):
    """Buffers (registers of their descriptors) with a request whose scalar offset is not a minimum with a buffer's size."""
    last, out = {}, {}
    for line in code:
        name, ops = operands(line)
        if name == "buffer_load_dwordx4" and line.endswith(" lds"):
            out.setdefault(ops[1], []).append(last.get(ops[2].split()[0]) == "s_min_u32")
        elif name.startswith("s_") and ops and re.fullmatch(r"s\d+", ops[0]):
            last[ops[0]] = name
    return out, {d for d, bounded in out.items() if not all(bounded)}


def test_no_request_of_a_query_tile_starts_beyond_its_buffer(listing):
    """(the statistics' offset is a whole tile's and needs no minimum)"""
    kernels = dict(wide_kernels(listing))
    assert kernels
    for name, lines in kernels.items():
        buffers, unbounded = unbounded_requests(lines)
        assert len(buffers) == 3 and len(unbounded) <= 1, (name, unbounded)
        assert sorted(map(len, buffers.values()))[1:] == [16 if "Li128E" in name else 8] * 2, name      # four tiles in the code, PT pieces each


def resources(path):
    """Registers, and registers kept in scratch, of every kernel by its mangled name."""
    with open(path) as f:
        for block in f.read().split("\n  - .agpr_count:")[1:]:
            field = lambda key: re.search(rf"\.{key}:\s+(\S+)", block).group(1)
            yield field("name"), (int(field("vgpr_count")), int(field("vgpr_spill_count")))


def test_dq_kernels_keep_their_waves(listing):
    """A SIMD's 512 registers hold three waves of up to 168; the launch bounds only ask for two."""
    seen = 0
    for name, (registers, spilled) in resources(listing):
        m = re.search(r"flash_attn_bwd_dq_kernelILi(64|128)ELb([01])ELNS_8AttnMaskE([012])ELb([01])E", name)
        if not m:
            continue
        D, causal, mask, split = map(int, m.groups())
        seen += 1
        if D == 64 and causal and (mask != 2 or split):
            assert registers <= 168, (name, registers)
        assert spilled <= (0 if causal or D == 64 else 52), (name, spilled)
    assert seen == 24


def test_what_comes_too_early_is_found():
    mfma = "v_mfma_f32_16x16x32_bf16 v[0:3], v[4:7], v[8:11], v[0:3]"
    assert violations(["v_mov_b32 v4, 0", mfma]) and not violations(["v_mov_b32 v4, 0", "s_nop 1", mfma])
    assert violations([mfma, "s_nop 6", "v_mul_f32 v20, v1, v1"]) and not violations([mfma, "s_nop 7", "v_mul_f32 v20, v1, v1"])
    assert violations([mfma, "ds_read_b128 v[0:3], v30"]) and not violations([mfma, mfma])
    acc = "v_mfma_f32_32x32x16_bf16 a[0:15], v[4:7], v[8:11], a[0:15]"
    assert violations([acc, "s_nop 7", "v_accvgpr_read_b32 v20, a3"])
    assert violations(straight([".LBB0_1:", "v_mul_f32 v20, v1, v1", mfma, "s_cbranch_scc1 .LBB0_1"]))
