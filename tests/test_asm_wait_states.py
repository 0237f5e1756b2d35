"""What the gfx950 assembly of the attention backward has to show (compiled here, no GPU needed).

Wait states around the matrix products that flash_attn_bwd_dkv_wide_kernel issues in asm, where the compiler, which puts
them in for its own products, does not see any.  Every product of those kernels is checked against the instructions around it
on every path, over forward and backward branches:
  * no operand is written by an ordinary vector instruction less than 2 wait states before the product,
  * no result is read or written by another kind of instruction less than 8 (16x16x32) or 12 (32x32x16) wait states behind it,
  * no accumulator operand of a product in flight is written,
  * no product starts from a part of another's result, or from one of another kind, in that time.
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


class Flight:
    """What may still be under way at a point: register -> wait states that are left, for ordinary writes, results of products (with the
    product's whole result and kind) and accumulators that products read."""

    def __init__(self):
        self.written, self.results, self.sources = {}, {}, {}

    def merge(self, other):
        """Takes over what is longer under way in `other`; whether anything was."""
        grown = False
        for mine, theirs in ((self.written, other.written), (self.results, other.results), (self.sources, other.sources)):
            for r, x in theirs.items():
                have = mine.get(r, (0, *x[1:]))
                joined = (max(have[0], x[0]), *(p if p == q else None for p, q in zip(have[1:], x[1:])))
                if mine.get(r) != joined:
                    mine[r] = joined
                    grown = True
        return grown

    def copy(self):
        out = Flight()
        out.written, out.results, out.sources = dict(self.written), dict(self.results), dict(self.sources)
        return out

    def passes(self, states):
        for d in (self.written, self.results, self.sources):
            for r in [r for r, x in d.items() if x[0] <= states]:
                del d[r]
            for r, x in d.items():
                d[r] = (x[0] - states, *x[1:])

    def step(self, line):
        """One instruction; whether it came too early."""
        name, ops = operands(line)
        if name == "s_nop":
            self.passes(int(ops[0], 0) + 1)
            return False
        if name.startswith("v_mfma"):
            need = 12 if "32x32" in name else 8
            dst, a, b, c = (registers(o) for o in ops[:4])
            bad = any(r in self.written for r in a | b | c) or any(r in self.results for r in a | b)
            # a product in flight hands its result on to the accumulator of one like it, as a whole
            bad |= any(self.results[r][1:] != (frozenset(x), name[:12]) for x in (dst, c) for r in x if r in self.results)
            self.passes(1)
            for r in dst:
                self.results[r] = (need, frozenset(dst), name[:12])
            for r in c:
                self.sources[r] = (need,)
            return bad
        used = registers(" ".join(ops))
        stores = name.startswith(("global_store", "buffer_", "ds_write", "scratch_store", "s_"))
        writes = set() if stores or not ops else registers(ops[0]) | (registers(ops[1]) if "swap" in name else set())
        bad = any(r in self.results for r in used) or any(r in self.sources for r in writes)
        self.passes(1)
        for r in writes:
            self.results.pop(r, None)
            self.written.pop(r, None)
            if name.startswith("v_"):
                self.written[r] = (2,)
        return bad


def violations(lines):
    """Instructions that come too early on some path: every branch is followed, taken and not, until nothing new is under way."""
    at = {m.group(1): i for i, l in enumerate(lines) if (m := re.match(r"(\.?\w+):", l))}
    before = {0: Flight()}
    todo, bad = [0], set()
    while todo:
        i = todo.pop()
        state = before[i].copy()
        while i < len(lines):
            line = lines[i]
            if not line.endswith(":"):
                if state.step(line):
                    bad.add(i)
                m = re.match(r"s_(c?)branch\S*\s+(\S+)", line)
                if m:
                    goal = at[m.group(2)]
                    if goal not in before:
                        before[goal] = state.copy()
                        todo.append(goal)
                    elif before[goal].merge(state):
                        todo.append(goal)
                    if not m.group(1):
                        break
                if line.startswith("s_endpgm"):
                    break
            elif i in before:                        # a label that is reached from above too
                if before[i].merge(state):
                    todo.append(i)
                state = before[i].copy()
            i += 1
    return [lines[i] for i in sorted(bad)]


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
        assert violations(lines) == [], name


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
    assert violations([acc, "s_nop 10", "v_accvgpr_read_b32 v20, a3"]) and not violations([acc, "s_nop 11", "v_accvgpr_read_b32 v20, a3"])
    assert violations([mfma, "v_mfma_f32_16x16x32_bf16 v[2:5], v[12:15], v[8:11], v[2:5]"])          # overlaps a result in flight
    assert violations([mfma, "v_mfma_f32_32x32x16_bf16 v[16:31], v[4:7], v[8:11], v[0:15]"])         # another kind of product


def test_every_branch_is_followed():
    mfma, use, nop = "v_mfma_f32_16x16x32_bf16 v[0:3], v[4:7], v[8:11], v[0:3]", "v_mul_f32 v20, v1, v1", "s_nop 7"
    # a loop: the product at its end, the use at its start
    assert violations([".LBB0_1:", use, mfma, "s_cbranch_scc1 .LBB0_1", "s_endpgm"])
    assert not violations([".LBB0_1:", use, mfma, nop, "s_cbranch_scc1 .LBB0_1", "s_endpgm"])
    # a block out of line, behind the kernel's end: from the branch into it, and back
    away = [mfma, "s_cbranch_scc1 .LBB0_2", nop, ".LBB0_1:", "s_endpgm", ".LBB0_2:"]
    assert violations(away + [use, "s_branch .LBB0_1"])
    assert not violations(away + [nop, use, "s_branch .LBB0_1"])
    back = ["s_cbranch_scc1 .LBB0_2", ".LBB0_1:", mfma, "s_endpgm", ".LBB0_2:"]
    assert violations(back + ["v_mov_b32 v4, 0", "s_branch .LBB0_1"])
    assert not violations(back + ["v_mov_b32 v4, 0", "s_nop 0", "s_branch .LBB0_1"])
    # a block skipped: the use behind it
    assert violations([mfma, "s_cbranch_execz .LBB0_1", nop, ".LBB0_1:", use, "s_endpgm"])
