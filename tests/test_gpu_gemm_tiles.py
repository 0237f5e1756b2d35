"""The small and medium GEMM tiles and their dispatch: sizes around every tile edge, ragged K (a last piece of 16 bytes
up to 128), one to many pieces per k-group, K split over workgroups, and outputs that must stay inside C."""
import pytest
import torch

from oracle import libtorch_path as lt
from tests.util import rel_fro

pytestmark = pytest.mark.gpu
TOL_FRO = 1e-2

# (M, N, K): the first extents pick tiles of 16..192 rows and 16..256 columns, one less and one more row than a tile each
SHAPES = [(1, 16, 16), (1, 272, 2048), (15, 4096, 144), (17, 1040, 4096), (33, 272, 528), (31, 4112, 1040), (64, 48, 80), (65, 1296, 3088),
          (95, 4096, 2064), (97, 2064, 272), (127, 1024, 4112), (129, 528, 1296), (200, 16, 8192), (3, 512, 8192), (333, 1408, 6608),
          (255, 6144, 400), (385, 2560, 2048), (1000, 2576, 1024), (1290, 4080, 256), (2050, 1040, 1552)]


def worst_line(got, want):
    """Largest relative error of a row or column (a wrong tile edge would drown in the norm of the whole)."""
    err, worst = got.float() - want, 0.0
    for dim in (0, 1):
        n = want.norm(dim=dim)
        worst = max(worst, float((err.norm(dim=dim) / n.clamp_min(float(n.mean()))).max()))
    return worst


@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_tiles_match_the_f32_product(M, N, K, trans_b):
    import tyr_amd
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    a = (torch.randn(M, K, generator=g, device="cuda") * K ** -0.25).bfloat16()
    b = (torch.randn(K, N, generator=g, device="cuda") * K ** -0.25).bfloat16()
    bb = b.t().contiguous() if trans_b else b
    want = a.float() @ b.float()
    c = tyr_amd.gemm_bf16(a, bb, trans_b=trans_b)
    assert rel_fro(c, want) <= 3e-3
    assert torch.equal(tyr_amd.gemm_bf16(a, bb, trans_b=trans_b), c)
    assert worst_line(c, want) <= TOL_FRO
    aq, sa = tyr_amd.quantize_e4m3(a)
    bq, sb = tyr_amd.quantize_e4m3(b)
    bqb = bq.t().contiguous() if trans_b else bq
    want8 = (aq.float() @ bq.float()) * (sa * sb)
    rs = torch.rand(M, generator=g, device="cuda") + 0.5
    cs = torch.rand(N, generator=g, device="cuda") + 0.5
    f = tyr_amd.gemm_fp8_scaled(aq, bqb, rs, cs, scale=sa * sb, trans_b=trans_b)
    assert rel_fro(f, want8 * rs[:, None] * cs[None, :]) <= 1e-4
    c8 = tyr_amd.gemm_fp8(aq, bqb, sa, sb, trans_b=trans_b)
    assert rel_fro(c8, want8) <= 3e-3
    assert worst_line(c8, want8) <= TOL_FRO


def test_every_k_step_of_a_sum_arrives():
    # operands of ones: each output counts the k it saw (the last products of a tile included)
    import tyr_amd
    for M, N in ((16, 64), (40, 1024), (130, 4096), (333, 4096), (640, 2048), (1500, 4096)):
        for K in (128, 144, 1024, 4096):
            for trans_b in (False, True):
                a = torch.ones(M, K, device="cuda").to(torch.float8_e4m3fn)
                b = torch.ones((N, K) if trans_b else (K, N), device="cuda").to(torch.float8_e4m3fn)
                c = tyr_amd.gemm_fp8_scaled(a, b, trans_b=trans_b)
                assert bool((c == K).all()), (M, N, K, trans_b)
                c = tyr_amd.gemm_bf16(a.bfloat16(), b.bfloat16(), trans_b=trans_b)
                assert bool((c == K).all()), (M, N, K, trans_b)


@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("M,N,K", [(5, 24, 4096), (33, 1032, 264), (100, 8, 6000), (130, 4088, 512)])
def test_tiles_write_only_c(M, N, K, trans_b):
    from tyr_amd import _lib
    lib = _lib.load()
    a, b = lt.make_inputs(M + N + K, (M, K), (K, N), std=K ** -0.25)
    ad, bd = a.cuda(), (b.t().contiguous() if trans_b else b).cuda()
    guard = 4096
    buf = torch.full((guard + M * N + guard,), -7.0, dtype=torch.bfloat16, device="cuda")
    need = lib.tyr_hip_gemm_workspace_bytes(1, M, N, K, 2, int(trans_b))
    ws = torch.full((need // 4 + 64,), 5.0, device="cuda")
    for w, nbytes in ((ws.data_ptr(), need), (None, 0)):
        buf.fill_(-7.0)
        rc = lib.tyr_hip_gemm_bf16_batched_ws(ad.data_ptr(), bd.data_ptr(), buf.data_ptr() + 2 * guard, 1, M, N, K, 0, 0, 0, int(trans_b),
                                              w, nbytes, 0)
        assert rc == 0
        torch.cuda.synchronize()
        assert bool((buf[:guard] == -7.0).all()) and bool((buf[guard + M * N:] == -7.0).all())
        assert bool((ws[need // 4:] == 5.0).all())
        assert rel_fro(buf[guard:guard + M * N].view(M, N).cpu(), a.float() @ b.float()) <= TOL_FRO


@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("M,N,K", [(1, 16, 16), (15, 4096, 144), (33, 272, 528), (65, 1296, 3088), (95, 4096, 2064), (127, 1024, 4112),
                                   (129, 528, 1296), (3, 512, 8192), (333, 1408, 6608), (385, 2560, 2048), (1000, 2576, 1024), (2050, 1040, 1552)])
def test_e4m3_output_of_the_tiles(M, N, K, trans_b):
    """The bytes are the f32 output of the same product (same tile, same sums), clamped and rounded to nearest even; scaled so
    that part of them saturate."""
    import tyr_amd
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    aq, sa = tyr_amd.quantize_e4m3(torch.randn(M, K, generator=g, device="cuda"))
    bq, sb = tyr_amd.quantize_e4m3(torch.randn(K, N, generator=g, device="cuda"))
    rs = (torch.rand(M, generator=g, device="cuda") + 0.5) * 300.0
    cs = torch.rand(N, generator=g, device="cuda") + 0.5
    scale = sa * sb * K ** -0.5
    bqb = bq.t().contiguous() if trans_b else bq
    f = tyr_amd.gemm_fp8_scaled(aq, bqb, rs, cs, scale=scale, trans_b=trans_b)
    want = (aq.float() @ bq.float()) * scale * rs[:, None] * cs[None, :]
    assert rel_fro(f, want) <= 1e-4 and worst_line(f, want) <= 1e-3
    if M * N > 1000:
        assert float((f.abs() > 448.0).float().mean()) > 0.01
    got = tyr_amd.gemm_fp8_scaled(aq, bqb, rs, cs, scale=scale, out_dtype=torch.float8_e4m3fn, trans_b=trans_b)
    assert torch.equal(got.view(torch.uint8), f.clamp(-448.0, 448.0).to(torch.float8_e4m3fn).view(torch.uint8))


@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("batch,M,N,K", [(2, 15, 4096, 144), (3, 33, 272, 528), (5, 65, 48, 80), (7, 1, 1040, 2048), (2, 129, 528, 1296),
                                         (3, 200, 16, 4096), (4, 333, 1408, 1608), (2, 1000, 2576, 264)])
def test_batches_of_tiles(batch, M, N, K, trans_b):
    """Every entry has the bits of a product of its own without scratch (K in the same order), and nothing is written between
    the entries of C."""
    from tyr_amd import _lib
    import tyr_amd
    lib = _lib.load()
    g = torch.Generator(device="cuda").manual_seed(batch + M + N + K)
    a = (torch.randn(batch, M, K, generator=g, device="cuda") * K ** -0.25).bfloat16()
    b = (torch.randn(batch, *((N, K) if trans_b else (K, N)), generator=g, device="cuda") * K ** -0.25).bfloat16()
    gap = 64
    c = torch.full((batch, M * N + gap), -7.0, dtype=torch.bfloat16, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    rc = lib.tyr_hip_gemm_bf16_batched(a.data_ptr(), b.data_ptr(), c.data_ptr(), batch, M, N, K, M * K, N * K, M * N + gap, int(trans_b), stream)
    assert rc == 0
    assert bool((c[:, M * N:] == -7.0).all())
    shared = tyr_amd.matmul_bf16(a, b[0].contiguous(), trans_b=trans_b)
    assert torch.equal(tyr_amd.matmul_bf16(a, b, trans_b=trans_b), c[:, :M * N].view(batch, M, N))
    one = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    for i in range(batch):
        for got, bi in ((c[i, :M * N].view(M, N), b[i]), (shared[i], b[0])):
            want = a[i].float() @ (bi.float().t() if trans_b else bi.float())
            assert rel_fro(got, want) <= 3e-3 and worst_line(got, want) <= TOL_FRO
            assert lib.tyr_hip_gemm_bf16(a[i].data_ptr(), bi.data_ptr(), one.data_ptr(), M, N, K, int(trans_b), stream) == 0
            assert torch.equal(got, one)


@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("M,N,K", [(1, 4096, 4096), (15, 264, 8192), (31, 4104, 2056), (33, 4096, 1024), (63, 4088, 2048), (65, 4096, 200),
                                   (250, 4080, 1040), (257, 2048, 4096), (333, 4096, 4096), (512, 4088, 656)])
def test_tiles_whose_k_range_twice_the_waves_share(M, N, K, trans_b):
    """One workgroup a CU: eight waves on a tile instead of four.  Around the tiles' edges, with fewer pieces than waves and with
    rows that start on cache lines or not; bf16 takes these tiles with scratch only, so the product without sums in another order."""
    from tyr_amd import _lib
    lib = _lib.load()
    test_tiles_match_the_f32_product(M, N - N % 16, K - K % 16, trans_b)      # whole chunks of e4m3
    g = torch.Generator(device="cuda").manual_seed(M)
    a = (torch.randn(M, K, generator=g, device="cuda") * K ** -0.25).bfloat16()
    b = (torch.randn(*((N, K) if trans_b else (K, N)), generator=g, device="cuda") * K ** -0.25).bfloat16()
    want = a.float() @ (b.float().t() if trans_b else b.float())
    need = lib.tyr_hip_gemm_workspace_bytes(1, M, N, K, 2, int(trans_b))
    ws = torch.full((need + 64,), 3, dtype=torch.uint8, device="cuda")
    for w, nbytes in ((ws.data_ptr(), need), (ws.data_ptr(), max(0, need - 1)), (None, 0)):
        c = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
        assert lib.tyr_hip_gemm_bf16_batched_ws(a.data_ptr(), b.data_ptr(), c.data_ptr(), 1, M, N, K, 0, 0, 0, int(trans_b), w, nbytes, 0) == 0
        torch.cuda.synchronize()
        assert rel_fro(c, want) <= 3e-3 and worst_line(c, want) <= TOL_FRO
    assert bool((ws[need:] == 3).all()) and (need != 16 or bool((ws == 3).all()))


@pytest.mark.parametrize("rows,cols", [(True, True), (True, False), (False, True)])
@pytest.mark.parametrize("M,N,K", [(1065, 7136, 448), (1281, 6896, 256), (4097, 4112, 528), (1, 272, 2048), (33, 528, 1040), (333, 4096, 1040), (2000, 3088, 1040)])
def test_scales_are_one_factor_an_element(M, N, K, rows, cols):
    """Whatever tile computes them (the first three: 256x256, cut in both directions), scaled results are the unscaled f32 ones
    times the row's factor times the column's, bit for bit in every output type; infinite and NaN factors too."""
    import tyr_amd
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    a, _ = tyr_amd.quantize_e4m3((torch.randn(M, K, generator=g, device="cuda") * K ** -0.25).bfloat16())
    b, _ = tyr_amd.quantize_e4m3((torch.randn(N, K, generator=g, device="cuda") * K ** -0.25).bfloat16())
    plain = tyr_amd.gemm_fp8_scaled(a, b, trans_b=True)
    # the matrix unit aligns the 64 products of a step to the largest one: 2^-14 of it is lost at most, i.e. 6e-5 of a sum
    assert rel_fro(plain, a.float() @ b.float().t()) <= 1e-4
    scale = 0.75 / float(plain.abs().mean())
    rs = torch.rand(M, generator=g, device="cuda") * 900 if rows else None
    cs = torch.rand(N, generator=g, device="cuda") + 0.5 if cols else None
    if rows:
        rs[-1], rs[M // 2] = float("inf"), float("nan")
    if cols:
        cs[-1], cs[N // 2] = float("-inf"), float("nan")
    factor = torch.full((M,), scale, device="cuda") * (rs if rows else 1.0)
    want = plain * factor[:, None]
    want = want * cs if cols else want
    for out in (torch.float32, torch.bfloat16, torch.float8_e4m3fn):
        got = tyr_amd.gemm_fp8_scaled(a, b, rs, cs, scale=scale, out_dtype=out, trans_b=True).float()
        ref = (want.clamp(-448, 448) if out == torch.float8_e4m3fn else want).to(out).float()
        assert torch.equal(got.isnan(), ref.isnan()) and torch.equal(got.nan_to_num(0), ref.nan_to_num(0))
