"""The forms an attention launch can take (paired query tiles, single ones, 64-row tiles whose keys two waves share) and the
backward's dK / dV cut into parts: head counts and lengths on both sides of where the choice changes, with every mask."""
import math

import pytest
import torch

from tests.util import rel_fro

pytestmark = pytest.mark.gpu

# (B, Hq, Hkv, N, D): few heads with short and long rows, part of a tile in the last one, more heads than CUs
SHAPES = [(1, 1, 1, 65, 128), (1, 4, 4, 191, 64), (2, 4, 1, 257, 128), (1, 8, 2, 1000, 128), (1, 16, 16, 1025, 64), (3, 8, 4, 577, 128),
          (4, 16, 16, 700, 128), (2, 32, 8, 449, 64), (8, 32, 8, 300, 128), (1, 4, 1, 3001, 128)]


def reference(q, k, v, g, visible):
    """f32 attention and its gradients; visible [B, 1, N, N]."""
    B, Hq, N, D = q.shape
    rep = Hq // k.shape[1]
    q, k, v = (t.float().requires_grad_() for t in (q, k, v))
    kk, vv = k.repeat_interleave(rep, 1), v.repeat_interleave(rep, 1)
    s = (torch.matmul(q, kk.transpose(-1, -2).contiguous()) / math.sqrt(D)).masked_fill(~visible, float("-inf"))
    lse = torch.logsumexp(s, -1)
    p = torch.exp(s - lse.masked_fill(lse == float("-inf"), 0.0)[..., None])
    o = torch.matmul(p, vv)
    return (o.detach(), lse.detach(), *torch.autograd.grad(o, (q, k, v), g.float()))


@pytest.mark.parametrize("mask", ["causal", "full", "window", "lens", "keys"])
@pytest.mark.parametrize("B,Hq,Hkv,N,D", SHAPES)
def test_every_launch_form_matches_the_f32_reference(B, Hq, Hkv, N, D, mask):
    import tyr_amd
    gen = torch.Generator(device="cuda").manual_seed(B + Hq + N)
    q, k, v, g = (torch.randn(B, h, N, D, device="cuda", generator=gen).bfloat16() for h in (Hq, Hkv, Hkv, Hq))
    i = torch.arange(N, device="cuda")
    visible = (i[None, :] <= i[:, None] if mask != "full" else torch.ones(N, N, dtype=torch.bool, device="cuda"))[None, None].expand(B, 1, N, N)
    opt = dict(causal=mask != "full")
    if mask == "window":
        opt["window"] = N // 3 + 1
        visible = visible & (i[:, None] - i[None, :] < opt["window"])
    if mask == "lens":
        opt["kv_lens"] = torch.tensor([N - b * (N // (2 * B)) for b in range(B)], dtype=torch.int32, device="cuda")
        visible = visible & (i[None, None, None, :] < opt["kv_lens"][:, None, None, None])
    if mask == "keys":
        opt["key_mask"] = torch.rand(B, N, device="cuda", generator=gen) > 0.3
        opt["key_mask"][:, 0] = True
        visible = visible & opt["key_mask"][:, None, None, :]
    o, lse = tyr_amd.flash_attn_fwd(q, k, v, **opt)
    grads = tyr_amd.flash_attn_bwd(q, k, v, o, lse, g, **opt)
    want_o, want_lse, *want = reference(q, k, v, g, visible)
    assert float((o.float() - want_o).abs().max()) <= 2e-2 and float((lse - want_lse).abs().max()) <= 2e-2
    for got, ref in zip(grads, want):
        assert rel_fro(got, ref) <= 1e-2
        # a row lost at the edge of a tile or part would drown in the norm of the whole
        err, n = (got.float() - ref).norm(dim=-1), ref.norm(dim=-1)
        assert float((err / n.clamp_min(float(n[n > 0].mean()))).max()) <= 4e-2
    again = tyr_amd.flash_attn_bwd(q, k, v, o, lse, g, **opt)
    assert all(torch.equal(a, b) for a, b in zip(grads, again))


@pytest.mark.parametrize("mask", ["causal", "full", "window", "lens", "keys"])
@pytest.mark.parametrize("B,Hq,Hkv,N,D", [(1, 1, 1, 33, 64), (1, 1, 1, 64, 128), (5, 3, 3, 77, 128), (1, 16, 16, 512, 64), (1, 8, 2, 1024, 128), (1, 8, 2, 1025, 64)])
def test_backward_in_one_launch_and_in_two(B, Hq, Hkv, N, D, mask):
    """dQ and dK/dV side by side (few workgroups), up to and beyond the last such length.  From 33 rows on: with a handful of
    keys dP and delta (of an O rounded to 2^-9) nearly cancel, and 1e-2 of what is left is less than that rounding."""
    test_every_launch_form_matches_the_f32_reference(B, Hq, Hkv, N, D, mask)


def padded_masks(N):
    """Key masks by what is hidden: nothing, either end across tile edges, both, all but one key, a hole of whole tiles, all."""
    i = torch.arange(N)
    return torch.stack([i >= 0, i >= 64, i >= min(63, N - 1), i >= min(65, N - 1), i >= N // 2, i < N - N // 3, (i >= N // 4) & (i < N - N // 4),
                        i == N - 1, i == 0, (i < 40) | (i >= N - 40), i < 0])


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("Hq,Hkv,N,D", [(1, 1, 3, 64), (2, 1, 65, 128), (4, 2, 130, 64), (4, 1, 700, 128), (16, 4, 700, 64), (2, 2, 1350, 128)])
def test_tiles_hidden_by_the_key_mask_are_skipped(Hq, Hkv, N, D, causal):
    import tyr_amd
    gen = torch.Generator(device="cuda").manual_seed(N + D)
    mask = padded_masks(N).cuda().contiguous()
    B = mask.shape[0]
    q, k, v, g = (torch.randn(B, h, N, D, device="cuda", generator=gen).bfloat16() for h in (Hq, Hkv, Hkv, Hq))
    i = torch.arange(N, device="cuda")
    visible = mask[:, None, None, :].expand(B, 1, N, N)
    if causal:
        visible = visible & (i[None, :] <= i[:, None])
    opt = dict(causal=causal, key_mask=mask)
    o, lse = tyr_amd.flash_attn_fwd(q, k, v, **opt)
    grads = tyr_amd.flash_attn_bwd(q, k, v, o, lse, g, **opt)

    rq, rk, rv = (t.float().requires_grad_() for t in (q, k, v))
    kk, vv = rk.repeat_interleave(Hq // Hkv, 1), rv.repeat_interleave(Hq // Hkv, 1)
    s = (torch.matmul(rq, kk.transpose(-1, -2).contiguous()) / math.sqrt(D)).masked_fill(~visible, -1e30)
    m = s.detach().amax(-1, keepdim=True)
    p = torch.exp(s - m) * visible
    total = p.sum(-1, keepdim=True)
    want_o = torch.matmul(p / total.clamp_min(1e-30), vv)
    seen = visible.any(-1).expand(B, Hq, N)
    want_lse = (m + torch.log(total)).squeeze(-1).detach()
    want = torch.autograd.grad(want_o, (rq, rk, rv), g.float())
    assert torch.equal(torch.isneginf(lse), ~seen) and not bool(o[~seen].any())
    assert float((o.float() - want_o).abs().max()) <= 2e-2
    assert float((lse - want_lse)[seen].abs().max()) <= 2e-2
    used = visible.any(-2).expand(B, Hkv, N)             # keys that some query sees
    for got, ref, alive in zip(grads, want, (seen, used, used)):
        assert rel_fro(got, ref) <= 1e-2
        assert not bool(got[~alive].any())


@pytest.mark.parametrize("mask", ["causal", "full", "window", "lens", "keys"])
@pytest.mark.parametrize("B,Hq,Hkv,N,D", [(1, 4, 1, 700, 128), (1, 8, 2, 1000, 64), (2, 16, 4, 1500, 128), (1, 8, 2, 2049, 64)])
def test_backward_with_the_least_workspace(B, Hq, Hkv, N, D, mask):
    """Shapes whose dK / dV are cut into parts where there is scratch for them (the first two beside dQ in one launch): with
    the minimum, and with all but 16 bytes of what parts need, whole key tiles run and nothing else of the buffer is touched."""
    from tyr_amd import _lib
    lib = _lib.load()
    gen = torch.Generator(device="cuda").manual_seed(N)
    q, k, v, g = (torch.randn(B, h, N, D, device="cuda", generator=gen).bfloat16() for h in (Hq, Hkv, Hkv, Hq))
    i = torch.arange(N, device="cuda")
    causal, window, lens, keys = int(mask != "full"), 0, None, None
    visible = (i[None, :] <= i[:, None] if causal else torch.ones(N, N, dtype=torch.bool, device="cuda"))[None, None].expand(B, 1, N, N)
    if mask == "window":
        window = N // 2 + 1
        visible = visible & (i[:, None] - i[None, :] < window)
    if mask == "lens":
        lens = torch.tensor([N - b * (N // (2 * B)) for b in range(B)], dtype=torch.int32, device="cuda")
        visible = visible & (i[None, None, None, :] < lens[:, None, None, None])
    if mask == "keys":
        keys = (torch.rand(B, N, device="cuda", generator=gen) > 0.3).to(torch.uint8)
        keys[:, 0] = 1
        visible = visible & (keys != 0)[:, None, None, :]
    want_o, want_lse, *want = reference(q, k, v, g, visible)
    o, lse = want_o.bfloat16(), want_lse.contiguous()
    least = lib.tyr_hip_flash_attn_bwd_workspace_bytes(B, Hq, N, D)
    full = lib.tyr_hip_flash_attn_bwd_parts_workspace_bytes(B, Hq, Hkv, N, D, causal, window)
    assert full > least
    buf = torch.empty(full + 4096, dtype=torch.uint8, device="cuda")
    results = []
    for nbytes in (least, full - 16, least, full):
        buf.fill_(0xA5)
        grads = [torch.full_like(t, float("nan")) for t in (q, k, v)]
        ptrs = [t.data_ptr() for t in (q, k, v, o, g, lse, *grads)]
        if keys is not None:
            rc = lib.tyr_hip_flash_attn_bwd_mask(*ptrs, B, Hq, Hkv, N, D, causal, keys.data_ptr(), D ** -0.5, buf.data_ptr(), nbytes,
                                                 torch.cuda.current_stream().cuda_stream)
        else:
            rc = lib.tyr_hip_flash_attn_bwd_gqa(*ptrs, B, Hq, Hkv, N, D, causal, window, lens.data_ptr() if lens is not None else None,
                                                D ** -0.5, buf.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream)
        assert rc == 0, lib.tyr_hip_strerror(rc)
        assert bool((buf[least if nbytes < full else full:] == 0xA5).all())
        results.append(grads)
    for other in results[1:3]:
        assert all(torch.equal(a, b) for a, b in zip(results[0], other))
    for got, ref, parts in zip(results[0], want, results[3]):
        assert rel_fro(got, ref) <= 1e-2
        # row by row against the parts: f32 sums of the same terms in another order, each rounded to bf16, i.e. elements one
        # unit apart at most (2^-8 of them; twice that allowed, and 1e-5 of a mean row where all terms cancel)
        n = parts.float().norm(dim=-1)
        assert bool(((got.float() - parts.float()).norm(dim=-1) <= 2 ** -7 * n + 1e-5 * n.mean()).all())


@pytest.mark.parametrize("mask", ["causal", "full", "window", "lens", "keys"])
@pytest.mark.parametrize("B,Hq,Hkv,N", [(4, 16, 4, 577), (4, 16, 4, 640), (4, 16, 16, 769), (2, 32, 8, 1153), (4, 8, 1, 1025), (9, 16, 4, 200), (4, 16, 4, 200)])
def test_backward_that_keeps_ds(B, Hq, Hkv, N, mask):
    """Few heads at D = 128, where dK / dV leave dS for dQ: rows one past a tile, whole tiles, whole and cut key tiles.  Hidden keys
    come first, in the middle (more than one block of 128) and last, with values that would outweigh every visible one."""
    import tyr_amd
    from tyr_amd import _lib
    lib, D = _lib.load(), 128
    gen = torch.Generator(device="cuda").manual_seed(N)
    q, k, v, g = (torch.randn(B, h, N, D, device="cuda", generator=gen).bfloat16() for h in (Hq, Hkv, Hkv, Hq))
    i = torch.arange(N, device="cuda")
    visible = (i[None, :] <= i[:, None] if mask != "full" else torch.ones(N, N, dtype=torch.bool, device="cuda"))[None, None].expand(B, 1, N, N)
    opt, window = dict(causal=mask != "full"), 0
    shown = torch.ones(B, N, dtype=torch.bool, device="cuda")
    if mask == "window":
        opt["window"] = window = N - 37
        visible = visible & (i[:, None] - i[None, :] < window)
    if mask == "lens":
        opt["kv_lens"] = torch.tensor(([N, 0, N // 2 + 1, 129] * B)[:B], dtype=torch.int32, device="cuda")
        shown = i[None, :] < opt["kv_lens"][:, None]
    if mask == "keys":
        shown = torch.rand(B, N, device="cuda", generator=gen) > 0.3
        shown[:, :70] = shown[:, 130:400] = shown[0, -140:] = shown[-1] = False
        opt["key_mask"] = shown
    visible = visible & shown[:, None, None, :]
    loud = torch.where(shown[:, None, :, None], 1.0, 300.0).bfloat16()
    k, v = k * loud, v * loud
    least = lib.tyr_hip_flash_attn_bwd_workspace_bytes(B, Hq, N, D)
    if (B, N, mask) != (9, 200, "window"):               # 64-key tiles, as fast (42.8 us, 42.9 with dS)
        assert lib.tyr_hip_flash_attn_bwd_full_workspace_bytes(B, Hq, Hkv, N, D, int(opt["causal"]), window) - least >= B * Hq * N * N
    o, lse = tyr_amd.flash_attn_fwd(q, k, v, **opt)
    grads = tyr_amd.flash_attn_bwd(q, k, v, o, lse, g, **opt)
    *_, wq, wk, wv = reference(q, k, v, g, visible)
    for got, ref in zip(grads, (wq, wk, wv)):
        assert rel_fro(got, ref) <= 1e-2
        err, n = (got.float() - ref).norm(dim=-1), ref.norm(dim=-1)
        # a dQ row with one heavy key takes delta's error whole: sum of g o r over D = 128, |r| <= 2^-8 the rounding of o, about
        # 0.4 * 2^-8 rms, so 11.3 * 0.0016 = 0.018 times |scale K| = 1; five such are 0.09, and a mean row is 1.2 or more
        assert float((err / n.clamp_min(float(n[n > 0].mean()))).max()) <= 8e-2
    assert all(torch.equal(a, b) for a, b in zip(grads, tyr_amd.flash_attn_bwd(q, k, v, o, lse, g, **opt)))
    # with the least scratch dQ makes dS itself, from the same bf16 operands: what may differ is the order of f32 sums, and
    # with it one rounding to bf16 (2^-8 of an element) here and there
    ws, plain = torch.empty(least, dtype=torch.uint8, device="cuda"), [torch.empty_like(t) for t in (q, k, v)]
    ptrs = [t.data_ptr() for t in (q, k, v, o, g, lse, *plain)]
    tail = (D ** -0.5, ws.data_ptr(), least, torch.cuda.current_stream().cuda_stream)
    if mask == "keys":
        rc = lib.tyr_hip_flash_attn_bwd_mask(*ptrs, B, Hq, Hkv, N, D, 1, opt["key_mask"].data_ptr(), *tail)
    else:
        lens = opt["kv_lens"].data_ptr() if mask == "lens" else None
        rc = lib.tyr_hip_flash_attn_bwd_gqa(*ptrs, B, Hq, Hkv, N, D, int(opt["causal"]), window, lens, *tail)
    assert rc == 0
    assert all(rel_fro(a, b.float()) <= 1e-3 for a, b in zip(grads, plain))


@pytest.mark.parametrize("lengths", [False, True])
@pytest.mark.parametrize("B,Hq,Hkv,N,window", [(2, 8, 1, 1029, 68), (5, 4, 4, 927, 102), (7, 4, 4, 708, 321), (7, 4, 4, 768, 257), (3, 32, 8, 850, 389), (1, 8, 2, 2079, 390)])
def test_kept_ds_of_a_narrow_window(B, Hq, Hkv, N, window, lengths):
    """dS where a query tile has places for a few key tiles only: windows below and above one tile, whole and cut key tiles, and with
    lengths (none, one row past a tile), whose hidden keys would outweigh every visible one."""
    import tyr_amd
    from tyr_amd import _lib
    lib, D = _lib.load(), 128
    gen = torch.Generator(device="cuda").manual_seed(N)
    q, k, v, g = (torch.randn(B, h, N, D, device="cuda", generator=gen).bfloat16() for h in (Hq, Hkv, Hkv, Hq))
    i = torch.arange(N, device="cuda")
    visible = ((i[None, :] <= i[:, None]) & (i[:, None] - i[None, :] < window))[None, None].expand(B, 1, N, N)
    opt = dict(causal=True, window=window)
    if lengths:
        opt["kv_lens"] = torch.tensor(([N // 2 + 1, N, 0, 129, N - 1] * B)[:B], dtype=torch.int32, device="cuda")
        shown = i[None, :] < opt["kv_lens"][:, None]
        visible = visible & shown[:, None, None, :]
        loud = torch.where(shown[:, None, :, None], 1.0, 300.0).bfloat16()
        k, v = k * loud, v * loud
    parts, full = (f(B, Hq, Hkv, N, D, 1, window) for f in (lib.tyr_hip_flash_attn_bwd_parts_workspace_bytes, lib.tyr_hip_flash_attn_bwd_full_workspace_bytes))
    assert full - parts >= B * Hq * N * min(window, N) * 2
    o, lse = tyr_amd.flash_attn_fwd(q, k, v, **opt)
    grads = tyr_amd.flash_attn_bwd(q, k, v, o, lse, g, **opt)
    *_, wq, wk, wv = reference(q, k, v, g, visible)
    seen, used = visible.any(-1).expand(B, Hq, N), visible.any(-2).expand(B, Hkv, N)
    for got, ref, alive in zip(grads, (wq, wk, wv), (seen, used, used)):
        assert rel_fro(got, ref) <= 1e-2
        err, n = (got.float() - ref).norm(dim=-1), ref.norm(dim=-1)
        assert float((err / n.clamp_min(float(n[n > 0].mean()))).max()) <= 8e-2         # as in test_backward_that_keeps_ds
        assert not bool(got[~alive].any())
    assert all(torch.equal(a, b) for a, b in zip(grads, tyr_amd.flash_attn_bwd(q, k, v, o, lse, g, **opt)))


@pytest.mark.parametrize("mask", ["causal", "full", "window", "lens", "keys"])
@pytest.mark.parametrize("B,Hq,Hkv,N,D", [(1, 1, 1, 1, 64), (2, 4, 4, 64, 128), (2, 4, 4, 65, 64), (3, 4, 4, 130, 128), (6, 4, 4, 263, 128), (2, 4, 4, 449, 64),
                                          (2, 8, 8, 685, 128), (9, 16, 4, 129, 128), (9, 8, 2, 193, 64), (6, 2, 1, 63, 128), (1, 2, 2, 2001, 64), (1, 4, 4, 2001, 64)])
def test_backward_of_64_key_tiles(B, Hq, Hkv, N, D, mask):
    """Small launches: one to 32 steps a tile, rows one past a tile, all heads of a group in one run; hidden keys that would
    outweigh every visible one, a whole tile of them among others, and a sequence without any key."""
    import tyr_amd
    from tyr_amd import _lib
    gen = torch.Generator(device="cuda").manual_seed(N + D)
    q, k, v, g = (torch.randn(B, h, N, D, device="cuda", generator=gen).bfloat16() for h in (Hq, Hkv, Hkv, Hq))
    i = torch.arange(N, device="cuda")
    visible = (i[None, :] <= i[:, None] if mask != "full" else torch.ones(N, N, dtype=torch.bool, device="cuda"))[None, None].expand(B, 1, N, N)
    opt = dict(causal=mask != "full")
    shown = torch.ones(B, N, dtype=torch.bool, device="cuda")
    if mask == "window":
        opt["window"] = N // 3 + 1
        visible = visible & (i[:, None] - i[None, :] < opt["window"])
    if mask == "lens":
        opt["kv_lens"] = torch.tensor(([N, 0, N // 2 + 1, N - 1] * B)[:B], dtype=torch.int32, device="cuda")
        shown = i[None, :] < opt["kv_lens"][:, None]
    if mask == "keys":
        shown = torch.rand(B, N, device="cuda", generator=gen) > 0.3
        shown[:, 60:130] = False
        opt["key_mask"] = shown
    visible = visible & shown[:, None, None, :]
    loud = torch.where(shown[:, None, :, None], 1.0, 300.0).bfloat16()
    k, v = k * loud, v * loud
    lib = _lib.load()
    full = lib.tyr_hip_flash_attn_bwd_full_workspace_bytes(B, Hq, Hkv, N, D, int(opt["causal"]), opt.get("window", 0))
    if (Hq, N) != (2, 2001) or mask in ("full", "window"):     # else key tiles in parts: 31.3 us causal, 37.3 with 64-key tiles
        assert full == lib.tyr_hip_flash_attn_bwd_workspace_bytes(B, Hq, N, D)      # no parts, no dS
    o, lse = tyr_amd.flash_attn_fwd(q, k, v, **opt)
    grads = tyr_amd.flash_attn_bwd(q, k, v, o, lse, g, **opt)
    *_, wq, wk, wv = reference(q, k, v, g, visible)
    for got, ref in zip(grads, (wq, wk, wv)):
        assert rel_fro(got, ref) <= 1e-2 or float(ref.norm()) == 0.0 and float(got.float().norm()) <= 1e-2
        err, n = (got.float() - ref).norm(dim=-1), ref.norm(dim=-1)
        if bool((n > 0).any()) and N >= 63:
            # as in test_backward_that_keeps_ds: 0.11 of sqrt(D / 128) against a mean row of 1.2 or more
            assert float((err / n.clamp_min(float(n[n > 0].mean()))).max()) <= 8e-2
    assert all(torch.equal(a, b) for a, b in zip(grads, tyr_amd.flash_attn_bwd(q, k, v, o, lse, g, **opt)))


def test_backward_without_memory_for_ds():
    """Where the full scratch cannot be had, the call runs with parts, and does not make the allocator empty its cache to find out."""
    import tyr_amd
    from tyr_amd import _lib
    lib = _lib.load()
    gen = torch.Generator(device="cuda").manual_seed(0)
    q, g = (torch.randn(1, 32, 2000, 128, device="cuda", generator=gen).bfloat16() for _ in range(2))
    k, v = (torch.randn(1, 8, 2000, 128, device="cuda", generator=gen).bfloat16() for _ in range(2))
    o, lse = tyr_amd.flash_attn_fwd(q, k, v, causal=True)
    want = tyr_amd.flash_attn_bwd(q, k, v, o, lse, g, causal=True)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.set_per_process_memory_fraction(torch.cuda.memory_reserved() / total)
    held, size = [], 1 << 30                 # what other tests left in the cache is not for this one
    while size >= 1 << 20:
        try:
            held.append(torch.empty(size, dtype=torch.uint8, device="cuda"))
        except torch.cuda.OutOfMemoryError:
            size >>= 1
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (96 << 20)) / total)
    before = torch.cuda.memory_stats()
    try:
        got = tyr_amd.flash_attn_bwd(q, k, v, o, lse, g, causal=True)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    after = torch.cuda.memory_stats()
    assert all(after[n] == before[n] for n in ("num_alloc_retries", "num_ooms", "num_device_free"))
    assert all(rel_fro(a, b.float()) <= 1e-3 for a, b in zip(got, want))
    parts = lib.tyr_hip_flash_attn_bwd_parts_workspace_bytes(1, 32, 8, 2000, 128, 1, 0)
    ws, cut = torch.empty(parts, dtype=torch.uint8, device="cuda"), [torch.empty_like(t) for t in (q, k, v)]
    assert 0 == lib.tyr_hip_flash_attn_bwd_gqa(*(t.data_ptr() for t in (q, k, v, o, g, lse, *cut)), 1, 32, 8, 2000, 128, 1, 0, None, 128 ** -0.5,
                                               ws.data_ptr(), parts, torch.cuda.current_stream().cuda_stream)
    assert all(torch.equal(a, b) for a, b in zip(got, cut))
