"""Backward with dK / dV by key tiles of 256 (launches of many whole tiles): lengths around its 64-row query tiles, 64-key waves and
256-key tiles, grouped queries, head counts that are no multiple of the XCDs, every mask; and by tiles of 64 where two workgroups share
a CU.  Four (sequence, kv head) pairs of each launch against float64 gradients of the bf16 inputs, the last one among them: its rows end
where Q and dO do, and the memory behind those holds NaN.  Bounds as in test_gpu_attention_bwd."""
import pytest
import torch

from tests.util import rel_fro

pytestmark = pytest.mark.gpu


def reference(q, k, v, g, visible):
    """float64 dQ, dK, dV of the G query heads [G, N, D] of one kv head [N, D]."""
    q, k, v, g = (x.double() for x in (q, k, v, g))
    scale = q.shape[-1] ** -0.5
    p = torch.softmax((q @ k.T * scale).masked_fill(~visible, float("-inf")), -1).nan_to_num(0.0)
    dp = g @ v.T
    ds = p * (dp - (p * dp).sum(-1, keepdim=True)) * scale
    return ds @ k, sum(d.T @ x for d, x in zip(ds, q)), sum(d.T @ x for d, x in zip(p, g))


FIELDS = "B,Hq,Hkv,N,D,causal,mask,window"
# test_host_launches checks that these take the kernels they are here for
WIDE = [
    (16, 32, 8, 1025, 128, True, None, 0), (16, 32, 8, 1279, 128, True, None, 0), (16, 32, 32, 960, 128, True, None, 0),
    (16, 32, 8, 513, 64, True, None, 0), (16, 32, 32, 768, 64, True, None, 0),
    (16, 32, 8, 449, 128, False, None, 0), (16, 32, 8, 512, 128, False, None, 0), (17, 12, 4, 513, 64, False, None, 0),
    (16, 32, 8, 1100, 128, True, "lens", 0), (17, 12, 4, 600, 64, False, "lens", 0), (16, 32, 8, 500, 128, False, "lens", 0),
    (16, 32, 8, 1100, 128, True, "keys", 0), (17, 12, 4, 600, 64, False, "keys", 0), (16, 32, 8, 700, 64, True, "keys", 0),
    (16, 32, 8, 1216, 128, True, None, 600), (16, 32, 8, 1153, 128, True, "lens", 600),
    # causal, kv heads that are no multiple of the XCDs (60, 90, 44), or no multiple of eight on each (14, 15): the order's last group of
    # heads is a part of one
    (15, 12, 4, 1160, 128, True, None, 0), (15, 18, 6, 929, 128, True, "keys", 0), (11, 12, 4, 1400, 64, True, None, 0),
    (14, 32, 8, 681, 128, True, "lens", 0), (15, 16, 8, 1100, 64, True, None, 0)]
TWO_A_CU = [
    (16, 8, 8, 130, 64, False, None, 0), (6, 8, 8, 320, 64, False, "lens", 0), (8, 16, 4, 385, 64, False, "keys", 0),
    (3, 16, 16, 283, 64, True, None, 70), (5, 16, 4, 511, 64, True, "lens", 100), (2, 4, 4, 1400, 64, True, None, 129)]


@pytest.mark.parametrize(FIELDS, WIDE)
def test_wide_key_tiles_match_float64(B, Hq, Hkv, N, D, causal, mask, window):
    compare(B, Hq, Hkv, N, D, causal, mask, window)


@pytest.mark.parametrize(FIELDS, TWO_A_CU)
def test_two_workgroups_of_64_key_tiles_on_a_cu(B, Hq, Hkv, N, D, causal, mask, window):
    compare(B, Hq, Hkv, N, D, causal, mask, window)


def before_nan(x):
    """The same values in front of 64 KB that read as NaN, in one allocation."""
    room = torch.full((x.numel() + 32768,), float("nan"), dtype=x.dtype, device=x.device)
    room[:x.numel()] = x.flatten()
    return room[:x.numel()].view(x.shape)


def compare(B, Hq, Hkv, N, D, causal, mask, window):
    import tyr_amd
    gen = torch.Generator(device="cuda").manual_seed(N + D)
    q, g = (before_nan(torch.randn(B, Hq, N, D, generator=gen, device="cuda").bfloat16()) for _ in range(2))
    k, v = (torch.randn(B, Hkv, N, D, generator=gen, device="cuda").bfloat16() for _ in range(2))
    opt = dict(causal=causal)
    i = torch.arange(N, device="cuda")
    visible = (i[None, :] <= i[:, None]) if causal else torch.ones(N, N, dtype=torch.bool, device="cuda")
    keys = torch.ones(B, N, dtype=torch.bool, device="cuda")
    if mask == "lens":
        lens = torch.tensor([(N, 257, 1, 0, 64, 320)[b % 6] for b in range(B)], dtype=torch.int32, device="cuda")
        keys = i[None, :] < lens[:, None]
        opt["kv_lens"] = lens
    elif mask == "keys":
        keys = torch.rand(B, N, generator=gen, device="cuda") < 0.6
        keys[:, 100:300] = False
        keys[1::3, :270] = False
        opt["key_mask"] = keys
    if window:
        visible = visible & (i[:, None] - i[None, :] < window)
        opt["window"] = window
    o, lse = tyr_amd.flash_attn_fwd(q, k, v, **opt)
    got = tyr_amd.flash_attn_bwd(q, k, v, o, lse, g, **opt)
    G = Hq // Hkv
    for b, h in ((0, 0), (1, Hkv - 1), (B - 2, 1), (B - 1, Hkv - 1)):
        want = reference(q[b, h * G:(h + 1) * G], k[b, h], v[b, h], g[b, h * G:(h + 1) * G], visible & keys[b][None, :])
        for name, x, y in zip(("dq", "dk", "dv"), (got[0][b, h * G:(h + 1) * G], got[1][b, h], got[2][b, h]), want):
            assert bool(((x.double() - y).abs() <= 3e-2 + 3e-2 * y.abs()).all()), (name, b, h)
            if float(y.norm()) > 1e-3:
                assert rel_fro(x.cpu().float(), y.cpu()) <= 1e-2, (name, b, h, rel_fro(x.cpu().float(), y.cpu()))
        assert not bool(got[1][b, h][~keys[b]].any()) and not bool(got[2][b, h][~keys[b]].any())
