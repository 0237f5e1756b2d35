"""Row kernels where their launch changes: how many waves share a LayerNorm row, rows that do not fill a workgroup, and the
size from which a launch streams past the last-level cache (its results equal those of the same rows in smaller launches)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 2, 3, 5])
@pytest.mark.parametrize("d", [8, 504, 512, 520, 1016, 1024, 1032, 1536, 2048, 2056, 3000, 4096, 4104, 5000, 8192])
def test_layernorm_row_lengths(rows, d):
    import tyr_amd
    g = torch.Generator(device="cuda").manual_seed(rows * 10007 + d)
    x, r = (torch.randn(rows, d, generator=g, device="cuda").bfloat16() for _ in range(2))
    x += 3.0                                            # a mean to cancel
    w, b = (torch.randn(d, generator=g, device="cuda").bfloat16() for _ in range(2))
    out, resid = tyr_amd.layernorm_residual(x, r, w, b)
    want_r = (x.float() + r.float()).bfloat16()
    assert torch.equal(resid, want_r)
    want = torch.nn.functional.layer_norm(want_r.double(), (d,), w.double(), b.double(), 1e-5)
    assert float((out.double() - want).abs().max()) <= 2.0 ** -7 * max(1.0, float(want.abs().max()))


def test_streaming_launches_equal_smaller_ones():
    import tyr_amd
    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn(1, 5200, 64, 128, generator=g, device="cuda").bfloat16()         # 85 MB in, 85 MB out
    c, s = (torch.randn(5200, 64, generator=g, device="cuda") for _ in range(2))
    assert torch.equal(tyr_amd.rope_fwd(x, c, s)[:, :700], tyr_amd.rope_fwd(x[:, :700].contiguous(), c[:700].contiguous(), s[:700].contiguous()))
    assert torch.equal(tyr_amd.copy(x), x)
    flat = x.view(-1, 4096)
    w = torch.randn(4096, generator=g, device="cuda").bfloat16()
    for whole, part in zip(tyr_amd.layernorm_residual(flat, flat, w, w), tyr_amd.layernorm_residual(flat[-9:].contiguous(), flat[-9:].contiguous(), w, w)):
        assert torch.equal(whole[-9:], part)
    p = torch.randn(x.shape, generator=g, device="cuda")
    for whole, part in zip(tyr_amd.sgd_step(p, x, 0.3), tyr_amd.sgd_step(p[:, -8:].contiguous(), x[:, -8:].contiguous(), 0.3)):
        assert torch.equal(whole[:, -8:], part)
    loss, d_o = tyr_amd.mse_loss_grad(x, x.flip(1))
    diff = x.float() - x.flip(1).float()
    assert torch.equal(d_o, (diff / diff.numel()).bfloat16())
    assert abs(float(loss) - 0.5 * float((diff.double() ** 2).mean())) <= 1e-6 * float(loss)
