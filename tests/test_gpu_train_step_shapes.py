"""The element-wise train-step kernels where their work is cut: a wave's two runs of 256 elements, the largest size one
workgroup takes and the next, partial sums that are not a multiple of the four a lane loads, more than it loads at once."""
import numpy as np
import pytest
import torch

from oracle import libtorch_path as lt
from tests.util import bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [8, 248, 256, 264, 512, 520, 2040, 2056, 8192, 8200, 32760, 32768, 32776, 2048 * 19, 2048 * 4100 * 4 + 2048 * 3 + 8])
def test_elementwise_sizes(n):
    import tyr_amd
    out, target = lt.make_inputs(n % 1000, (n,), (n,))
    loss, d_o = tyr_amd.mse_loss_grad(out.cuda(), target.cuda())
    want_loss, want_d = lt.loss_and_grad_out(out, target)
    assert np.array_equal(bits(d_o), bits(want_d))
    exact = 0.5 * float(((out.float() - target.float()).double() ** 2).mean())
    assert abs(float(loss) - exact) <= 1e-6 * exact
    param = torch.randn(n, generator=torch.Generator().manual_seed(n))
    new, low = tyr_amd.sgd_step(param.cuda(), out.cuda(), 0.37)
    want = lt.sgd_update(param, out, 0.37)
    assert np.array_equal(new.cpu().numpy().view(np.uint32), want.numpy().view(np.uint32))
    assert np.array_equal(bits(low), bits(want.to(torch.bfloat16)))
