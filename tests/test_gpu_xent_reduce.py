"""The cross-entropy module's sum and mean in one kernel against the per-row losses reduced in float64, with
the gradient, on both sides of the row limit and with every row ignored."""
import pytest
import torch

from gpu_util import gpu_or_skip, log
from lit_gpt import fused_cross_entropy as fce

pytestmark = pytest.mark.gpu


# the sums run in float64: the losses' own f32 rounding (2^-23) and one division
@pytest.mark.parametrize("reduction", ["mean", "sum"])
@pytest.mark.parametrize("n,dtype", [(1, torch.int64), (63, torch.int32), (1025, torch.int64), (65536, torch.int32),
                                     (65537, torch.int64)])
def test_reduction_matches_float64(reduction, n, dtype):
    dev = gpu_or_skip()
    log(f"case xent reduce n={n} {reduction} {dtype}")
    g = torch.Generator().manual_seed(n)
    x = torch.randn(n, 40, generator=g).to(dev).requires_grad_()
    y = torch.randint(0, 40, (n,), generator=g).to(dtype)
    y[1::7] = -100
    y = y.to(dev)
    kw = dict(label_smoothing=0.1, lse_square_scale=1e-3)
    losses, z = fce.cross_entropy_loss(x, y, **kw)
    div = int((y != -100).sum()) if reduction == "mean" else 1
    loss, z_loss = fce.FusedCrossEntropyLoss(reduction=reduction, return_z_loss=True, **kw)(x, y)
    assert abs(float(loss) - float(losses.double().sum() / div)) <= 2e-6 * abs(float(loss))
    assert abs(float(z_loss) - float(z.double().sum() / div)) <= 2e-6 * abs(float(z_loss))
    want = torch.autograd.grad(losses, x, torch.full_like(losses, 3.0 / div))[0]
    loss *= 3  # an output that may be scaled in place, as gradient accumulation does
    got = torch.autograd.grad(loss, x)[0]
    assert float((got - want).abs().max()) <= 1e-6 * float(want.abs().max())


def test_mean_of_no_rows_is_nan_with_zero_gradient():
    dev = gpu_or_skip()
    x = torch.randn(5, 33, device=dev, requires_grad=True)
    loss = fce.FusedCrossEntropyLoss()(x, torch.full((5,), -100, device=dev))
    assert torch.isnan(loss)
    assert float(torch.autograd.grad(loss, x)[0].abs().max()) == 0
