"""The short convolution's walk in runs of 8 to 32 tokens (groups of 4 rows, wave-uniform edges): run and
block edges, channel counts that leave lanes idle, a missing gradient, against float64; and the packed
q|k|v launch against three single-group launches."""
import pytest
import torch
import torch.nn.functional as F

from gpu_util import gpu_or_skip, log, rel
from lit_gpt.kdn_ops.short_conv import causal_conv1d, qkv_causal_conv1d

pytestmark = pytest.mark.gpu


def _ref(x, w):  # float64 [B,T,D], [D,4]
    return F.silu(F.conv1d(F.pad(x.transpose(1, 2), (3, 0)), w[:, None], groups=w.shape[0])).transpose(1, 2)


# a bf16 result is within 2^-9 of its value; in f32 the exponential (2^-22) and 4-term sums are below 1e-6,
# the weight gradient's sums of up to T terms below 1e-5; the packed bf16 backward rounds the preactivation
# (2^-9 of it, through silu'' <= 0.5) and its results
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,T,D", [(1, 1, 8), (2, 3, 72), (1, 4, 256), (1, 7, 264), (2, 33, 64), (1, 129, 520),
                                   (4, 1027, 1544), (2, 4099, 8)])
def test_packed_and_single_convolution(dtype, B, T, D):
    dev = gpu_or_skip()
    log(f"case conv B={B} T={T} D={D} {dtype}")
    g = torch.Generator().manual_seed(B + T + D)
    x = torch.randn(B, T, 3 * D, generator=g).to(dtype)
    w = (0.5 * torch.randn(3 * D, 4, generator=g)).to(dtype)
    dy = [torch.randn(B, T, D, generator=g).to(dtype) for _ in range(2)] + [None]
    x64, w64 = x.double().requires_grad_(), w.double().requires_grad_()
    ys = _ref(x64, w64).split(D, -1)
    dx64, dw64 = torch.autograd.grad(sum((y * d.double()).sum() for y, d in zip(ys, dy) if d is not None), (x64, w64))

    xg, wg = x.to(dev).requires_grad_(), w.to(dev).requires_grad_()
    out = qkv_causal_conv1d(xg, wg)
    dx, dw = torch.autograd.grad([o for o, d in zip(out, dy) if d is not None], (xg, wg),
                                 [d.to(dev) for d in dy if d is not None])
    tol = 1e-5 if dtype == torch.float32 else 6e-3
    for y, o in zip(ys, out):
        assert rel(o.float().cpu(), y) < tol
    assert rel(dx.float().cpu(), dx64) < tol and rel(dw.float().cpu(), dw64) < tol
    assert float(dx[..., 2 * D:].abs().max()) == 0 and float(dw[2 * D:].abs().max()) == 0

    for i in range(2):
        xi = xg.detach()[..., i * D:(i + 1) * D].requires_grad_()
        wi = wg.detach()[i * D:(i + 1) * D].requires_grad_()
        yi, _ = causal_conv1d(xi, wi)
        assert torch.equal(yi, out[i])
        dxi, dwi = torch.autograd.grad(yi, (xi, wi), dy[i].to(dev))
        if dtype == torch.float32:  # no rounding of the preactivation in either: only the run length may differ
            assert torch.equal(dxi, dx[..., i * D:(i + 1) * D])
        assert rel(dwi.float().cpu(), dw64[i * D:(i + 1) * D]) < tol
