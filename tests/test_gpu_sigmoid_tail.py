"""The sigmoid of the short convolution and the gated norm where it is subnormal (arguments from -87.3 to -88.7),
against float64: what multiplies it can bring the result back into the normal range."""
import pytest
import torch

from gpu_util import gpu_or_skip, log
from lit_gpt.kdn_ops.gated_norm import rms_norm_gated
from lit_gpt.kdn_ops.short_conv import causal_conv1d, short_conv_step

pytestmark = pytest.mark.gpu

ARGS = [-86.0, -87.2, -87.5, -88.0, -88.6]
# the exponential's argument x log2(e) is rounded to 2^-24 of up to 128, so e^-x is off by up to 5.3e-6 and an ulp;
# a subnormal sigmoid of 3e-39 is rounded to 2^-149, 5e-7 of it
TOL = 1e-5


def _check(name, got, ref):
    err = float(((got.double().cpu() - ref).abs() / ref.abs()).max())
    log(f"  {name}: largest relative error {err:.2e}")
    assert err < TOL


def _sigmoid(x):
    return torch.exp(x) / (1 + torch.exp(x))


@pytest.mark.parametrize("activation", ["sigmoid", "swish"])
def test_gated_norm_tail(activation):
    dev = gpu_or_skip()
    log(f"case gated norm sigmoid tail {activation}")
    a = torch.tensor(ARGS, dtype=torch.float64)
    g = a.float()[:, None].expand(-1, 64).contiguous().to(dev).requires_grad_()
    x = torch.ones(len(ARGS), 64, device=dev)
    scale = 2.0 ** 60
    y = rms_norm_gated(x, g, torch.full((64,), scale, device=dev), activation=activation, eps=0.0)
    dg, = torch.autograd.grad(y, g, torch.ones_like(y))
    s = _sigmoid(a)
    act, grad = (s, s * (1 - s)) if activation == "sigmoid" else (a * s, s * (1 + a * (1 - s)))
    _check("y", y.detach()[:, 0], scale * act)
    _check("dg", dg[:, 0], scale * grad)


def test_short_convolution_tail():
    dev = gpu_or_skip()
    log("case short convolution sigmoid tail")
    a = torch.tensor(ARGS, dtype=torch.float64)
    x = a.float()[None, :, None].expand(1, -1, 8).contiguous().to(dev).requires_grad_()
    w = torch.zeros(8, 4, device=dev)
    w[:, 3] = 1.0
    s, scale = _sigmoid(a), 2.0 ** 60
    y, _ = causal_conv1d(x, w)
    _check("y", y.detach()[0, :, 0], a * s)
    dx, = torch.autograd.grad(y, x, torch.full_like(y, scale))
    _check("dx", dx[0, :, 0], scale * s * (1 + a * (1 - s)))
    steps = torch.stack([short_conv_step(x.detach()[:, i:i + 1].contiguous(), torch.zeros(1, 3, 8, device=dev), w)[0, 0, 0]
                         for i in range(len(ARGS))])
    _check("step", steps, a * s)
