"""``kdn_decode_mixer`` against the float64 oracle: convolution, gate frontends, Kalman gain, memory and gated norm
of one token, with strong decays (below the diagonal memory path's floor of 1e-6), omega_min > 0, r_min and
info_scale off their defaults, head counts whose packed rows need padding, and rows further apart than they are wide."""
import math

import pytest
import torch

from gpu_util import gpu_or_skip, log, rel
from lit_gpt.kdn_ops.step import kdn_decode_mixer
from oracle import kdn_oracle as ko

pytestmark = pytest.mark.gpu


def _step64(p, off, tails, taps, Wf, Wo, bo, Wg, bg, ob, rb, A_log, dt, *, omega_min, r_min, info_scale, precision, memory,
            nw, eps, iso):
    """One token in float64 -> y, tails, precision, memory."""
    B, H, K, _ = memory.shape
    n = H * K
    f, w, r, g = off
    d = lambda t: None if t is None else t.double()  # noqa: E731
    p, memory, precision = d(p), d(memory), d(precision)
    tail = torch.cat([d(t) for t in tails], -1)  # [B,3,3n]
    seq = torch.cat([tail, p[:, None, :3 * n]], 1)
    q, k, v = (t.reshape(B, 1, H, K) for t in ko.short_conv_silu(seq, torch.cat([d(t) for t in taps], 0))[:, 3:].split(n, -1))
    heads = lambda t: t.reshape(B, 1, H, K)  # noqa: E731
    g_raw, gate = p[:, f:f + K] @ d(Wf).T, p[:, g:g + K] @ d(Wg).T + (d(bg) if bg is not None else 0)
    mu = torch.zeros(H, dtype=torch.float64)
    if iso:
        gl, _, a, omega, rr, _ = ko.iso_gate_frontend(heads(g_raw), p[:, None, r:r + 2 * H], d(ob), d(rb), d(A_log), d(dt), mu,
                                                      omega_min=omega_min, r_min=r_min)
        q, k = ko.l2norm_fla(q), ko.l2norm_fla(k)
        beta, prec = ko.iso_gain_unit_key(a, omega, rr, precision, posterior_scale=info_scale / K, output_final_state=True)
        kappa = beta[..., None] * k
    else:
        omega_raw = p[:, w:w + K] @ d(Wo).T + (d(bo) if bo is not None else 0)
        gl, _, alpha, omega, _, _ = ko.diag_frontend(heads(g_raw), heads(omega_raw), p[:, None, r:r + H], d(A_log), d(dt), mu)
        q, k = ko.diag_normalize(q), ko.diag_normalize(k)
        kappa, prec = ko.diag_gain_tokenwise(k, alpha, omega, r_min + ko.softplus(p[:, None, r:r + H]), info_scale=info_scale,
                                             initial_precision=precision, output_final_state=True)
    o, S = ko.memory_tokenwise(q, k, v, gl.exp(), kappa, scale=K ** -0.5, initial_state=memory)
    y = ko.rms_norm_gated(o, heads(gate), d(nw), eps=eps)
    return y.reshape(B, n), seq[:, 1:], prec, S


@pytest.mark.parametrize("iso", [True, False])
@pytest.mark.parametrize("B,H,K,strong,bias", [(1, 18, 128, False, True), (3, 5, 64, True, True), (2, 1, 128, True, False),
                                               (17, 4, 64, False, False), (5, 18, 64, True, True)])
def test_mixer_step_matches_float64(iso, B, H, K, strong, bias):
    dev = gpu_or_skip()
    log(f"case decode_mixer iso={iso} B={B} H={H} K={K} strong={strong} bias={bias}")
    gen = torch.Generator().manual_seed(B + 7 * H + K + iso)
    n = H * K

    def rnd(*s, scale=1.0, dtype=torch.bfloat16):
        return (scale * torch.randn(*s, generator=gen)).to(dtype)

    if iso:
        off, width = (3 * n, 0, 3 * n + K, 3 * n + K + 2 * H), 3 * n + 2 * K + 2 * H
    else:
        off, width = (3 * n, 3 * n + K, 3 * n + 3 * K, 3 * n + 2 * K), 3 * n + 3 * K + H
    rows = rnd(B, width + 13)
    p = rows[:, :width + 5]
    tails = [rnd(B, 3, 3 * n)] if iso else [rnd(B, 3, n) for _ in range(3)]
    taps = [rnd(3 * n, 4, scale=0.5)] if iso else [rnd(n, 4, scale=0.5) for _ in range(3)]
    # strong: -ell = 16 softplus(N(0, 2)) for most heads, from near 0 far past the floor at 13.8
    Wf, Wg = rnd(n, K, scale=(2.0 if strong else 1.0) * K ** -0.5), rnd(n, K, scale=K ** -0.5)
    Wo = None if iso else rnd(n, K, scale=K ** -0.5)
    bg, bo = (rnd(n) if bias else None), (rnd(n) if bias and not iso else None)
    ob, rb = (rnd(H, dtype=torch.float32), rnd(H, dtype=torch.float32)) if iso else (None, None)
    A_log = torch.full((H,), math.log(16.0 if strong else 0.3))
    A_log[0] = math.log(0.3)
    dt = rnd(n, scale=0.3, dtype=torch.float32)
    precision = 0.5 + 2 * torch.rand(B, H, *(() if iso else (K,)), generator=gen)
    memory, nw = rnd(B, H, K, K, dtype=torch.float32), (1 + 0.1 * torch.randn(K, generator=gen)).bfloat16()
    kw = dict(omega_min=0.07 if iso else 0.0, r_min=0.05, info_scale=0.3 * K, eps=1e-5, iso=iso)
    args = (p, off, tails, taps, Wf, Wo, bo, Wg, bg, ob, rb, A_log, dt)
    y_ref, seq, prec_ref, s_ref = _step64(*args, precision=precision, memory=memory, nw=nw, **kw)

    def to(t):
        return [to(x) for x in t] if isinstance(t, list) else t.to(dev) if isinstance(t, torch.Tensor) else t

    gargs = [to(a) for a in args]
    gargs[0] = to(rows)[:, :width + 5]
    gt, gp, gm = tuple(gargs[2]), to(precision), to(memory)
    gargs[2], gargs[3] = gt, tuple(gargs[3])
    y = kdn_decode_mixer(*gargs, precision=gp, memory=gm, norm_weight=to(nw), **kw)
    assert torch.equal(torch.cat([t.double().cpu() for t in gt], -1), seq)  # moved, not computed
    # nothing is rounded to 16 bits inside.  The largest error of a precision is its omega's: softplus = log(1 + y) from
    # y = 1e-3 on, 2^-24 / 1e-3 = 6e-5 of the value at worst; the memory's entries are of order 1 and take part of it
    e_p = float(((gp.double().cpu() - prec_ref) / prec_ref).abs().max())
    e_s = rel(gm, s_ref)
    log(f"  precision {e_p:.2e} memory {e_s:.2e} y {rel(y.float(), y_ref):.2e}")
    assert e_p < 1e-4 and e_s < 1e-5
    assert rel(y.float(), y_ref) < 4e-3  # one rounding to bf16, 2^-8 of the largest
