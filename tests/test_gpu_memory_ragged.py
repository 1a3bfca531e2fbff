"""Memory scan forward and backward where the last chunk is ragged at the edges of the 16-row tiles
(the state passes stage v and dO rows, and copy delta and dX, in whole tiles), against the float64
token-wise oracle; and a scan long enough for the state pass without readout (several chunk groups)."""
import pytest

from gpu_util import gpu_or_skip, log, memory_inputs
from test_gpu_memory import TOL_BF16, TOL_F32, _check, _gpu, _oracle, _tol_grad

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant", ["iso", "diag"])
@pytest.mark.parametrize("B,T,H,d", [(1, 15, 1, 64), (1, 16, 2, 128), (2, 17, 1, 128), (1, 49, 1, 64), (1, 63, 2, 128),
                                     (1, 65, 1, 128), (2, 127, 1, 64), (1, 1041, 1, 128)])
def test_ragged_last_chunk(variant, B, T, H, d):
    dev = gpu_or_skip()
    log(f"case memory ragged {variant} B={B} T={T} H={H} d={d}")
    iso = variant == "iso"
    q, k, v, ell, kap, do = memory_inputs(29 + T + d, B, T, H, d, d, diag=not iso)
    scale = d ** -0.5
    o_ref, _, g_ref = _oracle(q, k, v, ell, kap, do, iso=iso, scale=scale)
    o, _, dq, dkk, dv, dell, dkap, _ = _gpu(q, k, v, ell, kap, do, iso=iso, scale=scale, dev=dev)
    _check("o", o, o_ref, TOL_F32)
    _check("dq", dq, g_ref[0], TOL_BF16)
    _check("dk", dkk, g_ref[1], TOL_BF16)
    _check("dv", dv, g_ref[2], TOL_BF16)
    _check("dgate", dell, g_ref[3], _tol_grad(iso, q, v))
    _check("dbeta" if iso else "dkappa", dkap, g_ref[4], _tol_grad(iso, q, v))
