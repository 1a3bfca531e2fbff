"""Chunk groups, whose intra-chunk build forms U = A V for the state passes: every head width, a ragged last chunk, a
first-group and a later chunk on the exact path and one on the block anchors, against the float64 token-wise oracle;
the same output and final state with and without a backward to follow (without one A is not written)."""
import pytest
import torch

from gpu_util import chunk_prefix_base2, gpu_or_skip, log, memory_inputs
from oracle import kdn_oracle as ko
from test_gpu_memory import TOL_F32, _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant", ["iso", "diag"])
@pytest.mark.parametrize("B,T,H,K,V", [(1, 1041, 1, 128, 128), (2, 1100, 1, 64, 64), (1, 1087, 2, 128, 64), (1, 1024, 1, 64, 128)])
def test_grouped_scan_with_flagged_chunks(variant, B, T, H, K, V):
    dev = gpu_or_skip()
    from lit_gpt.kdn_ops import _memscan
    iso = variant == "iso"
    log(f"case grouped scan {variant} B={B} T={T} H={H} K={K} V={V}")
    assert _memscan.state_groups(B, T, H, K, V) > 1
    q, k, v, ell, kap, _ = memory_inputs(7 + T + K, B, T, H, K, V, diag=not iso)
    for t in (70, T - 130):  # 25 tokens at e^-12: the exact path
        ell[:, t:t + 25, :, :6] = -12.0
    ell[:, 400:440, :, :6] = -4.0  # 58 to 104 bits per block, over 200 per chunk: the block anchors
    h0 = 0.1 * torch.randn(B, H, K, V, generator=torch.Generator().manual_seed(T))
    scale = K ** -0.5
    qd, kd, kapd = q.double(), k.double(), kap.double()
    o_ref, s_ref = ko.memory_tokenwise(qd, kd, v.double(), ell.double().exp(), kapd[..., None] * kd if iso else kapd,
                                       scale=scale, initial_state=h0.double())
    G = chunk_prefix_base2(ell, 64).float()
    args = [x.to(dev).contiguous() for x in (q, k, kap.float())] + [iso] + [x.to(dev).contiguous() for x in (v, G)]
    runs = [_memscan.mem_fwd(*args, scale, initial_state=h0.to(dev), output_final_state=True, need_backward=nb)
            for nb in (True, False)]
    for o, _, s in runs:
        _check("o", o, o_ref, TOL_F32)
        _check("final state", s, s_ref, TOL_F32)
    assert torch.equal(runs[0][0], runs[1][0]) and torch.equal(runs[0][2], runs[1][2])
