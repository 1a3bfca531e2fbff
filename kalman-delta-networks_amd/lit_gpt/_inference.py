"""Inference-time caches for the decode path (no autograd).

A decode step runs one token through every block, so every separate small GEMM and dtype cast
is one more launch.  Projections that read the same input are packed into one weight, and the
small gate parameters' fp32 copies are kept, both cached on the owning module and rebuilt when a
source tensor's storage or version changes (``load_state_dict``, an optimiser step, ``.to()``).
The caches are plain attributes, not buffers, so they never enter a state dict.

Memory cost: a packed weight is a second copy of the packed projections (at iso_kdn_1.3B in bf16,
about 33 MB of input projections and 66 MB of SwiGLU w1|w2 per layer, 1.8 GB over 18 layers).  Packing
is therefore limited to modules in eval mode (``module.training`` False) under no_grad, and
``clear_inference_caches(model)`` drops every cache of a model.
"""
from __future__ import annotations

import torch
import torch.nn.functional as F

# at most this many rows (B * T) take the packed projections: the launch-bound decode regime;
# longer inputs keep the separate GEMMs, whose outputs are contiguous
PACK_MAX_ROWS = 64
# at most this many rows with bf16 activations and weights go through the weight-streaming GEMV
GEMV_MAX_ROWS = 8


def use_packed(x: torch.Tensor, module: torch.nn.Module) -> bool:
    """The packed-projection path: no autograd, ``module`` in eval mode, at most PACK_MAX_ROWS rows."""
    return not torch.is_grad_enabled() and not module.training and x.numel() // x.shape[-1] <= PACK_MAX_ROWS


def clear_inference_caches(model: torch.nn.Module) -> None:
    """Drop the packed weights and fp32 parameter copies cached on ``model``'s modules."""
    for m in model.modules():
        m.__dict__.pop("_kdn_inference_cache", None)


def _key(tensors):
    return tuple((t.data_ptr(), t._version, t.dtype, t.device) for t in tensors)


def packed_weight(owner, name: str, tensors, row_multiple: int = 1) -> torch.Tensor:
    """torch.cat(tensors, 0) followed by zero rows up to a multiple of ``row_multiple`` rows (so the
    packed product's rows start on aligned addresses), cached on ``owner`` under ``name``."""
    cache = owner.__dict__.setdefault("_kdn_inference_cache", {})
    key = (_key(tensors), row_multiple)
    hit = cache.get(name)
    if hit is None or hit[0] != key:
        parts = [t.detach() for t in tensors]
        rows = sum(t.shape[0] for t in parts)
        pad = (-rows) % row_multiple
        if pad:
            parts.append(parts[0].new_zeros((pad,) + tuple(parts[0].shape[1:])))
        hit = (key, torch.cat(parts, 0))
        cache[name] = hit
    return hit[1]


def packed_bias(owner, name: str, parts) -> torch.Tensor:
    """A packed product's bias, cached on ``owner``: ``parts`` are tensors, or row counts for zeros."""
    cache = owner.__dict__.setdefault("_kdn_inference_cache", {})
    key = (_key([t for t in parts if not isinstance(t, int)]), tuple(t for t in parts if isinstance(t, int)))
    hit = cache.get(name)
    if hit is None or hit[0] != key:
        like = next(t for t in parts if not isinstance(t, int)).detach()
        hit = (key, torch.cat([like.new_zeros(t) if isinstance(t, int) else t.detach() for t in parts]))
        cache[name] = hit
    return hit[1]


def as_f32(owner, name: str, t: torch.Tensor) -> torch.Tensor:
    """``t.float()``; under no_grad the converted copy of a non-fp32 tensor is cached on ``owner``."""
    if t.dtype == torch.float32 or torch.is_grad_enabled():
        return t.float()
    cache = owner.__dict__.setdefault("_kdn_inference_cache", {})
    key = _key((t,))
    hit = cache.get(name)
    if hit is None or hit[0] != key:
        hit = (key, t.detach().float())
        cache[name] = hit
    return hit[1]


def _gemv_ok(x, weight, bias) -> bool:
    return (not torch.is_grad_enabled() and x.is_cuda and x.dtype == torch.bfloat16 and weight.dtype == torch.bfloat16
            and (bias is None or bias.dtype == torch.bfloat16) and x.shape[-1] % 8 == 0 and weight.is_contiguous()
            and x.numel() // max(x.shape[-1], 1) <= GEMV_MAX_ROWS
            and not torch.is_autocast_enabled("cuda"))


def linear(x: torch.Tensor, weight: torch.Tensor, bias=None) -> torch.Tensor:
    """``F.linear``; a no-grad call of at most ``GEMV_MAX_ROWS`` rows with bf16 activations, weight
    and bias (the one-token decode step of a bf16 model) reads the weight through ``kdn_gemv``
    instead of a small-M GEMM."""
    if _gemv_ok(x, weight, bias):
        from .kdn_ops.step import kdn_gemv
        return kdn_gemv(x, weight, bias)
    return F.linear(x, weight, bias)


def swiglu_gate(x: torch.Tensor, w12: torch.Tensor) -> torch.Tensor:
    """silu(x w1^T) * (x w2^T) for a packed ``w12`` = [w1; w2]; in the decode regime of ``linear``
    one ``kdn_gemv`` launch computes both products and the gate."""
    if _gemv_ok(x, w12, None) and w12.shape[0] % 2 == 0:
        from .kdn_ops.step import kdn_gemv
        return kdn_gemv(x, w12, None, gated=True)
    h1, h2 = linear(x, w12).chunk(2, dim=-1)
    return F.silu(h1) * h2


def _plain(module) -> bool:
    """No hook sits on ``module`` or below it, so its parts need not be called one by one."""
    from torch.nn.modules import module as M
    if M._global_forward_hooks or M._global_forward_pre_hooks:
        return False
    return not any(m._forward_hooks or m._forward_pre_hooks or "forward" in m.__dict__ for m in module.modules())


def _decode_rows(x, module) -> bool:
    return (not torch.is_grad_enabled() and not module.training and x.is_cuda and x.dtype == torch.bfloat16 and x.ndim == 3
            and x.shape[1] == 1 and 0 < x.shape[0] <= PACK_MAX_ROWS and x.shape[-1] % 8 == 0 and x.is_contiguous()
            and not torch.is_autocast_enabled("cuda"))


def _bf16_dense(*params) -> bool:
    return all(p is None or (p.dtype == torch.bfloat16 and p.is_contiguous() and p.is_cuda and p.data_ptr() % 16 == 0)
               for p in params)


# kdn_decode_proj keeps x in registers up to this K (8 waves x 9 steps of 32)
_PROJ_RESIDENT_K = 2304


def proj_fused(M: int, N: int, K: int, norm: bool, gated: bool) -> bool:
    """Whether a decode projection of ``M`` rows runs as one ``kdn_decode_proj`` launch rather than apart (the norm
    kernel, ``linear`` / ``swiglu_gate``, the addition).

    * With x in registers (M <= 32, K <= 2304) one launch is the faster, K 512 to 2304: [2 x 7208, 2304] gated at M 1 /
      32 takes 18.0 / 22.3 us, apart 19.7 / 27.2.  (Only the widest product, a head's, loses from 17 rows on: up to
      5 us of 30.)
    * A normed or gated product past either limit re-reads x for every tile of 16 output rows: [32000, 2304] at M 33 /
      64 takes 112 / 152 us, apart 35; [2 x 7680, 2560] gated at M 1 / 32 takes 24 / 45, apart 21 / 30.  It stays one
      launch for 5 to 8 rows, which the GEMV multiplies one by one (M 8: 26 us, apart 46), gated also for 9 to 16 up
      to K 3072 (M 9 / 16: 26 / 29, apart 31), and beyond 32 rows where x is small and all tiles run at once (K <= 1024,
      256 tiles; [2 x 3072, 1024] gated at M 64: 10.6, apart 18.6).
    * A product by itself splits a longer K and stays one launch ([2560, 7680] at M 1 / 16 / 64: 14.7 / 15.7 / 23.9 us,
      apart 14.9 / 16.2 / 26.1)."""
    if not (norm or gated):
        return True
    if M <= 32:
        return K <= _PROJ_RESIDENT_K or 5 <= M <= (16 if gated and K <= 3072 else 8)
    return K <= 1024 and N <= 16 * 256


def _decode_proj(x, weight, *, norm=None, bias=None, residual=None, gated=False):
    """``kdn_decode_proj`` (``norm``: an RMS-norm module) by the rule of ``proj_fused``: in one launch, or apart."""
    from .kdn_ops import step
    N = weight.shape[0] // 2 if gated else weight.shape[0]
    if proj_fused(x.shape[0], N, x.shape[1], norm is not None, gated):
        return step.kdn_decode_proj(x, weight, norm_weight=None if norm is None else norm.weight,
                                    eps=0.0 if norm is None else norm.eps, bias=bias, residual=residual, gated=gated)
    h = x if norm is None else norm(x)
    y = swiglu_gate(h, weight) if gated else linear(h, weight, bias)
    return y if residual is None else residual + y


def decode_block(block, x, state):
    """One token through ``block`` on an in-place ``state`` in five launches (``kdn_decode_proj`` and
    ``kdn_decode_mixer``; a few more where ``proj_fused`` takes a product apart), or None where the call is not
    of that form: bf16 parameters and activations, eval mode under no_grad, at most PACK_MAX_ROWS sequences,
    pre-norm RMS-norm blocks with an (unbiased w1 | w2) SwiGLU, no parts of other types than the model's own, and
    no hooks that would miss the parts' calls.

    At iso_kdn_1.3B width a two-layer step takes 144 us at one sequence and 216 at 32, against 199 and 325
    through the layers' own launches (16 per block)."""
    from .diag_kdn import DiagonalKalmanDeltaNetwork, ShortConvolution
    from .iso_kdn import IsotropicKalmanDeltaNetwork
    from .kdn_ops import step
    from .kdn_ops.gated_norm import FusedRMSNormGated
    from .kdn_state import KDNLayerState, check_state
    from .model import LLaMAMLP, SwiGLU
    from .rmsnorm import FusedRMSNorm
    attn, mlp = block.attn, getattr(block, "mlp", None)
    iso = type(attn) is IsotropicKalmanDeltaNetwork
    if not (isinstance(state, KDNLayerState) and state.inplace and _decode_rows(x, block)
            and (iso or type(attn) is DiagonalKalmanDeltaNetwork) and type(mlp) is LLaMAMLP
            and not block.config.parallel_residual and type(block.norm_1) is FusedRMSNorm
            and type(getattr(block, "norm_2", None)) is FusedRMSNorm and type(mlp.swiglu) is SwiGLU
            and type(attn.o_norm) is FusedRMSNormGated
            and (iso or all(type(c) is ShortConvolution for c in (attn.q_conv1d, attn.k_conv1d, attn.v_conv1d)))
            and _plain(block)):
        return None
    sw, on = mlp.swiglu, attn.o_norm
    if sw.w1.bias is not None or sw.w2.bias is not None or on.activation != "sigmoid" or on.weight is None:
        return None
    B, H, K = x.shape[0], attn.num_heads, attn.head_k_dim
    n = H * K
    check_state(state, B, H, K, K, 1 if iso else 3, (B, H) if iso else (B, H, K), x.device)
    wf = attn.f_proj[1].weight
    if iso:
        taps = (attn.qkv_pack.convolution_weight,)
        inputs = (attn.qkv_pack.projection_weight, attn.f_omega_r_proj.weight, attn.g_proj[0].weight)
        offsets = (3 * n, 0, 3 * n + K, 3 * n + K + 2 * H)
        wo = bo = None
    else:
        taps = tuple(c.weight.view(n, 4) for c in (attn.q_conv1d, attn.k_conv1d, attn.v_conv1d))
        inputs = (attn.q_proj.weight, attn.k_proj.weight, attn.v_proj.weight, attn.f_proj[0].weight,
                  attn.omega_proj[0].weight, attn.g_proj[0].weight, attn.r_proj.weight)
        offsets = (3 * n, 3 * n + K, 3 * n + 3 * K, 3 * n + 2 * K)
        wo, bo = attn.omega_proj[1].weight, attn.omega_proj[1].bias
    wg, bg = attn.g_proj[1].weight, attn.g_proj[1].bias
    if not (_bf16_dense(*inputs, *taps, wf, wo, bo, wg, bg, on.weight, attn.o_proj.weight, block.norm_1.weight,
                        block.norm_2.weight, sw.w1.weight, sw.w2.weight, sw.w3.weight, sw.w3.bias, *state.conv)
            and state.memory.is_contiguous() and state.precision.is_contiguous()
            and (iso or (attn.r_proj.bias is not None and attn.r_proj.bias.dtype == torch.bfloat16))
            and sw.w3.weight.shape[1] % 8 == 0):
        return None
    w_in = packed_weight(attn, "in_proj", inputs, row_multiple=8 if iso else 1)  # the layers' own packing
    b_in = None if iso else packed_bias(attn, "in_proj_bias", (3 * n + 3 * K, attn.r_proj.bias))
    x0 = x.view(B, -1)
    p = _decode_proj(x0, w_in, norm=block.norm_1, bias=b_in)
    o = step.kdn_decode_mixer(
        p, offsets, tuple(state.conv), taps, wf, wo, bo, wg, bg,
        as_f32(attn, "omega_bias", attn.omega_proj.bias) if iso else None,
        as_f32(attn, "r_bias", attn.r_proj.bias) if iso else None, as_f32(attn, "A_log", attn.A_log),
        as_f32(attn, "dt_bias", attn.dt_bias), omega_min=attn.omega_min, r_min=attn.r_min, info_scale=attn.info_scale,
        precision=state.precision, memory=state.memory, norm_weight=on.weight, eps=on.eps, iso=iso)
    x1 = _decode_proj(o, attn.o_proj.weight, residual=x0)
    hid = _decode_proj(x1, packed_weight(sw, "w12", (sw.w1.weight, sw.w2.weight)), norm=block.norm_2, gated=True)
    x2 = _decode_proj(hid, sw.w3.weight, bias=sw.w3.bias, residual=x1)
    state.seen_tokens += 1
    return x2.view(x.shape)


def decode_head(x, norm, head, model):
    """The logits of ``norm(x)`` and ``head``'s weight (which is all that ``GPT.forward`` uses of it) for the one-token
    step in one launch, or None (as ``decode_block``, or where ``proj_fused`` takes them apart)."""
    from .kdn_ops import step
    from .rmsnorm import FusedRMSNorm
    if not (_decode_rows(x, model) and type(norm) is FusedRMSNorm and type(head) is torch.nn.Linear
            and proj_fused(x.shape[0], head.out_features, x.shape[2], True, False)
            and _bf16_dense(norm.weight, head.weight) and _plain(norm)):
        return None
    y = step.kdn_decode_proj(x.view(x.shape[0], -1), head.weight, norm_weight=norm.weight, eps=norm.eps)
    return y.view(x.shape[0], 1, -1)


__all__ = ("PACK_MAX_ROWS", "GEMV_MAX_ROWS", "use_packed", "clear_inference_caches", "packed_weight", "packed_bias",
           "as_f32", "linear", "swiglu_gate", "decode_block", "decode_head")
