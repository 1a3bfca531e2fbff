"""The decode step's fused launches: ``kdn_decode_proj`` against float64 (row tiles of 16 / 32 / 64, N and K
remainders, every prologue and epilogue), and a block's one-token step on an in-place state through
``decode_block`` against the layers' own launches, with the advanced states."""
import copy

import pytest
import torch

from gpu_util import gpu_or_skip, log, rel
from lit_gpt import _inference, model as model_mod
from lit_gpt.kdn_ops.step import kdn_decode_proj
from lit_gpt.kdn_state import KDNLayerState

pytestmark = pytest.mark.gpu


# bf16 results: 2^-9 of the value; the normed operand x nw rounds once more (2^-9 per term, averaging over K)
@pytest.mark.parametrize("M,N,K,norm,gated,bias,res", [
    (1, 7204, 2304, True, False, False, False), (1, 33, 8, False, False, True, False), (3, 17, 40, True, True, True, False),
    (16, 2304, 6144, False, False, False, True), (17, 100, 1160, True, False, True, True),
    (32, 513, 2304, True, True, False, False), (33, 48, 128, False, True, False, False),
    (17, 500, 2312, False, False, True, True), (32, 2304, 6912, False, False, False, True), (64, 40, 4616, False, False, True, False),
    (64, 1000, 2304, True, False, False, False), (64, 64, 264, True, True, True, True)])
def test_decode_proj_matches_fp64(M, N, K, norm, gated, bias, res):
    dev = gpu_or_skip()
    log(f"case decode_proj M={M} N={N} K={K} norm={norm} gated={gated} bias={bias} res={res}")
    g = torch.Generator().manual_seed(M + N + K)
    R = 2 * N if gated else N
    x = torch.randn(M, K + 8, generator=g).bfloat16()[:, :K]  # rows K + 8 elements apart
    W = (torch.randn(R, K, generator=g) / K ** 0.5).bfloat16()
    nw = (1 + 0.1 * torch.randn(K, generator=g)).bfloat16() if norm else None
    b = torch.randn(R, generator=g).bfloat16() if bias else None
    r = torch.randn(M, N, generator=g).bfloat16() if res else None
    xd = x.double()
    if norm:
        xd = xd * (xd.square().mean(-1, keepdim=True) + 1e-5).rsqrt() * nw.double()
    h = xd @ W.double().T + (b.double() if bias else 0)
    ref = torch.nn.functional.silu(h[:, :N]) * h[:, N:] if gated else h
    ref = ref + r.double() if res else ref
    dx = torch.empty(M, K + 8, dtype=torch.bfloat16, device=dev)[:, :K].copy_(x)
    to = lambda t: t.to(dev) if t is not None else None  # noqa: E731
    y = kdn_decode_proj(dx, W.to(dev), norm_weight=to(nw), eps=1e-5, bias=to(b), residual=to(r), gated=gated)
    assert rel(y.float().cpu(), ref) < 6e-3


@pytest.mark.parametrize("mixer_type", ["iso_kdn", "diag_kdn"])
@pytest.mark.parametrize("B,H,d", [(1, 2, 128), (3, 4, 64), (17, 1, 128), (64, 2, 64)])
def test_decode_block_matches_the_layers_launches(mixer_type, B, H, d, monkeypatch):
    dev = gpu_or_skip()
    log(f"case decode_block {mixer_type} B={B} H={H} d={d}")
    torch.manual_seed(B + H + d)
    cfg = model_mod.Config.from_name(("iso" if mixer_type == "iso_kdn" else "diag") + "_kdn_1.3B", n_layer=1, n_head=H,
                                     n_embd=H * d, intermediate_size=3 * H * d, kdn_info_scale=float(d))
    m = model_mod.GPT(cfg).to(dev).to(torch.bfloat16).eval()
    if mixer_type == "diag_kdn":  # its omega projection starts at zero
        with torch.no_grad():
            m.transformer.h[0].attn.omega_proj[1].weight.uniform_(-0.1, 0.1)
            m.transformer.h[0].attn.omega_proj[1].bias.uniform_(-0.1, 0.1)
    idx = torch.randint(0, 200, (B, 6), device=dev)

    def inplace(s):
        return KDNLayerState(tuple(c.clone() for c in s.conv), s.memory.clone(), s.precision.clone(), s.seen_tokens, True)

    with torch.no_grad():
        _, st = m(idx[:, :3], return_state=True)
        fused, plain = [inplace(s) for s in st], [inplace(s) for s in st]
        calls = []
        monkeypatch.setattr(model_mod, "decode_block", lambda *a: calls.append(_inference.decode_block(*a)) or calls[-1])
        a = [m(idx[:, t:t + 1], state=fused, return_state=True)[0] for t in range(3, 6)]
        assert len(calls) == 3 and all(c is not None for c in calls)
        monkeypatch.setattr(model_mod, "decode_block", lambda *a: None)
        monkeypatch.setattr(model_mod, "decode_head", lambda *a: None)
        b = [m(idx[:, t:t + 1], state=plain, return_state=True)[0] for t in range(3, 6)]
    torch.cuda.synchronize()
    # both round activations to bf16 at 6 to 12 places on the way (2^-9 each)
    for x, y in zip(a, b):
        assert rel(x.float(), y.float()) < 2e-2
    for s, p in zip(fused, plain):
        assert s.seen_tokens == p.seen_tokens == 6
        assert rel(s.memory, p.memory) < 2e-2 and rel(s.precision, p.precision) < 1e-2
        for c, e in zip(s.conv, p.conv):
            assert rel(c.float(), e.float()) < 1e-2


def test_decode_block_steps_aside():
    """Hooks, training mode, autograd, longer inputs and states that are not in place keep the layers' launches."""
    dev = gpu_or_skip()
    cfg = model_mod.Config.from_name("iso_kdn_1.3B", n_layer=1, n_head=1, n_embd=128, intermediate_size=256)
    m = model_mod.GPT(cfg).to(dev).to(torch.bfloat16).eval()
    block = m.transformer.h[0]
    with torch.no_grad():
        st = m(torch.zeros(1, 4, dtype=torch.long, device=dev), return_state=True)[1][0]
        live = KDNLayerState(tuple(c.clone() for c in st.conv), st.memory.clone(), st.precision.clone(), 4, True)
        x = torch.randn(1, 1, 128, device=dev).bfloat16()
        assert _inference.decode_block(block, x, st) is None
        assert _inference.decode_block(block, x.float(), live) is None
        assert _inference.decode_block(block, x.expand(1, 2, 128).contiguous(), live) is None
        hook = block.attn.register_forward_hook(lambda *a: None)
        assert _inference.decode_block(block, x, live) is None
        hook.remove()
        block.train()
        assert _inference.decode_block(block, x, live) is None
        block.eval()
        assert _inference.decode_block(block, x, live) is not None
    assert _inference.decode_block(block, x, live) is None  # autograd on
    assert copy.copy(live).seen_tokens == 5


@pytest.mark.parametrize("mixer_type,part", [("iso_kdn", "mlp.swiglu"), ("iso_kdn", "attn.o_norm"),
                                             ("diag_kdn", "attn.q_conv1d"), ("diag_kdn", "attn.v_conv1d")])
def test_decode_block_keeps_a_replaced_parts_forward(mixer_type, part):
    """A part that a user exchanged for one of a derived type answers through its own forward (here twice the
    part's value), so the step goes through the layers' launches."""
    dev = gpu_or_skip()
    log(f"case decode_block replaced part {mixer_type} {part}")
    cfg = model_mod.Config.from_name(("iso" if mixer_type == "iso_kdn" else "diag") + "_kdn_1.3B", n_layer=1, n_head=1,
                                     n_embd=128, intermediate_size=256)
    m = model_mod.GPT(cfg).to(dev).to(torch.bfloat16).eval()
    block = m.transformer.h[0]
    with torch.no_grad():
        st = m(torch.zeros(1, 4, dtype=torch.long, device=dev), return_state=True)[1][0]
        live = KDNLayerState(tuple(c.clone() for c in st.conv), st.memory.clone(), st.precision.clone(), 4, True)
        module = block.get_submodule(part)
        module.__class__ = type("Doubled", (type(module),), {"forward": lambda self, *a, **k: 2 * type(self).__base__.forward(self, *a, **k)})
        assert _inference.decode_block(block, torch.randn(1, 1, 128, device=dev).bfloat16(), live) is None
    assert live.seen_tokens == 4


def test_decode_head_takes_the_weight_alone():
    """``GPT.forward`` multiplies by the head's weight and leaves a bias out, for one token as for many."""
    dev = gpu_or_skip()
    cfg = model_mod.Config.from_name("iso_kdn_1.3B", n_layer=1, n_head=1, n_embd=128, intermediate_size=256)
    m = model_mod.GPT(cfg)
    m.lm_head = torch.nn.Linear(128, m.lm_head.out_features, bias=True)
    torch.nn.init.constant_(m.lm_head.bias, 3.0)
    m = m.to(dev).to(torch.bfloat16).eval()
    x = torch.randn(2, 1, 128, device=dev).bfloat16()
    with torch.no_grad():
        y = _inference.decode_head(x, m.transformer.ln_f, m.lm_head, m)
        ref = m.transformer.ln_f(x).double() @ m.lm_head.weight.double().T
    assert rel(y.float(), ref) < 6e-3  # two bf16 roundings


# K past 2304 in splits from 9 rows on; each split's tiles fit its share of the CUs (2048 rows in 3: 79 workgroups)
@pytest.mark.parametrize("M,N,K,bias,res", [(8, 100, 2312, True, True), (9, 100, 2312, True, True), (16, 2048, 6144, False, True),
                                            (12, 3, 4616, True, False), (33, 5, 20744, False, True),
                                            (64, 2048, 6144, True, False), (17, 4100, 2560, False, False)])
def test_split_projection_matches_fp64(M, N, K, bias, res):
    dev = gpu_or_skip()
    log(f"case decode_proj split M={M} N={N} K={K} bias={bias} res={res}")
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g).bfloat16()
    W = (torch.randn(N, K, generator=g) / K ** 0.5).bfloat16()
    b = torch.randn(N, generator=g).bfloat16() if bias else None
    r = torch.randn(M, N, generator=g).bfloat16() if res else None
    ref = x.double() @ W.double().T + (b.double() if bias else 0) + (r.double() if res else 0)
    to = lambda t: t.to(dev) if t is not None else None  # noqa: E731
    y = kdn_decode_proj(to(x), to(W), bias=to(b), residual=to(r))
    assert float(((y.double().cpu() - ref).abs() / (ref.abs() + 1)).max()) < 2.0 ** -8  # one rounding (2^-9 of the value), fp32 sums


@pytest.mark.parametrize("mixer_type,B,H,d", [("iso_kdn", 33, 9, 128), ("diag_kdn", 33, 9, 128), ("iso_kdn", 2, 20, 128),
                                              ("diag_kdn", 6, 38, 64), ("diag_kdn", 9, 20, 128)])
def test_decode_block_with_projections_apart(mixer_type, B, H, d, monkeypatch):
    """Beyond 32 rows and past K 2304 the normed and gated products leave the one launch (K 1152 and 2432, 2560)."""
    test_decode_block_matches_the_layers_launches(mixer_type, B, H, d, monkeypatch)


@pytest.mark.parametrize("mixer_type,B,H", [("iso_kdn", 9, 9), ("iso_kdn", 64, 18), ("diag_kdn", 33, 9), ("iso_kdn", 2, 20)])
def test_captured_step_replays_as_the_eager_step(mixer_type, B, H):
    """The decoder's graph where it holds split products (9 rows, w3 of K 3456) and where it holds library products
    (33 and 64 rows, K 2560): every replay against the eager step, with eager work between the replays."""
    dev = gpu_or_skip()
    from lit_gpt.decode import KDNDecoder
    log(f"case captured step {mixer_type} B={B} H={H}")
    torch.manual_seed(B + H)
    cfg = model_mod.Config.from_name(("iso" if mixer_type == "iso_kdn" else "diag") + "_kdn_1.3B", n_layer=1, n_head=H,
                                     n_embd=128 * H, intermediate_size=3 * 128 * H, kdn_info_scale=128.0)
    m = model_mod.GPT(cfg).to(dev).to(torch.bfloat16).eval()
    idx = torch.randint(0, 200, (B, 9), device=dev)
    eager, graph = KDNDecoder(m, B, use_graph=False), KDNDecoder(m, B, use_graph=True)
    eager.prefill(idx[:, :4])
    graph.prefill(idx[:, :4])
    for t in range(4, 9):
        a = eager.step(idx[:, t]).clone()
        torch.cuda.synchronize()
        b = graph.step(idx[:, t]).clone()
        torch.cuda.synchronize()
        # the same launches; a library product may take another order of its fp32 sum when captured (bf16 after it)
        assert rel(b.float(), a.float()) < 2e-2
    for s, p in zip(graph.state, eager.state):
        assert s.seen_tokens == p.seen_tokens == 9
        assert rel(s.memory, p.memory) < 2e-2 and rel(s.precision, p.precision) < 1e-2
