"""The operators as autograd functions: a trace records each as a node that replays on other inputs, and a tangent or a
function transform is refused, not dropped.  On the CPU the native module is replaced by a stand-in that, like it, writes
its result behind torch's back; on the GPU the operators themselves run."""
import ctypes
import warnings

import pytest
import torch
from torch.autograd import forward_ad

from util import note

OPS = ["flex_attn", "norm_rope_pool", "attn_pool", "topk_select", "chunk_weights", "sparse_attn", "chunk_log_z"]


class _StandIn:
    """Every operator: twice its first input, in a tuple where the native one returns a tuple."""

    def __getattr__(self, name):
        def op(x, *_):
            if torch.is_grad_enabled() and x.requires_grad:
                y = x * 2
            else:
                y = torch.empty_like(x)
                src = (x.detach() * 2).contiguous()
                ctypes.memmove(y.data_ptr(), src.data_ptr(), src.numel() * src.element_size())
            if name == "topk_select":
                return torch.zeros(x.shape[:3] + (2,), dtype=torch.int32), y
            if name == "norm_rope_pool":
                return y, None
            return (y, y.detach().float().sum(-1)) if name in ("flex_attn", "attn_pool") else y
        return op


def _operator(pkg, name, seed, dev="cpu"):
    """(function of the differentiable input that returns the differentiable output, that input)"""
    gen = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=gen).bfloat16().to(dev)
    B, L, HQ, H, D, K, N = 1, 128, 4, 2, 64, 2, 2
    q, k, v = r(B, L, HQ, D), r(B, L, H, D), r(B, L, H, D)
    lse, w = r(B, L, HQ).float() + 2, torch.softmax(r(B, L, HQ, K).float(), -1).bfloat16()
    idx = torch.zeros(B, L, H, K, dtype=torch.int32, device=dev)
    idx[..., 1] = -1
    lmk, mu, kc = r(B, N, H, D), r(B, N, HQ, D), r(B, N, 64, H, D)
    sc = r(B, L, HQ, K)
    if name == "flex_attn":
        return lambda x: pkg.flex_attn_tl(x, k, v, 64, 64)[0], q
    if name == "norm_rope_pool":
        return lambda x: pkg.norm_rope_pool(x, pool=False)[0], k
    if name == "attn_pool":
        return lambda x: pkg.chunk_attn_pool(x, kc)[0], mu
    if name == "topk_select":
        # (every query sees the same chunks here: the scores are a smooth function of q)
        return lambda x: pkg.online_softmax_topk_head(x, lmk, lse, K, 64, 1, is_causal=False)[1], q
    if name == "chunk_weights":
        return lambda x: pkg.chunk_weights(x, lse), sc
    if name == "sparse_attn":
        return lambda x: pkg.HiLS_block_M_head(x, k, v, w, idx), q
    return lambda x: pkg.exact_chunk_log_z_tl(x, k, chunk_size=64, window_size=1), q


def _check_operator(pkg, name, dev):
    f, x = _operator(pkg, name, 1, dev)
    y = _operator(pkg, name, 2, dev)[1]
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")
        traced = torch.jit.trace(f, (x,), check_trace=False)
    assert "PythonOp" in str(traced.inlined_graph) or "^" in str(traced.inlined_graph), "the call is a node of the trace"
    assert torch.equal(traced(y), f(y)), "the trace computes on its own inputs"
    assert not torch.equal(f(y).nan_to_num(neginf=0.), f(x).nan_to_num(neginf=0.))
    # gradients through a trace, and inside a dual level without tangents, are the direct call's
    g = torch.randn(f(y).shape, generator=torch.Generator().manual_seed(3)).to(dev, f(y).dtype)
    g = torch.where(torch.isfinite(f(y)), g, torch.zeros_like(g))
    grads = []
    for call in (f, traced):
        leaf = y.clone().requires_grad_()
        grads.append(torch.autograd.grad(call(leaf), leaf, g)[0])
    with forward_ad.dual_level():
        leaf = y.clone().requires_grad_()
        grads.append(torch.autograd.grad(f(leaf), leaf, g)[0])
        assert torch.equal(f(y), f(x.copy_(y))), "a level without tangents changes nothing"
        with pytest.raises((NotImplementedError, RuntimeError), match="jvp"):
            f(forward_ad.make_dual(x, torch.ones_like(x)))
    assert grads[0].abs().sum() > 0
    assert torch.equal(grads[0], grads[1]) and torch.equal(grads[0], grads[2])
    for transformed in (lambda: torch.func.jvp(f, (x,), (x,)), lambda: torch.func.grad(lambda t: f(t).sum())(x),
                        lambda: torch.vmap(f)(x.unsqueeze(0))):
        with pytest.raises(RuntimeError):
            transformed()


@pytest.mark.parametrize("name", OPS)
def test_operator_is_an_autograd_function(pkg, monkeypatch, name):
    from hils_attention_amd.ops import _cabi
    monkeypatch.setattr(_cabi, "host", lambda: _StandIn())
    _check_operator(pkg, name, "cpu")


@pytest.mark.gpu
@pytest.mark.parametrize("name", OPS)
def test_operator_is_an_autograd_function_on_the_gpu(pkg, dev, name):
    note(name)
    _check_operator(pkg, name, dev)


def test_reference_names_are_autograd_functions(pkg):
    from hils_attention_amd.ops import (chunk_attn_pool_tilelang, exact_chunk_log_z_tilelang, flex_attn_tilelang,
                                        hils_fwd_bwd_head, topk_head_softmax)
    for cls in (chunk_attn_pool_tilelang.ChunkAttnPoolFunction, exact_chunk_log_z_tilelang._ExactChunkLogZ,
                flex_attn_tilelang._FlexAttnTL, hils_fwd_bwd_head._hils_block_M_attention_inverse,
                topk_head_softmax.SoftmaxTopKMaxPoolingFusedFn):
        assert issubclass(cls, torch.autograd.Function)
