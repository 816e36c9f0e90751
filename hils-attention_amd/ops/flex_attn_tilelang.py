"""Sliding-window attention of the local branch (drop-in for flex_attn_tl of the reference's
ops/flex_attn_tilelang.py)."""
from . import _cabi
from ._native_op import NativeOp


class _FlexAttnTL(NativeOp):
    """Mirrors _FlexAttnTL (ops/flex_attn_tilelang.py:1156-1255; kernels :26-267 forward,
    :270-1153 backward): the autograd node is native (csrc/host_ops.cpp).  lse is kept in natural-log
    units throughout."""

    @staticmethod
    def native(q, k, v, window_size, chunk_size, mask_lmk, expand_to_chunk, use_cache, sm_scale, kv_start):
        return _cabi.host().flex_attn(q, k, v, int(window_size), int(chunk_size), bool(mask_lmk),
                                      bool(expand_to_chunk), bool(use_cache), sm_scale, int(kv_start))

    @staticmethod
    def forward(ctx, *args):
        return NativeOp.record(ctx, _FlexAttnTL.native, args)


def flex_attn_tl(q, k, v, window_size: int, chunk_size: int, training: bool = True,
                 mask_lmk: bool = True, expand_to_chunk: bool = True, sm_scale: float = None,
                 kv_start: int = 0):
    """q (B,Lq,H_q,D), k (B,Lk,H_kv,D), v (B,Lk,H_kv,Dv) bf16 -> o (B,Lq,H_q,Dv) bf16 and
    lse (B,Lq,H_q) fp32 in natural-log units.  Causal window of ``window_size`` tokens whose left
    edge moves to the start of its chunk when ``expand_to_chunk``; ``mask_lmk`` hides the last
    token of every chunk.  ``training=False`` allows Lq <= Lk (queries are the last Lq positions)
    and a cache truncated at ``kv_start``."""
    if training and int(kv_start) != 0:
        raise ValueError("flex_attn_tl only supports non-zero kv_start in inference (training=False)")
    return _FlexAttnTL.apply(q, k, v, window_size, chunk_size, mask_lmk, expand_to_chunk, not training, sm_scale, kv_start)


def flex_attn_tl_two_phase(q, k, v, window_size: int, chunk_size: int, training: bool = True,
                           mask_lmk: bool = True, expand_to_chunk: bool = True, sm_scale: float = None,
                           kv_start: int = 0):
    """Same as ``flex_attn_tl`` (ops/flex_attn_tilelang.py:1313-1349 of the reference): the
    reference's variant with an atomic-free backward of two kernels (dQ over query blocks, dK/dV
    over key blocks, bf16 outputs written directly), which is how the backward here always works."""
    if training and int(kv_start) != 0:
        raise ValueError(
            "flex_attn_tl_two_phase only supports non-zero kv_start in inference (training=False)")
    return flex_attn_tl(q, k, v, window_size, chunk_size, training=training, mask_lmk=mask_lmk,
                        expand_to_chunk=expand_to_chunk, sm_scale=sm_scale, kv_start=kv_start)
