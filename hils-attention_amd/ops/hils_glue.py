"""Fused inter-chunk softmax of the HiLS layer (forward and backward).

The reference computes it with torch ops inside the layer
(models/FlashHiLS/hils_attention.py:585-610): gather the prior bias at the selected chunks,
add it to the scores, concatenate the local-branch LSE (and a zero logit when
``enable_softmax1``), softmax, cast to the hidden dtype.  ``chunk_weights`` does that in one
kernel; column K is the weight of the local (sliding-window) branch.
"""
import torch

from . import _cabi
from ._native_op import NativeOp


class _ChunkWeights(NativeOp):
    @staticmethod
    def native(scores, lse_swa, prior_b, indices, enable_softmax1):
        return _cabi.host().chunk_weights(scores, lse_swa, prior_b, indices, bool(enable_softmax1))

    @staticmethod
    def forward(ctx, *args):
        return NativeOp.record(ctx, _ChunkWeights.native, args)


def chunk_weights(scores, lse_swa, prior_b=None, indices=None, enable_softmax1=False):
    """scores (B,L,HQ,K) bf16, lse_swa (B,L,HQ) -> weights (B,L,HQ,K+1(+1)) bf16.
    ``prior_b`` (B,N,HQ) with ``indices`` (B,L,H,K) adds the gathered prior bias first.
    Differentiable in scores, lse_swa and prior_b."""
    return _ChunkWeights.apply(scores, lse_swa, prior_b, indices, enable_softmax1)


def topk_chunk_weights(q, lmks, lse_swa, topk, block_size, window_size, is_causal=True, q_offset=0,
                       sm_scale=None, prior_b=None, num_kv_heads=None):
    """Inference: ``online_softmax_topk_head`` (no Gumbel / drop mask) followed by ``chunk_weights``
    in one call, for the serving loop.  q (B,L,h_q,D) bf16, lmks (B,N,h_kv,D) bf16 (one chunk key per
    KV head) or, with ``num_kv_heads`` given, (B,N,h_q,D) (one per query head, the layer's
    attention-pooled keys), lse_swa (B,L,h_q) -> indices (B,L,h_kv,topk) int32, scores (B,L,h_q,topk)
    bf16, weights (B,L,h_q,topk+1) bf16.  ``prior_b`` (B,N,h_q): the layer's prior bias (its
    ``enable_prior_query`` mode, models/FlashHiLS/hils_attention.py:568-602), used as the selection's
    ``bias`` and gathered into the softmax.  With about one (query, KV head) row per compute unit the
    selection kernel writes the weights itself; otherwise two kernels run."""
    return _cabi.host().topk_chunk_weights(q, lmks, lse_swa, int(topk), int(block_size), int(window_size),
                                           bool(is_causal), int(q_offset), sm_scale, prior_b, num_kv_heads)


def head_major_chunk_keys(lmks, prior_b=None, capacity=None, num_kv_heads=None):
    """Chunk keys (B,N,h,D) (and the prior bias (B,N,h_q)) re-laid head-major, (B,h,cap,D) and
    (B,h_kv,cap,G): the N keys a decode row streams become one contiguous block.  What this
    package's cache layers keep; ``decode_step(..., lmk_head_major=True)`` takes them.  ``num_kv_heads``:
    needed for the bias when lmks carries one key per query head (h = h_q)."""
    B, N, h, D = lmks.shape
    cap = N if capacity is None else int(capacity)
    assert cap >= N
    out = torch.zeros((B, h, cap, D), dtype=lmks.dtype, device=lmks.device)
    out[:, :, :N] = lmks.permute(0, 2, 1, 3)
    if prior_b is None:
        return out
    h_kv = h if num_kv_heads is None else int(num_kv_heads)
    G = prior_b.shape[2] // h_kv
    pb = torch.zeros((B, h_kv, cap, G), dtype=torch.float32, device=lmks.device)
    pb[:, :, :N] = prior_b.reshape(B, N, h_kv, G).permute(0, 2, 1, 3).float()
    return out, pb


def decode_step(q, lmks, k, v, lse_swa, topk, block_size, window_size, q_offset=0, sm_scale=None,
                mask_last_token=True, _debug=None, prior_b=None, lmk_head_major=False, num_chunks=None):
    """Inference: the remote branch of a decode step, ``topk_chunk_weights`` followed by
    ``HiLS_block_M_head(..., is_training=False)`` on the selected chunks, as one kernel (one workgroup per
    (query, KV head) selects and then attends) or, with few rows for the chip, two that split a row over
    workgroups.  q (B,L,h_q,D), lmks (B,N,h_kv,D), k, v
    (B,Lkv,h_kv,D) bf16 (k, v may live in pinned host memory), lse_swa (B,L,h_q) -> o (B,L,h_q,D),
    weights (B,L,h_q,topk+1), indices (B,L,h_kv,topk), scores (B,L,h_q,topk).  ``prior_b`` (B,N,h_q):
    the layer's prior bias (selection bias and the bias of the inter-chunk softmax).
    ``lmk_head_major``: lmks is (B,h_kv,cap,D) and prior_b (B,h_kv,cap,G) (``head_major_chunk_keys``),
    of which the first ``num_chunks`` (default cap) chunks are looked at.  lmks may carry h_q heads
    instead of h_kv (one chunk key per query head, the layer's attention-pooled keys): (B,N,h_q,D) or,
    head-major, (B,h_q,cap,D).  What the fused kernels do not take (more than eight query heads per KV head,
    more chunks than fit the LDS, K and V shorter than the chunks) runs as the two calls, and so do 64 queries
    per sequence and more where the prefill kernels are ahead.
    q, k and v may have any strides (what is not contiguous is copied).  ``_debug`` (a dict) receives the fp32
    ``sel_logits`` and ``lse_total`` of the selection."""
    return _cabi.host().decode_step(q, lmks, k, v, lse_swa, int(topk), int(block_size), int(window_size),
                                    int(q_offset), sm_scale, bool(mask_last_token), prior_b, bool(lmk_head_major),
                                    num_chunks, _debug)
