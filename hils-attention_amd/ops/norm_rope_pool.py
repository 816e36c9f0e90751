"""Key / query preparation in one pass: per-head RMS norm, rotary embedding, chunk mean.

The reference has no single function for this; its attention layer runs the three steps one
after the other (models/FlashHiLS/hils_attention.py:314-321 k_norm, :479-483 apply_rotary_pos_emb,
:398 / :460 ``k_chunked.mean(dim=2)``), each a full pass over the (B, L, H, D) tensor.
"""
from . import _cabi
from ._native_op import NativeOp


class _NormRopePool(NativeOp):
    @staticmethod
    def native(x, norm_weight, cos, sin, chunk_size, eps, pool):
        return _cabi.host().norm_rope_pool(x, norm_weight, cos, sin, int(chunk_size), float(eps), bool(pool))

    @staticmethod
    def forward(ctx, *args):
        return NativeOp.record(ctx, _NormRopePool.native, args)


def norm_rope_pool(x, norm_weight=None, cos=None, sin=None, chunk_size=64, eps=1e-6, pool=True):
    """x (B,L,H,D) bf16 -> (out (B,L,H,D), lmk (B,L//chunk_size,H,D) or None).

    ``out = rope(rms_norm(x) * norm_weight)`` with the roundings of the layer's bf16 sequence;
    ``lmk`` is the mean of ``out`` over every whole chunk (``pool=False`` skips it: the query
    side).  ``norm_weight`` (D,) or None (no norm); ``cos`` / ``sin`` (L,D), (1,L,D) or (B,L,D),
    HF rotate-half convention, or None (no rotation).  Differentiable in ``x`` and ``norm_weight``.
    """
    return _NormRopePool.apply(x, norm_weight, cos, sin, chunk_size, eps, pool)
