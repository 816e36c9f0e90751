"""Exact per-chunk log Z (drop-in for the reference's ops/exact_chunk_log_z_tilelang.py)."""
from typing import Optional

import torch

from . import _cabi
from ._native_op import NativeOp


class _ExactChunkLogZ(NativeOp):
    """Mirrors _ExactChunkLogZ (ops/exact_chunk_log_z_tilelang.py:394-478): the autograd node is native
    (csrc/host_ops.cpp)."""

    @staticmethod
    def native(q, k, chunk_size, window_size, sm_scale, mask_lmk=False):
        return _cabi.host().chunk_log_z(q, k, int(chunk_size), int(window_size), float(sm_scale), bool(mask_lmk))

    @staticmethod
    def forward(ctx, *args):
        return NativeOp.record(ctx, _ExactChunkLogZ.native, args)


def exact_chunk_log_z_tl(q: torch.Tensor, k: torch.Tensor, *, chunk_size: int, window_size: int,
                         sm_scale: Optional[float] = None, mask_lmk: bool = False) -> torch.Tensor:
    """log_Z[b,t,h,c] = log sum_{j in chunk c} exp(sm_scale*<q_t,k_j>) for chunks fully
    before the local window; (B, L, H_q, ceil(L/chunk_size)) fp32, -inf elsewhere.
    ``mask_lmk=True`` also masks landmark keys and is forward-only (backward raises)."""
    if sm_scale is None:
        sm_scale = (1.0 / q.shape[-1]) ** 0.5
    return _ExactChunkLogZ.apply(q, k, chunk_size, window_size, sm_scale, mask_lmk)
