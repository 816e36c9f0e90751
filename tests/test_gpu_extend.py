"""Many queries per sequence on a cache (a prompt's next slice): decode_step on both sides of its rule for leaving the
one-launch kernel, against the two calls and the oracle."""
import pytest
import torch

from util import assert_close_bf16, note

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Lq,Lkv,HQ,H,D,K", [(1, 64, 8192, 16, 2, 64, 8),    # at the rule's line
                                               (1, 63, 4100, 16, 2, 64, 32),   # too few queries for the prefill kernels
                                               (2, 130, 4133, 8, 2, 128, 16),
                                               (1, 70, 40000, 4, 4, 64, 16)])  # few queries on a long cache
def test_decode_step_with_many_queries(pkg, orc, dev, B, Lq, Lkv, HQ, H, D, K):
    note(f"decode_step B{B} Lq{Lq} Lkv{Lkv} HQ{HQ} H{H} D{D} K{K}")
    gen = torch.Generator().manual_seed(82)
    q = torch.randn(B, Lq, HQ, D, generator=gen).bfloat16()
    k = torch.randn(B, Lkv, H, D, generator=gen).bfloat16()
    v = torch.randn(B, Lkv, H, D, generator=gen).bfloat16()
    lse = torch.randn(B, Lq, HQ, generator=gen) * 3 + 2
    qd, kd, vd, lsed = q.to(dev), k.to(dev), v.to(dev), lse.to(dev)
    N = Lkv // 64
    lmk = pkg.chunk_mean_pool(kd[:, : N * 64].contiguous(), 64)
    o, w, idx, sc = pkg.decode_step(qd, pkg.head_major_chunk_keys(lmk), kd, vd, lsed, K, 64, 1, q_offset=Lkv - Lq,
                                    lmk_head_major=True)
    idx0, sc0, w0 = pkg.topk_chunk_weights(qd, lmk, lsed, K, 64, 1, q_offset=Lkv - Lq)
    assert torch.equal(idx, idx0) and torch.equal(sc, sc0) and torch.equal(w, w0)
    assert_close_bf16(o, orc.sparse_attn(q, k, v, w.cpu(), idx.cpu(), chunk_size=64), "output")
