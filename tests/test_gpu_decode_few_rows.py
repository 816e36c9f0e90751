"""The one-launch decode step at one to a few dozen rows and from one chunk on: selection rule on its own logits,
attention against the oracle."""
import pytest
import torch

from util import assert_close_bf16, note

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Lq,ctx,HQ,H,D,K,perq,prior", [(1, 1, 65, 4, 1, 64, 8, False, False),     # one chunk
                                                         (1, 1, 4097, 16, 2, 64, 16, False, True),
                                                         (1, 2, 700, 8, 2, 128, 32, True, True),     # fewer chunks than topk
                                                         (3, 1, 30001, 6, 2, 128, 32, False, False),
                                                         (2, 1, 20001, 16, 2, 64, 32, True, True),
                                                         (1, 1, 131072, 32, 4, 128, 32, True, True),  # 4 MiB of keys a row
                                                         (5, 1, 90001, 16, 4, 64, 64, False, True),
                                                         (1, 1, 131072, 4, 1, 128, 32, False, False)])
def test_decode_step_few_rows(pkg, orc, dev, B, Lq, ctx, HQ, H, D, K, perq, prior):
    note(f"decode_step B{B} Lq{Lq} ctx{ctx} HQ{HQ} H{H} D{D} K{K} perq={perq} prior={prior}")
    gen = torch.Generator().manual_seed(91)
    N, G = ctx // 64, HQ // H
    q = torch.randn(B, Lq, HQ, D, generator=gen).bfloat16()
    lmk = torch.randn(B, N, HQ if perq else H, D, generator=gen).bfloat16()
    pb = torch.randn(B, N, HQ, generator=gen) if prior else None
    lse = torch.randn(B, Lq, HQ, generator=gen) * 2 + 3
    k = torch.randn(B, ctx, H, D, generator=gen).bfloat16()
    v = torch.randn(B, ctx, H, D, generator=gen).bfloat16()
    off = ctx - Lq
    hm = pkg.head_major_chunk_keys(lmk.to(dev), None if pb is None else pb.to(dev), capacity=N + 3, num_kv_heads=H)
    lmk_hm, pb_hm = hm if prior else (hm, None)
    args = (q.to(dev), lmk_hm, k.to(dev), v.to(dev), lse.to(dev), K, 64, 1)
    kw = dict(q_offset=off, prior_b=pb_hm, lmk_head_major=True, num_chunks=N)
    o, w, idx, sc = pkg.decode_step(*args, **kw)
    lmk32 = lmk.float().repeat_interleave(1 if perq else G, 2)
    logits = torch.einsum("blhd,bnhd->blhn", q.float(), lmk32) / D ** 0.5
    biased = logits if pb is None else logits + pb.permute(0, 2, 1).unsqueeze(1)
    lim = orc.causal_chunk_limit(Lq, off, 1, 64)
    vis = torch.arange(N).view(1, 1, 1, N) < lim.view(1, Lq, 1, 1)
    biased = biased.masked_fill(~vis, float("-inf"))
    tot = torch.logaddexp(torch.logsumexp(biased, -1), lse)
    want = orc.topk_select(biased.view(B, Lq, H, G, N), tot.view(B, Lq, H, G), lim, K)
    same = (idx.cpu() == want).float().mean().item()
    assert same > 0.99, f"{same:.4f} of the indices as selected from fp32 logits"
    got = idx.cpu().clamp_min(0).long().unsqueeze(3).expand(B, Lq, H, G, K).reshape(B, Lq, HQ, K)
    ref_sc = torch.gather(logits, 3, got).masked_fill((idx.cpu() < 0).repeat_interleave(G, 2), float("-inf"))
    assert_close_bf16(sc, ref_sc, "scores")
    ref_w = orc.inter_chunk_softmax(sc.cpu(), lse, None if pb is None else pb.bfloat16(), None if pb is None else idx.cpu())
    assert_close_bf16(w, ref_w, "weights", max_abs=8e-3)
    assert_close_bf16(o, orc.sparse_attn(q, k, v, w.cpu(), idx.cpu(), chunk_size=64), "output")
    o2, w2, idx2, sc2 = pkg.decode_step(*args, **kw)
    assert torch.equal(o, o2) and torch.equal(w, w2) and torch.equal(idx, idx2) and torch.equal(sc, sc2)
