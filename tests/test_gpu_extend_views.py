"""decode_step with many queries on tensors as a program holds them: a query transposed from (B, H, L, D), the views that
the cache layer's update hands out, and with the selection's logits asked for."""
import pytest
import torch

from util import assert_close_bf16, note

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Lq,Lkv,HQ,H,D,K,perq", [
    (2, 512, 4133, 4, 4, 64, 8, False),     # the prefill kernels
    (3, 300, 8200, 32, 4, 128, 32, True),   # ... with a key and a bias per query head
    (2, 70, 4133, 16, 2, 64, 32, False),    # the one-launch kernel
    (2, 65, 190, 16, 1, 64, 8, False),      # more heads than it takes (eight; the selection takes 16): two calls
])
def test_decode_step_takes_views(pkg, orc, dev, B, Lq, Lkv, HQ, H, D, K, perq):
    note(f"decode_step on views B{B} Lq{Lq} Lkv{Lkv} HQ{HQ} H{H} D{D} K{K} perq={perq}")
    gen = torch.Generator().manual_seed(Lq)
    q = torch.randn(B, HQ, Lq, D, generator=gen).bfloat16().to(dev).transpose(1, 2)
    k = torch.randn(B, Lkv, H, D, generator=gen).bfloat16().to(dev)
    v = torch.randn(B, Lkv, H, D, generator=gen).bfloat16().to(dev)
    N, G = Lkv // 64, HQ // H
    mu = torch.randn(B, N, HQ, D, generator=gen).bfloat16().to(dev) if perq else None
    cache = pkg.HiLSDynamicLayer(chunk_size=64, capacity=Lkv + 1000, offload=False, chunk_pooling=not perq)
    kk, vv = cache.update(k, v, mu_q=mu)
    assert not kk.is_contiguous() and not q.is_contiguous()
    lse = (torch.randn(B, Lq, HQ, generator=gen) * 2 + 3).to(dev)
    lmk, pb = cache.lmk_k[:, :N].contiguous(), cache.prior_b[:, :N].contiguous() if perq else None
    kw = dict(q_offset=Lkv - Lq, prior_b=pb)
    dbg = {}
    o, w, idx, sc = pkg.decode_step(q, lmk, kk, vv, lse, K, 64, 1, **kw)
    o1, w1, idx1, sc1 = pkg.decode_step(q.contiguous(), lmk, k, v, lse, K, 64, 1, _debug=dbg, **kw)
    for a, b in ((o, o1), (w, w1), (idx, idx1), (sc, sc1)):
        assert torch.equal(a, b)
    assert dbg["lse_total"].shape == (B, Lq, H, G) and dbg["sel_logits"].shape == (B, Lq, H, G, N)
    lim = orc.causal_chunk_limit(Lq, Lkv - Lq, 1, 64)
    assert torch.equal(idx.cpu(), orc.topk_select(dbg["sel_logits"].cpu(), dbg["lse_total"].cpu(), lim, K))
    assert_close_bf16(o, orc.sparse_attn(q.cpu().contiguous(), k.cpu(), v.cpu(), w.cpu(), idx.cpu(), chunk_size=64), "output")
    # the layer's own call, on its buffers
    o2, w2, idx2 = cache.hils_attend(q, lse, K, 1)
    assert torch.equal(idx2, idx) and torch.equal(w2, w)
    assert_close_bf16(o2, o.float(), "the layer's call")
