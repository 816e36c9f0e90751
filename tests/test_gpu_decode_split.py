"""Decode steps with few rows: several workgroups per row (logits in a kernel of their own, the attention split over
workgroups) against the oracle's stages, and against the one-launch kernel, whose selection they must repeat exactly."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _case(B, Lkv, HQ, H, D, perq, dev, seed):
    gen = torch.Generator(device=dev).manual_seed(seed)
    bf = dict(device=dev, dtype=torch.bfloat16)
    N, G = Lkv // 64, HQ // H
    q = torch.randn(B, 1, HQ, D, generator=gen, **bf)
    k = torch.randn(B, Lkv, H, D, generator=gen, **bf)
    v = torch.randn(B, Lkv, H, D, generator=gen, **bf)
    lmk = torch.randn(B, HQ if perq else H, N, D, generator=gen, **bf)
    bias = torch.randn(B, H, N, G, generator=gen, device=dev) if perq else None
    lse = torch.randn(B, 1, HQ, generator=gen, device=dev) + 4
    return q, k, v, lmk, bias, lse


@pytest.mark.parametrize("B,Lkv,HQ,H,D,topk,perq", [
    (1, 8229, 32, 4, 128, 32, False),    # 4 rows, four workgroups each
    (8, 12801, 32, 8, 128, 32, False),   # 64 rows
    (1, 2049, 32, 4, 64, 32, True),      # a key and a bias per query head, fewest chunks
    (2, 30001, 16, 2, 64, 17, True),     # a selection that does not divide by the workgroups
    (1, 131072, 6, 2, 64, 8, False),     # three heads, many chunks, one chunk per wavefront
    (3, 40000, 32, 8, 128, 20, True),
    (1, 250000, 4, 1, 128, 32, True),    # the bias shares the logits' array
])
def test_decode_split(pkg, dev, B, Lkv, HQ, H, D, topk, perq):
    from hils_attention_amd.ops import _cabi
    q, k, v, lmk, bias, lse = _case(B, Lkv, HQ, H, D, perq, dev, Lkv)
    N, W, scale = Lkv // 64, 512, 1 / math.sqrt(D)
    assert _cabi.load().hils_decode_step_workspace(B, 1, N, HQ, H, D, topk, int(perq), 0) > 0, "the case must be split"
    o, w, idx, sc = pkg.decode_step(q, lmk, k, v, lse, topk, 64, W, q_offset=Lkv - 1, prior_b=bias, lmk_head_major=True)
    # the one-launch kernel: the same entry point without a workspace
    o1, w1, idx1, sc1 = (torch.empty_like(x) for x in (o, w, idx, sc))
    _cabi.call("hils_decode_step", _cabi.ptr(q), _cabi.ptr(lmk), _cabi.ptr(k), _cabi.ptr(v), _cabi.ptr(lse), _cabi.ptr(bias),
               _cabi.ptr(idx1), _cabi.ptr(sc1), _cabi.ptr(w1), _cabi.ptr(o1), None, None, B, 1, Lkv, N, HQ, H, D, topk, 64,
               W, Lkv - 1, scale, scale, 1, 1, N, int(perq))
    assert torch.equal(idx, idx1) and torch.equal(sc, sc1) and torch.equal(w, w1)
    # attention over the chunks that were selected, fp32
    G = HQ // H
    for b in range(B):
        for h in range(H):
            c = idx[b, 0, h]
            c = c[c >= 0].long()
            tok = (c[:, None] * 64 + torch.arange(63, device=dev)).reshape(-1)
            kk, vv = k[b, tok, h].float().view(-1, 63, D), v[b, tok, h].float().view(-1, 63, D)
            qq = q[b, 0, h * G:(h + 1) * G].float()
            p = torch.softmax(torch.matmul(kk, qq.t()) * scale, dim=1)                 # (chunks, 63, G)
            oc = (p.unsqueeze(-1) * vv.unsqueeze(2)).sum(1)                            # (chunks, G, D)
            ref = (oc * w[b, 0, h * G:(h + 1) * G, : len(c)].float().t().unsqueeze(-1)).sum(0)
            torch.testing.assert_close(o[b, 0, h * G:(h + 1) * G].float(), ref, atol=2e-2, rtol=2e-2)
    torch.testing.assert_close(o.float(), o1.float(), atol=1e-2, rtol=1e-2)


@pytest.mark.parametrize("D,Dv,HQ,H,B,Lq,Lk,W,mask", [
    (64, 64, 4, 4, 1, 1, 70, 64, True), (128, 128, 32, 8, 2, 1, 640, 512, False), (64, 128, 16, 1, 1, 3, 33, 16, True),
    (128, 64, 8, 4, 3, 5, 129, 100, True), (64, 64, 16, 2, 1, 40, 600, 512, False),
])
def test_swa_rows(pkg, dev, D, Dv, HQ, H, B, Lq, Lk, W, mask):
    """The local branch of few queries on the tail of a cache buffer (strided between sequences)."""
    gen = torch.Generator(device=dev).manual_seed(W)
    bf = dict(device=dev, dtype=torch.bfloat16)
    q = torch.randn(B, Lq, HQ, D, generator=gen, **bf)
    kbuf, vbuf = torch.randn(B, Lk + 128, H, D, generator=gen, **bf), torch.randn(B, Lk + 128, H, Dv, generator=gen, **bf)
    k, v = kbuf[:, 64:64 + Lk], vbuf[:, 64:64 + Lk]
    start = 192
    o, lse = pkg.flex_attn_tl(q, k, v, W, 64, training=False, mask_lmk=mask, kv_start=start)
    G = HQ // H
    pos = start + torch.arange(Lk, device=dev)
    qpos = (start + Lk - Lq + torch.arange(Lq, device=dev)).view(-1, 1)
    lo = torch.div(qpos - W + 1, 64, rounding_mode="floor") * 64
    see = (pos >= lo) & (pos <= qpos)
    if mask:
        see &= (pos + 1) % 64 != 0
    kf = k.float().repeat_interleave(G, 2).permute(0, 2, 3, 1).contiguous()
    s = torch.matmul(q.float().permute(0, 2, 1, 3).contiguous(), kf) / math.sqrt(D)
    s = s.masked_fill(~see, float("-inf"))
    ref_lse = torch.logsumexp(s, -1).permute(0, 2, 1)
    vf = v.float().repeat_interleave(G, 2).permute(0, 2, 1, 3).contiguous()
    ref = torch.matmul(torch.nan_to_num(torch.softmax(s, -1)), vf).permute(0, 2, 1, 3)
    fin = torch.isfinite(ref_lse)
    assert torch.equal(fin, torch.isfinite(lse))
    torch.testing.assert_close(lse[fin], ref_lse[fin], atol=1e-3, rtol=1e-3)
    torch.testing.assert_close(o.float(), ref, atol=2e-2, rtol=2e-2)
