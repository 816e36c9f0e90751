"""Backward kernels that share a result between workgroups: chunks whose (query, slot) pairs are cut into segments, token
blocks of the local branch whose rows are split, and the small query blocks of short calls; against autograd in fp32."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _selected(B, L, H, K, dev, gen, crowd):
    """Ascending chunk indices, -1 padded; `crowd`: every query takes the first chunks it can see."""
    N = L // 64
    vis = ((torch.arange(L, device=dev) - 63) // 64).clamp(0, N).view(1, L, 1, 1)
    r = torch.rand(B, L, H, N, device=dev, generator=gen)
    if crowd:
        r = -torch.arange(N, device=dev, dtype=torch.float32).expand(B, L, H, N)
    r = r.masked_fill(torch.arange(N, device=dev) >= vis, -1e9)
    val, idx = r.topk(min(K, N), -1)
    idx = torch.where(val < -1e8, N, idx).sort(-1).values
    idx = torch.where(idx == N, -1, idx)
    return torch.nn.functional.pad(idx, (0, K - idx.shape[-1]), value=-1).int().contiguous()


def _reference(q, k, v, w, idx, scale, mask_last):
    B, L, HQ, D = q.shape
    H, K, N = k.shape[2], idx.shape[-1], k.shape[1] // 64
    G = HQ // H
    out = []
    for b in range(B):
        for h in range(H):
            qq = q[b, :, h * G:(h + 1) * G]                                      # (L, G, D)
            kk = k[b, : N * 64, h].view(N, 64, D)
            vv = v[b, : N * 64, h].view(N, 64, -1)
            s = torch.matmul(qq.reshape(-1, D), kk.reshape(-1, D).t().contiguous()).view(L, G, N, 64) * scale
            if mask_last:
                s = torch.cat([s[..., :63], torch.full_like(s[..., :1], float("-inf"))], -1)
            p = torch.softmax(s, -1)
            ci = idx[b, :, h].long()
            wf = torch.zeros(L, G, N + 1, device=q.device)
            wf = wf.scatter_add(2, torch.where(ci < 0, N, ci).unsqueeze(1).expand(L, G, K), w[b, :, h * G:(h + 1) * G, :K])
            pw = (p * wf[..., :N].unsqueeze(-1)).view(L * G, N * 64)
            out.append(torch.matmul(pw, vv.reshape(N * 64, -1)).view(L, G, -1))
    return torch.stack(out).view(B, H, L, G, -1).permute(0, 2, 1, 3, 4).reshape(B, L, HQ, -1)


@pytest.mark.parametrize("B,L,HQ,H,D,Dv,K,crowd,mask_last", [
    (1, 1024, 8, 1, 64, 64, 8, True, True),     # 64-pair segments, the first chunks cut many times
    (2, 1000, 16, 2, 64, 64, 16, False, True),  # a ragged last chunk
    (1, 777, 4, 1, 128, 128, 8, True, False),
    (1, 2048, 4, 4, 64, 64, 32, True, True),    # one head per KV head
    (1, 640, 2, 1, 64, 128, 4, True, True),
    (1, 640, 16, 1, 128, 64, 10, False, True),  # all chunks selected
    (1, 192, 8, 2, 64, 64, 3, False, True),     # nothing is cut
])
def test_sparse_attn_backward(pkg, dev, B, L, HQ, H, D, Dv, K, crowd, mask_last):
    gen = torch.Generator(device=dev).manual_seed(L + D)
    scale = 1 / math.sqrt(D)
    q, k, v, w = (torch.randn(*s, device=dev, generator=gen).bfloat16() for s in
                  ((B, L, HQ, D), (B, L, H, D), (B, L, H, Dv), (B, L, HQ, K + 1)))
    d_o = torch.randn(B, L, HQ, Dv, device=dev, generator=gen).bfloat16()
    idx = _selected(B, L, H, K, dev, gen, crowd)
    xs = [x.clone().requires_grad_() for x in (q, k, v, w)]
    o = pkg.HiLS_block_M_head(*xs, idx, block_size=64, mask_last_token=mask_last)
    got = torch.autograd.grad(o, xs, d_o)
    fs = [x.float().requires_grad_() for x in (q, k, v, w)]
    ref_o = _reference(*fs, idx, scale, mask_last)
    ref = torch.autograd.grad(ref_o, fs, d_o.float())
    for name, a, b in zip(("o", "dq", "dk", "dv", "dw"), (o, *got), (ref_o, *ref)):
        err = (a.float() - b).norm() / b.norm().clamp_min(1e-20)
        assert err < 1.5e-2, (name, err.item())
    if mask_last and L >= 128:  # no query attends to a chunk's last token
        assert not got[1][:, 63].any() and not got[2][:, 63].any()


# blocks for more than one round of the compute units: narrow heads keep their own rows in LDS (short ones gather them),
# the last block of a sequence and most tiles of a visit are partly filled
@pytest.mark.parametrize("B,L,HQ,H,K,mask_last", [
    (6, 527, 16, 16, 5, True), (6, 650, 32, 16, 7, False), (4, 650, 64, 16, 6, True), (2, 650, 128, 16, 9, True),
    (1, 579, 256, 16, 3, False)])
def test_sparse_attn_backward_many_blocks(pkg, dev, B, L, HQ, H, K, mask_last):
    test_sparse_attn_backward(pkg, dev, B, L, HQ, H, 64, 64, K, False, mask_last)


# rows of more than 3 MiB per (batch, KV head): where a range's cells have rows enough (1024 on average with eight units and
# more, 2048 with fewer: all but the first two) the items go by ranges of queries (the last one ragged), every chunk is a
# sum of partial results, and the chunk nobody can see has none
@pytest.mark.parametrize("B,L,HQ,H,D,Dv,K,crowd,mask_last", [
    (1, 2111, 16, 2, 64, 128, 6, False, True), (1, 1601, 8, 1, 128, 128, 5, True, False), (2, 1600, 16, 1, 64, 64, 8, True, True),
    (1, 2111, 16, 2, 64, 128, 20, False, True), (1, 1601, 8, 1, 128, 128, 13, True, False), (2, 1601, 32, 8, 128, 128, 7, False, True)])
def test_sparse_attn_backward_ranges(pkg, dev, B, L, HQ, H, D, Dv, K, crowd, mask_last):
    test_sparse_attn_backward(pkg, dev, B, L, HQ, H, D, Dv, K, crowd, mask_last)


# the inverse index itself, out of the workspace of a score gather that uses it (G = 3), against a sort: pairs placed
# directly (few, or too few of a chunk per workgroup) and by way of LDS, ragged last segments, more chunks than threads
@pytest.mark.parametrize("B,L,N,H,K,hole", [(1, 77, 5, 2, 3, 0.3), (2, 300, 64, 1, 200, 0.5), (1, 2100, 12288, 1, 256, 0.),
                                            (1, 8195, 1024, 1, 64, 0.2), (3, 5003, 130, 2, 37, 0.), (1, 2049, 7, 1, 256, 0.99)])
def test_inverse_index(pkg, dev, B, L, N, H, K, hole):
    from hils_attention_amd.ops import _cabi
    lib, G, D = _cabi.load(), 3, 8
    gen = torch.Generator(device=dev).manual_seed(L)
    idx = torch.randint(0, N, (B, L, H, K), device=dev, generator=gen, dtype=torch.int32)
    idx.masked_fill_(torch.rand(B, L, H, K, device=dev, generator=gen) < hole, -1)
    size = lib.hils_topk_bwd_workspace(B, L, N, H, G, D, K)
    ws = torch.empty(size, dtype=torch.uint8, device=dev)
    g, q, lmks = (torch.zeros(*s, dtype=torch.bfloat16, device=dev) for s in ((B, L, H, G, K), (B, L, H, G, D), (B, N, H, D)))
    dq, dlmk = torch.empty_like(q), torch.zeros(B, N, H, D, device=dev)
    rc = lib.hils_topk_bwd(_cabi.ptr(g), _cabi.ptr(q), _cabi.ptr(lmks), _cabi.ptr(idx), _cabi.ptr(dq), _cabi.ptr(dlmk),
                           _cabi.ptr(ws), size, B, L, N, H, G, D, K, 0, 1.0, torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    cells = B * H * N
    part = ((cells + 1) * 4 + 255) // 256 * 256
    offsets = ws[part:part + (cells + 1) * 4].view(torch.int32).long()
    pairs = ws[3 * part:3 * part + idx.numel() * 4].view(torch.int32).long()
    b, t, h, s = torch.meshgrid(*(torch.arange(n, device=dev) for n in (B, L, H, K)), indexing="ij")
    ok = idx >= 0
    cell = ((b * H + h) * N + idx)[ok]
    ref = (cell * (1 << 32) + (t * 256 + s)[ok]).sort().values
    count = torch.bincount(cell, minlength=cells)
    assert torch.equal(offsets, torch.nn.functional.pad(count.cumsum(0), (1, 0)))
    got = torch.repeat_interleave(torch.arange(cells, device=dev), count) * (1 << 32) + pairs[:cell.numel()]
    assert torch.equal(got.sort().values, ref)


@pytest.mark.parametrize("B,L,HQ,H,D,W", [(1, 700, 8, 1, 64, 512), (2, 1024, 16, 2, 64, 512), (1, 513, 4, 1, 128, 300),
                                          (1, 2000, 4, 4, 64, 512)])
def test_swa_backward_split(pkg, dev, B, L, HQ, H, D, W):
    from hils_attention_amd.ops import _cabi
    assert _cabi.load().hils_swa_bwd_workspace(B, L, HQ, H, D, D, W) > 0, "the case must be split"
    gen = torch.Generator(device=dev).manual_seed(W)
    q, k, v = (torch.randn(B, L, h, D, device=dev, generator=gen).bfloat16() for h in (HQ, H, H))
    d_o = torch.randn(B, L, HQ, D, device=dev, generator=gen).bfloat16()
    d_lse = torch.randn(B, L, HQ, device=dev, generator=gen)
    xs = [x.clone().requires_grad_() for x in (q, k, v)]
    o, lse = pkg.flex_attn_tl(*xs, W, 64)
    got = torch.autograd.grad((o, lse), xs, (d_o, d_lse))
    fs = [x.float().requires_grad_() for x in (q, k, v)]
    G = HQ // H
    t = torch.arange(L, device=dev)
    see = (t >= (torch.div(t.view(-1, 1) - W + 1, 64, rounding_mode="floor") * 64)) & (t <= t.view(-1, 1)) & ((t + 1) % 64 != 0)
    s = torch.matmul(fs[0].permute(0, 2, 1, 3).contiguous(),
                     fs[1].repeat_interleave(G, 2).permute(0, 2, 3, 1).contiguous()) / math.sqrt(D)
    s = s.masked_fill(~see, float("-inf"))
    ro = torch.matmul(torch.softmax(s, -1), fs[2].repeat_interleave(G, 2).permute(0, 2, 1, 3).contiguous()).permute(0, 2, 1, 3)
    rl = torch.logsumexp(s, -1).permute(0, 2, 1)
    ref = torch.autograd.grad((ro, rl), fs, (d_o.float(), d_lse))
    for name, a, b in zip(("o", "lse", "dq", "dk", "dv"), (o, lse, *got), (ro, rl, *ref)):
        err = (a.float() - b).norm() / b.norm()
        assert err < 1.5e-2, (name, err.item())


# the score gather's backward by dense products: one query block a workgroup, walks of two to many with a ragged last one,
# blocks without any entry, exactly one tile of chunks and one more (which is not walked)
@pytest.mark.parametrize("B,L,N,H,G,D,K,per_qhead", [(1, 40, 3, 1, 1, 64, 2, 0), (2, 3001, 128, 16, 1, 64, 8, 0), (2, 3001, 129, 16, 1, 64, 8, 0),
                                                     (3, 1037, 16, 2, 16, 64, 5, 1), (1, 2500, 40, 8, 4, 128, 16, 0),
                                                     (9, 700, 11, 8, 4, 128, 33, 1), (4, 9001, 100, 4, 2, 64, 3, 0),
                                                     (1, 300, 20, 2, 4, 128, 6, 0), (2, 901, 140, 2, 4, 128, 9, 1)])
def test_dense_gather_backward_walks(pkg, dev, B, L, N, H, G, D, K, per_qhead):
    from hils_attention_amd.ops import _cabi
    lib, HK = _cabi.load(), H * G if per_qhead else H
    gen = torch.Generator(device=dev).manual_seed(L + N)
    q = torch.randn(B, L, H, G, D, device=dev, generator=gen).bfloat16()
    lmks = torch.randn(B, N, HK, D, device=dev, generator=gen).bfloat16()
    g = torch.randn(B, L, H, G, K, device=dev, generator=gen).bfloat16()
    score = torch.rand(B, L, H, max(N, K), device=dev, generator=gen)
    idx = score.topk(K, -1).indices
    idx = idx.masked_fill(idx >= N, -1)
    idx[:, 100:400] = -1
    idx = idx.int().contiguous()
    dq, dlmk = torch.empty_like(q), torch.zeros(B, N, HK, D, device=dev)
    rc = lib.hils_topk_bwd(_cabi.ptr(g), _cabi.ptr(q), _cabi.ptr(lmks), _cabi.ptr(idx), _cabi.ptr(dq), _cabi.ptr(dlmk),
                           None, 0, B, L, N, H, G, D, K, per_qhead, 0.125, torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    live = (idx >= 0).unsqueeze(3)
    a = torch.zeros(B, L, H, G, N, dtype=torch.float64, device=dev)
    a.scatter_add_(4, idx.clamp(min=0).long().unsqueeze(3).expand(B, L, H, G, K), (g.double() * 0.125).masked_fill(~live, 0.))
    a = a.permute(0, 2, 3, 1, 4).reshape(B, HK, -1, N)  # rows of a chunk-key head
    rows = q.double().permute(0, 2, 3, 1, 4).reshape(B, HK, -1, D)
    keys = lmks.double().permute(0, 2, 1, 3).contiguous()
    want_q = (a @ keys).reshape(B, H, G, L, D).permute(0, 3, 1, 2, 4)
    size_q = (a.abs() @ keys.abs()).reshape(B, H, G, L, D).permute(0, 3, 1, 2, 4)
    at = a.transpose(2, 3).contiguous()
    want_l, size_l = (at @ rows).permute(0, 2, 1, 3), (at.abs() @ rows.abs()).permute(0, 2, 1, 3)
    # fp32 sums of n terms are within n 2^-24 of their terms' absolute sum; dq is then rounded to eight bits
    assert bool(((dq.double() - want_q).abs() <= want_q.abs() * 2.0 ** -8 + (K + 1) * 2.0 ** -23 * size_q + 1e-30).all())
    assert bool(((dlmk.double() - want_l).abs() <= (L * G + 1) * 2.0 ** -24 * size_l + 1e-30).all())
