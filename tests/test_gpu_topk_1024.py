"""One-pass selection kernel with 513 to 1024 chunks, and the dispatch between it and one workgroup per row."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,N,h_kv,G,D,topk,perq,bias", [
    (300, 513, 2, 1, 64, 32, False, False), (700, 1024, 2, 4, 128, 32, False, False), (400, 1000, 1, 2, 64, 7, False, True),
    (260, 777, 2, 8, 64, 16, False, True), (520, 1023, 1, 6, 128, 32, True, True), (300, 600, 2, 3, 64, 32, True, False),
    (900, 1024, 4, 8, 64, 32, True, True), (1500, 900, 3, 1, 128, 32, False, True),
])
def test_topk_many_chunks(pkg, orc, dev, L, N, h_kv, G, D, topk, perq, bias):
    gen = torch.Generator(device=dev).manual_seed(N)
    h_q, S, W = h_kv * G, 64, 512
    off = N * S - L  # the last queries see all but the window's chunks, the first ones some fewer
    q = torch.randn(1, L, h_q, D, device=dev, generator=gen).bfloat16()
    lmk = torch.randn(1, N, h_q if perq else h_kv, D, device=dev, generator=gen).bfloat16()
    lse = torch.randn(1, L, h_q, device=dev, generator=gen) + 3
    pb = torch.randn(1, N, h_q, device=dev, generator=gen) if bias else None
    idx, sc, w = pkg.topk_chunk_weights(q, lmk, lse, topk, S, W, q_offset=off, prior_b=pb, num_kv_heads=h_kv)
    scale = 1 / math.sqrt(D)
    kf = (lmk if perq else lmk.repeat_interleave(G, 2)).float()[0].permute(1, 2, 0).contiguous()       # (h_q, D, N)
    s = torch.matmul(q.float()[0].permute(1, 0, 2).contiguous(), kf) * scale                            # (h_q, L, N)
    sel = s if pb is None else s + pb[0].t().unsqueeze(1)
    lim = torch.div(torch.arange(L, device=dev) + off - W + 1, S, rounding_mode="floor").clamp(0, N)
    vis = torch.arange(N, device=dev) < lim.view(L, 1)
    sel = sel.masked_fill(~vis, float("-inf"))
    tot = torch.logaddexp(torch.logsumexp(sel, -1), lse[0].t())                                         # (h_q, L)
    pooled = (sel - tot.unsqueeze(-1)).view(h_kv, G, L, N).amax(1)                                      # (h_kv, L, N)
    ref = pooled.topk(topk, -1)
    assert ((idx[0, :, :, 1:] > idx[0, :, :, :-1]) | (idx[0, :, :, 1:] < 0)).all(), "ascending"
    got = idx[0].permute(1, 0, 2).long()
    assert (got >= 0).all() and (got < lim.view(1, L, 1)).all()
    # the same scores up to rounding: every winner is at least as good as the reference's last, less a rounding
    worst = pooled.gather(-1, got).amin(-1)
    assert (worst >= ref.values[..., -1] - 2e-4).all()
    raw = s.view(h_kv, G, L, N).gather(-1, got.unsqueeze(1).expand(-1, G, -1, -1)).permute(2, 0, 1, 3).reshape(L, h_q, topk)
    torch.testing.assert_close(sc[0].float(), raw, atol=2e-2, rtol=1e-2)
    x = sc[0].float()
    if pb is not None:
        bw = pb[0].t().view(h_kv, G, 1, N).expand(-1, -1, L, -1).gather(-1, got.unsqueeze(1).expand(-1, G, -1, -1))
        x = (x + bw.permute(2, 0, 1, 3).reshape(L, h_q, topk).bfloat16().float()).bfloat16().float()
    wr = torch.softmax(torch.cat([x, lse[0].unsqueeze(-1)], -1), -1)
    torch.testing.assert_close(w[0].float(), wr, atol=1e-2, rtol=2e-2)


def test_equal_scores_past_512_chunks(pkg, dev):
    """All scores equal: the lowest chunks win, also through the search over all scores."""
    L, N, D = 600, 1024, 64
    q = torch.zeros(1, L, 4, D, device=dev).bfloat16()
    lmk = torch.randn(1, N, 1, D, device=dev).bfloat16()
    lse = torch.zeros(1, L, 4, device=dev)
    idx, _, _ = pkg.topk_chunk_weights(q, lmk, lse, 32, 64, 1, q_offset=N * 64 - L)
    assert torch.equal(idx, torch.arange(32, device=dev, dtype=torch.int32).expand_as(idx))


@pytest.mark.parametrize("G,perq", [(4, False), (3, True), (8, False), (2, False)])
@pytest.mark.parametrize("lim,topk", [(20, 8), (40, 32), (400, 31), (512, 32), (530, 32), (1024, 32)])
@pytest.mark.parametrize("kind", ["shuffled", "column", "far column", "ties"])
def test_selection_by_candidate_count(pkg, dev, G, perq, lim, topk, kind):
    """Exact scores whose candidates (those above the weakest lane's second largest score) are few, more than 128, or more
    than the kernel keeps, and ties at the threshold: the best scores win, of equal ones the lowest chunks."""
    L, S, D = 640, 64, 64
    N = min(1024, lim + 4)
    gen = torch.Generator().manual_seed(lim)
    v = torch.randperm(N, generator=gen)
    if kind.endswith("column"):  # the chunks of one lane hold nothing above the given rank
        low = N - 1 - (N // 2 if kind.startswith("far") else min(150, N // 4))
        col = (torch.arange(N) % 16 == 5).nonzero().view(-1)
        weak = torch.randperm(low, generator=gen)[: len(col)]
        rest = torch.ones(N, dtype=torch.bool).index_fill(0, weak, False).nonzero().view(-1)
        v = torch.empty(N, dtype=torch.long)
        v[col], v[torch.arange(N) % 16 != 5] = weak, rest[torch.randperm(len(rest), generator=gen)]
    elif kind == "ties":
        v = v // 3
    lmk = torch.zeros(1, N, G if perq else 1, D)
    lmk[..., 0], lmk[..., 1] = (v // 8 * 8).view(1, N, 1), (v % 8).view(1, N, 1)  # (each exact in bf16, so is their sum)
    q = torch.zeros(1, L, G, D)
    q[..., :2] = 1
    off = lim * S - L  # the last query's window of one token begins in chunk lim
    idx, _, _ = pkg.topk_chunk_weights(q.bfloat16().to(dev), lmk.bfloat16().to(dev), torch.zeros(1, L, G, device=dev), topk, S, 1,
                                       q_offset=off, num_kv_heads=1)
    seen = ((torch.arange(L) + off) // S).clamp(0, N)
    order = (v * 2048 - torch.arange(N)).expand(L, N).masked_fill(torch.arange(N) >= seen.view(L, 1), -(1 << 30))
    best = order.topk(topk, -1)
    want = torch.where(best.values > -(1 << 30), best.indices, torch.full_like(best.indices, 1 << 20)).sort(-1).values
    want = torch.where(want == 1 << 20, torch.full_like(want, -1), want)
    assert torch.equal(idx[0, :, 0].cpu().long(), want)


@pytest.mark.parametrize("G,perq", [(4, False), (4, True), (8, False), (8, True)])
@pytest.mark.parametrize("lim,topk", [(40, 32), (512, 32), (1024, 32)])
@pytest.mark.parametrize("kind", ["shuffled", "column", "far column", "ties"])
@pytest.mark.parametrize("biased", [False, True])
def test_selected_scores_by_candidate_count(pkg, dev, G, perq, lim, topk, kind, biased):
    """The scores that come back, also with the last three bits of the logits in the prior bias, of which they carry none."""
    _by_candidate_count(pkg, dev, G, perq, lim, topk, kind, biased)


@pytest.mark.parametrize("G", [3, 4])
@pytest.mark.parametrize("L", [8300, 4000])
@pytest.mark.parametrize("kind", ["shuffled", "column", "far column", "ties"])
def test_selection_by_candidate_count_wide_heads(pkg, dev, G, L, kind):
    """Heads of 128 with a bias and 385 to 512 chunks: more than one round of wavefronts and less."""
    _by_candidate_count(pkg, dev, G, False, 512, 16, kind, True, L, 128, 2)


def _by_candidate_count(pkg, dev, G, perq, lim, topk, kind, biased, L=640, D=64, B=1):
    S = 64
    N = min(1024, lim + 4)
    gen = torch.Generator().manual_seed(lim)
    v = torch.randperm(N, generator=gen)
    if kind.endswith("column"):  # the chunks of one lane hold nothing above the given rank
        low = N - 1 - (N // 2 if kind.startswith("far") else min(150, N // 4))
        col = (torch.arange(N) % 16 == 5).nonzero().view(-1)
        weak = torch.randperm(low, generator=gen)[: len(col)]
        rest = torch.ones(N, dtype=torch.bool).index_fill(0, weak, False).nonzero().view(-1)
        v = torch.empty(N, dtype=torch.long)
        v[col], v[torch.arange(N) % 16 != 5] = weak, rest[torch.randperm(len(rest), generator=gen)]
    elif kind == "ties":
        v = v // 3
    lmk = torch.zeros(B, N, G if perq else 1, D)
    lmk[..., 0], lmk[..., 1] = (v // 8 * 8).view(1, N, 1), (v % 8).view(1, N, 1)  # (each exact in bf16, so is their sum)
    q = torch.zeros(B, L, G, D)
    q[..., :1 if biased else 2] = 1
    bias = (v % 8 / 8).view(1, N, 1).expand(B, N, G).contiguous().to(dev) if biased else None  # (logits are sums / 8)
    off = lim * S - L  # the last query's window of one token begins in chunk lim
    idx, scores, _ = pkg.topk_chunk_weights(q.bfloat16().to(dev), lmk.bfloat16().to(dev), torch.zeros(B, L, G, device=dev), topk, S, 1,
                                            q_offset=off, num_kv_heads=1, prior_b=bias, sm_scale=1 / 8)
    seen = ((torch.arange(L) + off) // S).clamp(0, N)
    order = (v * 2048 - torch.arange(N)).expand(L, N).masked_fill(torch.arange(N) >= seen.view(L, 1), -(1 << 30))
    best = order.topk(topk, -1)
    want = torch.where(best.values > -(1 << 30), best.indices, torch.full_like(best.indices, 1 << 20)).sort(-1).values
    want = torch.where(want == 1 << 20, torch.full_like(want, -1), want)
    assert torch.equal(idx[:, :, 0].cpu().long(), want.expand(B, L, topk))
    raw = (v // 8 * 8 if biased else v).to(torch.float32)[want.clamp(min=0)] / 8
    raw = raw.masked_fill(want < 0, float("-inf")).bfloat16()
    assert torch.equal(scores.cpu(), raw.unsqueeze(1).expand(B, L, G, topk))
