"""Selection with one query head per KV head (queries as columns, threshold searched by value) against the kernel that the
exported logits run on (queries as rows, threshold searched bit by bit): ties, few and many chunks, scores of odd shapes."""
import pytest
import torch

from util import note

pytestmark = pytest.mark.gpu


def _inputs(kind, L, N, H, D, gen, dev):
    q = torch.randn(1, L, H, 1, D, device=dev, generator=gen)
    k = torch.randn(1, N, H, D, device=dev, generator=gen)
    bias = None
    if kind == "equal":          # every chunk ties
        q.zero_()
    elif kind == "few values":   # masses of ties on both sides of the threshold
        q = torch.randint(-1, 2, q.shape, device=dev, generator=gen).float()
        k = torch.randint(-1, 2, k.shape, device=dev, generator=gen).float()
    elif kind == "large":        # scores of thousands: one chunk has all the weight
        q *= 300.0
        k *= 30.0
    elif kind == "outlier":      # one score far above the others
        k[:, N // 2] *= 1000.0
    elif kind == "bias":
        bias = torch.randn(1, N, H, 1, device=dev, generator=gen) * 3
    elif kind == "closed":       # chunks that a bias takes out
        bias = torch.where(torch.rand(1, N, H, 1, device=dev, generator=gen) < 0.5, float("-inf"), 0.0)
    elif kind == "open":         # chunks that a bias puts before all others, more than are wanted
        bias = torch.where(torch.rand(1, N, H, 1, device=dev, generator=gen) < 0.5, float("inf"), 0.0)
    elif kind == "all open":
        bias = torch.full((1, N, H, 1), float("inf"), device=dev)
    elif kind == "one open":
        bias = torch.zeros(1, N, H, 1, device=dev)
        bias[:, N // 3] = float("inf")
    elif kind == "nan query":
        q[:, ::3, :, :, 5] = float("nan")
    elif kind == "nan key":
        k[:, ::4, :, 7] = float("nan")
    return q.bfloat16(), k.bfloat16(), bias


@pytest.mark.parametrize("kind", ["normal", "equal", "few values", "large", "outlier", "bias", "closed"])
@pytest.mark.parametrize("L,N,H,D,topk", [(333, 5, 2, 64, 8), (1000, 128, 3, 64, 32), (517, 129, 2, 128, 16),
                                          (800, 256, 2, 64, 32), (640, 200, 1, 128, 1)])
def test_one_head_equals_general_layout(pkg, dev, kind, L, N, H, D, topk):
    note(f"selection of one head, {kind}: L{L} N{N} H{H} D{D} top-{topk}")
    gen = torch.Generator(device=dev).manual_seed(N + topk)
    q, k, bias = _inputs(kind, L, N, H, D, gen, dev)
    lse = torch.randn(1, L, H, device=dev, generator=gen) + 3
    off = max(0, N * 64 - L + 65)  # the last query sees every chunk
    for offset in (off, 0):        # ... the first ones of the second call none
        args = (q, k, lse, topk, 64, 64)
        idx, sc = pkg.online_softmax_topk_head(*args, bias=bias, q_offset=offset, is_training=False)
        dbg = {}
        idx0, sc0 = pkg.online_softmax_topk_head(*args, bias=bias, q_offset=offset, is_training=False, _debug=dbg)
        if kind in ("equal", "few values", "closed", "outlier"):
            assert torch.equal(idx, idx0) and torch.equal(sc, sc0)
        # the two layouts add the log-sum-exp in another order: a difference of a few units in the last place, which
        # decides only between scores that are that close (below one selection in a thousand)
        diff = (idx != idx0).any(-1)
        assert diff.float().mean() <= 1e-3
        assert torch.equal(sc[~diff], sc0[~diff])
        if diff.any():
            # a score is rounded once more when the log-sum-exp is subtracted: only logits within a unit in the last place
            # of that difference (2^-23 of it, and as much again for the two log-sum-exps) can change places
            i1, i0, x = idx[diff].long(), idx0[diff].long(), dbg["sel_logits"][:, :, :, 0][diff]
            assert (i1[:, 1:] > i1[:, :-1]).all() and (i1 >= 0).all() and (i1 < N).all()
            a, b = (torch.gather(x, 1, i).sort(-1).values for i in (i1, i0))
            lse_total = dbg["lse_total"][..., 0][diff][:, None]
            assert ((a - b).abs() <= 2.0 ** -22 * (x.masked_fill(x.isinf(), 0).abs().amax(1, True) + lse_total.abs())).all()


# scores that are no numbers are not selected; infinite ones come first, at ties the lower chunks
@pytest.mark.parametrize("kind", ["open", "all open", "one open", "nan query", "nan key"])
@pytest.mark.parametrize("L,N,H,D,topk", [(333, 5, 2, 64, 8), (333, 128, 2, 64, 1), (500, 128, 3, 64, 32), (517, 129, 2, 128, 16),
                                          (400, 256, 2, 64, 32), (400, 256, 1, 128, 31)])
def test_one_head_without_numbers(pkg, dev, kind, L, N, H, D, topk):
    note(f"selection of one head, {kind}: L{L} N{N} H{H} D{D} top-{topk}")
    gen = torch.Generator(device=dev).manual_seed(N + topk)
    q, k, bias = _inputs(kind, L, N, H, D, gen, dev)
    lse = torch.randn(1, L, H, device=dev, generator=gen) + 3
    args = (q, k, lse, topk, 64, 64)
    off = max(0, N * 64 - L + 65)
    idx, _ = pkg.online_softmax_topk_head(*args, bias=bias, q_offset=off, is_training=False)
    idx0, _ = pkg.online_softmax_topk_head(*args, bias=bias, q_offset=off, is_training=False, _debug={})
    assert torch.equal(idx, idx0)
    if kind == "nan query":
        assert (idx[:, ::3] == -1).all() and (idx[:, L - L % 3 - 2, :, 0] >= 0).all()
    elif kind == "nan key":
        assert not ((idx >= 0) & (idx % 4 == 0)).any()
    elif kind == "all open":
        assert (idx[0, -1] == torch.where(torch.arange(topk, device=dev) < N, torch.arange(topk, device=dev), -1)).all()
    elif kind == "one open" and N >= topk:
        assert (idx[0, -1] == N // 3).any(-1).all()
