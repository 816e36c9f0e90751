"""chunk_weights backward with every combination of inputs that want a gradient."""
import itertools

import pytest
import torch

from util import assert_close_bf16, note

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("want", [w for w in itertools.product((False, True), repeat=3) if any(w)])
def test_only_what_is_asked_for(pkg, dev, want):
    note(f"chunk_weights gradients of scores, lse, prior: {want}")
    gen = torch.Generator(device=dev).manual_seed(23)
    B, L, HQ, H, K, N = 1, 64, 16, 4, 8, 100000
    sc = torch.randn(B, L, HQ, K, device=dev, generator=gen).bfloat16()
    lse = torch.randn(B, L, HQ, device=dev, generator=gen) + 1
    pb = torch.randn(B, N, HQ, device=dev, generator=gen).bfloat16()
    idx = torch.randint(0, N, (B, L, H, K), device=dev, generator=gen, dtype=torch.int32)
    g = torch.randn(B, L, HQ, K + 1, device=dev, generator=gen).bfloat16()
    ins = [x.clone().requires_grad_(w) for x, w in zip((sc, lse, pb), want)]
    ref_in = [x.float().clone().requires_grad_() for x in (sc, lse, pb)]
    at = idx.long().repeat_interleave(HQ // H, 2)                                            # (B, L, HQ, K)
    bias = ref_in[2][0].t()[torch.arange(HQ, device=dev).view(1, 1, HQ, 1), at]
    ref = torch.softmax(torch.cat([ref_in[0] + bias, ref_in[1].unsqueeze(-1)], -1), -1)
    ref_g = torch.autograd.grad(ref, ref_in, g.float())
    out = pkg.chunk_weights(ins[0], ins[1], ins[2], idx)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    out.backward(g)
    torch.cuda.synchronize()
    used = torch.cuda.max_memory_allocated() - before
    if not want[2]:
        assert used < 4 * N * HQ, "the prior's gradient was not asked for: nothing of its size is allocated"
    for name, x, w, r in zip(("scores", "lse", "prior"), ins, want, ref_g):
        assert (x.grad is not None) == w
        if w:
            assert_close_bf16(x.grad, r, name)


@pytest.mark.parametrize("B,K,L,repeated", [(2, 8, 4096, False), (2, 32, 2500, False), (2, 16, 700, True), (129, 32, 1001, False), (300, 16, 1801, False)])
def test_prior_gradient_of_large_gradients(pkg, dev, B, K, L, repeated):
    """Sums of a run of rows far past 2^23, small ones beside them, one index in all slots of a row, and a gradient that
    is no number; one round of runs of rows, two and three."""
    note(f"chunk_weights, large gradients, B{B} K={K} L{L} repeated {repeated}")
    gen = torch.Generator(device=dev).manual_seed(K)
    HQ, H, N = 2, 1, 64
    sc = torch.randn(B, L, HQ, K, device=dev, generator=gen).bfloat16()
    lse = torch.randn(B, L, HQ, device=dev, generator=gen) + 1
    pb = torch.zeros(B, N, HQ, device=dev, requires_grad=True)
    idx = torch.arange(K, device=dev, dtype=torch.int32).expand(B, L, H, K).contiguous()
    if repeated:
        idx.fill_(5)
    g = torch.randn(B, L, HQ, K + 1, device=dev, generator=gen)
    g[..., 0] += 2.0 ** 20
    g[:, :, 1] *= 2.0 ** 12
    g[1, 7, 0, 3] = float("nan")
    g = g.bfloat16()
    pkg.chunk_weights(sc, lse, pb, idx).backward(g)
    x = torch.cat([sc.double(), lse.double().unsqueeze(-1)], -1)
    y, g6 = torch.softmax(x, -1), g.double()
    d = (y * (g6 - (y * g6).sum(-1, keepdim=True)))[..., :K]
    size = (y * (g6.abs() + (y * g6).abs().sum(-1, keepdim=True)))[..., :K]
    at = idx.long().view(B, L, 1, K).expand(B, L, HQ, K).permute(0, 1, 3, 2).reshape(B, L * K, HQ)
    ref, most = (torch.zeros(B, N, HQ, dtype=torch.float64, device=dev).scatter_add_(1, at, t.permute(0, 1, 3, 2).reshape(B, L * K, HQ))
                 for t in (d, size))
    # an element is within some 16 roundings of its terms (exponentials, sum of K + 1, quotient), sums of n within n more
    bad = ref.isnan()
    assert bad[1, 5 if repeated else 3, 0] and pb.grad.isnan().equal(bad)
    err = (pb.grad.double() - ref).abs()
    assert bool((err <= (2 * K + 16 + L * K) * 2.0 ** -24 * most)[~bad].all())
