"""Chunk log-Z gradients where the key gradient's walks are cut into segments and the units of (batch, KV head) are dealt
out to one, two, four or eight XCDs; against autograd in fp32."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _reference(q, k, W):
    B, L, HQ, D = q.shape
    H, N = k.shape[2], L // 64
    kx = k[:, : N * 64].repeat_interleave(HQ // H, 2)
    s = torch.stack([torch.matmul(q[b].transpose(0, 1), kx[b].permute(1, 2, 0).contiguous()) for b in range(B)])
    s = s.view(B, HQ, L, N, 64) / math.sqrt(D)
    s = torch.nn.functional.pad(s, (0, 0, 0, -(-L // 64) - N))  # a last chunk in part is behind no query
    N = -(-L // 64)
    far = torch.arange(L, device=q.device)[:, None] >= (torch.arange(N, device=q.device) + 1) * 64 + W - 1
    return torch.logsumexp(s, -1).masked_fill(~far, float("-inf")).permute(0, 2, 1, 3)


@pytest.mark.parametrize("B,L,HQ,H,D,W", [
    (1, 1600, 8, 1, 64, 64),     # one unit: its blocks over all XCDs
    (1, 1601, 16, 2, 64, 512),   # two
    (1, 1087, 3, 3, 128, 1),     # three units, one head each
    (2, 1300, 8, 2, 128, 200),   # four
    (2, 900, 16, 4, 64, 64),     # eight
    (1, 255, 4, 1, 64, 64),      # a last pair with one chunk, nothing cut
    (1, 64, 2, 1, 64, 64),       # no chunk behind any query
])
def test_logz_gradients(pkg, dev, B, L, HQ, H, D, W):
    gen = torch.Generator(device=dev).manual_seed(L)
    q = torch.randn(B, L, HQ, D, device=dev, generator=gen).bfloat16()
    k = torch.randn(B, L, H, D, device=dev, generator=gen).bfloat16()
    qd, kd = q.clone().requires_grad_(), k.clone().requires_grad_()
    out = pkg.exact_chunk_log_z_tl(qd, kd, chunk_size=64, window_size=W)
    qf, kf = q.float().requires_grad_(), k.float().requires_grad_()
    ref = _reference(qf, kf, W)
    seen = torch.isfinite(ref)
    assert torch.equal(torch.isfinite(out), seen)
    assert (out[seen] - ref[seen]).abs().max().item() < 2e-3 if seen.any() else True
    g = torch.where(seen, torch.randn(ref.shape, device=dev, generator=gen), torch.zeros((), device=dev))
    out.backward(g)
    torch.where(seen, ref, torch.zeros((), device=dev)).mul(g).sum().backward()
    for got, want, name in ((qd.grad, qf.grad, "dq"), (kd.grad, kf.grad, "dk")):
        err = (got.float() - want).norm() / want.norm().clamp_min(1e-6)
        assert err.item() < 1.5e-2, (name, err.item())
    cut = pkg.ops._cabi.load().hils_chunk_logz_bwd_dk_workspace(B, L, HQ, H, D, 64, W)
    assert (cut > 0) == (L > 800)


@pytest.mark.parametrize("D,scale,step", [(64, 6.0, 1.0), (128, 12.0, 1.0), (64, 1.0, 40.0)])
def test_logz_far_from_the_last_chunk(pkg, dev, D, scale, step):
    """Scores in the hundreds, and chunks whose log sums jump by hundreds from one to the next: the last chunk's log sum
    is no reference point for the next one's exponentials there."""
    gen = torch.Generator(device=dev).manual_seed(D)
    q = (torch.randn(1, 700, 8, D, device=dev, generator=gen) * scale).bfloat16()
    k = torch.randn(1, 700, 2, D, device=dev, generator=gen) * scale
    k[:, :, :, :] *= 1 + (step - 1) * (torch.arange(700, device=dev) // 64 % 2).view(1, -1, 1, 1)
    k = k.bfloat16()
    out = pkg.exact_chunk_log_z_tl(q, k, chunk_size=64, window_size=64)
    ref = _reference(q.float(), k.float(), 64)
    seen = torch.isfinite(ref)
    assert torch.equal(torch.isfinite(out), seen)
    assert (out[seen] - ref[seen]).abs().max().item() < 1e-5 * ref[seen].abs().max().item() + 2e-3
