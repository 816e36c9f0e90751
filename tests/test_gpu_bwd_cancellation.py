"""dQ where the softmax's backward cancels exactly: one token has all the probability, so dP - sum(P dP) is zero."""
import pytest
import torch

from util import note

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("HQ,H,D", [(4, 4, 64), (8, 2, 128), (16, 2, 64), (4, 2, 128)])
def test_dq_of_a_certain_softmax_is_zero(pkg, dev, HQ, H, D):
    """q is along the first axis, every key far down it but one, which is orthogonal to q: its score is exactly 0, its
    probability exactly 1 and the others' underflow.  dS is zero whatever w, dO and V are, and so is dQ."""
    note(f"dQ of a certain softmax, heads {HQ}/{H} x {D}")
    gen = torch.Generator().manual_seed(19)
    B, L, N, K = 1, 128, 4, 2
    q = torch.zeros(B, L, HQ, D)
    q[..., 0] = 4096 + 32 * (torch.arange(L).view(1, L, 1) % 7)
    k = torch.zeros(B, N * 64, H, D)
    k[..., 0] = -1
    k[:, 5::64, :, 0] = 0
    k[:, 5::64, :, 1:] = 1 + torch.rand(B, N, H, D - 1, generator=gen)
    # (near the bounds of the fixed-point sums, whose unit would hide what does not cancel: 2^-25 of f dP)
    v = 1 + torch.rand(B, N * 64, H, D, generator=gen)
    d_o = torch.zeros(B, L, HQ, D)
    d_o[..., 3] = 1 + torch.rand(B, L, HQ, generator=gen)
    w = 1 + torch.rand(B, L, HQ, K, generator=gen)
    idx = torch.tensor([1, 3], dtype=torch.int32).expand(B, L, H, K).contiguous()
    q, k, v = (x.bfloat16().to(dev).requires_grad_() for x in (q, k, v))
    w, idx, d_o = w.bfloat16().to(dev), idx.to(dev), d_o.bfloat16().to(dev)
    # (a scale that is no power of two: products with it are rounded)
    o = pkg.HiLS_block_M_head(q, k, v, w, idx, sm_scale=0.1)
    want = (v.detach()[:, [64 + 5, 192 + 5]].float().repeat_interleave(HQ // H, 2).unsqueeze(1)
            * w.float().permute(0, 1, 3, 2).unsqueeze(-1)).sum(2)
    torch.testing.assert_close(o.float(), want, atol=2e-2, rtol=1e-2)
    dq, dv = torch.autograd.grad(o, (q, v), d_o)
    assert dv.abs().max() > 0
    assert dq.abs().max().item() == 0.0, f"dQ up to {dq.abs().max().item():.2e}"
