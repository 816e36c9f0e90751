"""Exact log Z and dQ: walks of one to nine chunks (the kernels take four steps a round and load three ahead), keys whose
sums jump between neighbouring chunks, the landmark mask, negative windows, keys at any address."""
import pytest
import torch

from util import LSE_TOL, assert_close_bf16, assert_close_f32, note

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("HQ,H,D", [(2, 2, 64), (8, 2, 128), (16, 1, 64), (4, 4, 128)])
@pytest.mark.parametrize("chunks,rest,mask_lmk", [(1, 0, False), (2, 1, True), (3, 63, False), (4, 0, True), (5, 17, False),
                                                  (6, 40, True), (9, 5, False)])
def test_walks(pkg, orc, dev, HQ, H, D, chunks, rest, mask_lmk):
    note(f"log Z walks {chunks} chunks + {rest}, heads {HQ}/{H} x {D}, mask {mask_lmk}")
    gen = torch.Generator().manual_seed(chunks * 100 + rest)
    L, W = (chunks + 1) * 64 + rest, 64
    q = torch.randn(2, L, HQ, D, generator=gen)
    k = torch.randn(2, L, H, D, generator=gen)
    k[:, 64:192] *= 5  # near its predecessor's sum, far, far and so on
    k[1, 256:320] *= 0.1
    q, k = q.bfloat16(), k.bfloat16()
    qd, kd = q.to(dev).requires_grad_(not mask_lmk), k.to(dev).requires_grad_(not mask_lmk)
    z = pkg.exact_chunk_log_z_tl(qd, kd, chunk_size=64, window_size=W, mask_lmk=mask_lmk)
    qf, kf = q.float().requires_grad_(), k.float().requires_grad_()
    ref = orc.exact_chunk_log_z(qf, kf, chunk_size=64, window_size=W, mask_lmk=mask_lmk)
    assert_close_f32(z.detach(), ref.detach(), LSE_TOL, "log_z")
    if mask_lmk:
        return  # forward only
    finite = torch.isfinite(ref)
    g = torch.randn(ref.shape, generator=gen) * finite
    z.backward(g.to(dev))
    torch.where(finite, ref, torch.zeros(())).mul(g).sum().backward()
    assert_close_bf16(qd.grad, qf.grad, "dq")
    assert_close_bf16(kd.grad, kf.grad, "dk")


@pytest.mark.parametrize("HQ,H,D", [(4, 2, 64), (16, 1, 128)])
@pytest.mark.parametrize("L,W", [(215, -1), (215, -40), (130, -63), (193, -200)])
def test_negative_window(pkg, orc, dev, HQ, H, D, L, W):
    """Chunks that end behind a query are visible to it up to the query itself, a ragged last one up to its end."""
    note(f"log Z, window {W}, L{L} heads {HQ}/{H} x {D}")
    gen = torch.Generator().manual_seed(L - W)
    q, k = torch.randn(2, L, HQ, D, generator=gen).bfloat16(), torch.randn(2, L, H, D, generator=gen).bfloat16()
    qd, kd = q.to(dev).requires_grad_(), k.to(dev).requires_grad_()
    z = pkg.exact_chunk_log_z_tl(qd, kd, chunk_size=64, window_size=W)
    qf, kf = q.float().requires_grad_(), k.float().requires_grad_()
    ref = orc.exact_chunk_log_z(qf, kf, chunk_size=64, window_size=W)
    assert_close_f32(z.detach(), ref.detach(), LSE_TOL, "log_z")
    finite = torch.isfinite(ref)
    g = torch.randn(ref.shape, generator=gen) * finite
    z.backward(g.to(dev))
    torch.where(finite, ref, torch.zeros(())).mul(g).sum().backward()
    assert_close_bf16(qd.grad, qf.grad, "dq")
    assert_close_bf16(kd.grad, kf.grad, "dk")


@pytest.mark.parametrize("HQ,H,D", [(4, 2, 64), (2, 2, 64), (8, 1, 128), (4, 1, 128)])
def test_gradients_beside_large_scores(pkg, orc, dev, HQ, H, D):
    """Scores past the exponential's range in chunks that a query does not see, but its workgroup walks."""
    L, W = 470, 64
    note(f"log Z, large scores, heads {HQ}/{H} x {D}")
    gen = torch.Generator().manual_seed(D + HQ)
    q, k = 8 * torch.randn(1, L, HQ, D, generator=gen), 8 * torch.randn(1, L, H, D, generator=gen)
    q, k = q.bfloat16(), k.bfloat16()
    qd, kd = q.to(dev).requires_grad_(), k.to(dev).requires_grad_()
    z = pkg.exact_chunk_log_z_tl(qd, kd, chunk_size=64, window_size=W)
    qf, kf = q.double().requires_grad_(), k.double().requires_grad_()
    s = torch.einsum("blhd,bjhd->blhj", qf, kf.repeat_interleave(HQ // H, 2)) * D ** -0.5
    n = z.shape[-1]
    s = torch.nn.functional.pad(s, (0, 64 * n - L), value=float("-inf")).unflatten(-1, (n, 64))
    seen = (torch.arange(1, n + 1) * 64 <= torch.arange(L).view(-1, 1) - W + 1).view(1, L, 1, n)
    assert s.detach().masked_fill(seen.unsqueeze(-1), 0)[0, :-64].amax() > 89  # (the exponential's range ends at 88.7)
    g = torch.randn(z.shape, generator=gen) * seen
    z.backward(g.to(dev))
    s.masked_fill(~seen.unsqueeze(-1), 0).logsumexp(-1).mul(g * seen).sum().backward()
    assert_close_bf16(qd.grad, qf.grad.float(), "dq")
    assert_close_bf16(kd.grad, kf.grad.float(), "dk")


@pytest.mark.parametrize("HQ,H,D", [(4, 2, 64), (8, 1, 128)])
@pytest.mark.parametrize("at", [1, 4])
def test_keys_at_any_address(pkg, dev, HQ, H, D, at):
    """A contiguous view that begins 2 or 8 bytes behind a multiple of 16: the same as a copy of it, by the operator and by
    the C entries."""
    from hils_attention_amd.ops import _cabi
    lib, B, L, W = _cabi.load(), 2, 470, 64
    note(f"log Z, keys {2 * at} bytes off, heads {HQ}/{H} x {D}")
    gen = torch.Generator(device=dev).manual_seed(at)
    store = torch.randn(at + B * L * H * D, device=dev, generator=gen).bfloat16()
    view = store[at:].view(B, L, H, D)
    assert view.is_contiguous() and view.data_ptr() % 16
    q = torch.randn(B, L, HQ, D, device=dev, generator=gen).bfloat16()
    out = []
    for k in (view, view.clone()):
        a, b = q.clone().requires_grad_(), k.detach().requires_grad_()
        z = pkg.exact_chunk_log_z_tl(a, b, chunk_size=64, window_size=W)
        g = torch.ones_like(z).masked_fill(z == float("-inf"), 0.)
        out.append([z.detach(), *torch.autograd.grad(z, [a, b], g)])
    assert all(torch.equal(x, y) for x, y in zip(*out))
    z, dq, dk = out[1]
    cz, cq, ck = torch.empty_like(z), torch.empty_like(dq), torch.empty_like(dk)
    p, s = _cabi.ptr, torch.cuda.current_stream().cuda_stream
    g = torch.ones_like(z).masked_fill(z == float("-inf"), 0.)
    assert lib.hils_chunk_logz_fwd(p(q), p(view), p(cz), B, L, HQ, H, D, 64, W, D ** -0.5, 0, s) == 0
    assert lib.hils_chunk_logz_bwd_dq(p(q), p(view), p(z), p(g), p(cq), B, L, HQ, H, D, 64, W, D ** -0.5, s) == 0
    assert lib.hils_chunk_logz_bwd_dk(p(q), p(view), p(z), p(g), p(ck), B, L, HQ, H, D, 64, W, D ** -0.5, s) == 0
    assert_close_f32(cz, z, LSE_TOL, "log_z")
    assert_close_bf16(cq, dq, "dq")
    assert_close_bf16(ck, dk, "dk")
