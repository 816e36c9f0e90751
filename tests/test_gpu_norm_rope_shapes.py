"""norm_rope_pool at the edges of its launch shapes: head counts that leave one, two or eight heads per workgroup,
four to sixteen wavefronts, ragged chunks, chunk lengths that are no multiple of a wavefront's tokens."""
import pytest
import torch

from util import assert_close_bf16, note

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,L,H,D,S", [(1, 64, 16, 64, 64),     # eight heads, one token a step, sixteen wavefronts
                                       (3, 1999, 2, 64, 64),    # two heads, four tokens a step, ragged tail
                                       (2, 515, 6, 128, 64),    # two of six heads
                                       (1, 130, 5, 128, 40),    # one head, chunk of ten steps
                                       (2, 97, 4, 256, 33),     # an odd chunk
                                       (40, 2048, 8, 128, 64)])  # more workgroups than fill the chip
def test_norm_rope_pool_shapes(pkg, orc, dev, B, L, H, D, S):
    note(f"norm_rope_pool B{B} L{L} H{H} D{D} S{S}")
    gen = torch.Generator().manual_seed(43)
    rows = min(B, 3)
    x = torch.randn(rows, L, H, D, generator=gen).bfloat16()
    w = (torch.rand(D, generator=gen) + 0.5).bfloat16()
    ang = torch.rand(L, D // 2, generator=gen) * 6.0
    cos, sin = (torch.cat([f(ang), f(ang)], -1).bfloat16() for f in (torch.cos, torch.sin))
    g_o = torch.randn(rows, L, H, D, generator=gen).bfloat16()
    g_l = torch.randn(rows, L // S, H, D, generator=gen).bfloat16()
    rep = lambda t: t.repeat(-(-B // rows), 1, 1, 1)[:B].to(dev)  # noqa: E731
    xd, wd = rep(x).requires_grad_(), w.to(dev).requires_grad_()
    out, lmk = pkg.norm_rope_pool(xd, wd, cos.to(dev), sin.to(dev), S)
    x64, w64 = x.double().requires_grad_(), w.double().requires_grad_()
    o64, l64 = orc.norm_rope_pool(x64, w64, cos.double(), sin.double(), S)
    assert_close_bf16(out[:rows], o64.detach().float(), "out")
    assert_close_bf16(lmk[:rows], l64.detach().float(), "pooled keys")
    dx, dw = torch.autograd.grad([out, lmk], [xd, wd], [rep(g_o), rep(g_l)])
    dx64, = torch.autograd.grad([o64, l64], [x64], [g_o.double(), g_l.double()], retain_graph=True)
    assert_close_bf16(dx[:rows], dx64.float(), "dx")
    # the batch repeats its first rows: the weight's gradient is the sum over the repeats
    dw64 = sum(torch.autograd.grad([o64[i % rows], l64[i % rows]], [w64], [g_o[i % rows].double(), g_l[i % rows].double()],
                                   retain_graph=True)[0] for i in range(B))
    assert dw.dtype == torch.bfloat16
    assert_close_bf16(dw, dw64.float(), "d_weight")
    w32 = w.float().to(dev).requires_grad_()  # an fp32 weight gets its gradient in fp32
    out32, _ = pkg.norm_rope_pool(xd.detach(), w32, cos.to(dev), sin.to(dev), S, pool=False)
    dw32, = torch.autograd.grad(out32, w32, rep(g_o))
    assert dw32.dtype == torch.float32


# without the mean a workgroup owns fewer tokens than a chunk: the same arithmetic row by row, so the same bits, and a
# weight gradient that differs by the order of its fp32 sum (2^-24 times sqrt of the rows added, rounded to bf16)
@pytest.mark.parametrize("B,L,H,D", [(1, 1999, 16, 64), (2, 1024, 2, 64), (1, 77, 5, 128), (3, 333, 4, 256), (1, 1, 1, 64),
                                     (16, 4096, 16, 64)])
def test_norm_rope_without_mean_equals_with(pkg, dev, B, L, H, D):
    gen = torch.Generator(device=dev).manual_seed(47)
    x = torch.randn(B, L, H, D, device=dev, generator=gen).bfloat16().requires_grad_()
    w = (torch.rand(D, device=dev, generator=gen) + 0.5).bfloat16().requires_grad_()
    ang = torch.rand(L, D // 2, device=dev, generator=gen) * 6.0
    cos, sin = (torch.cat([f(ang), f(ang)], -1).bfloat16() for f in (torch.cos, torch.sin))
    g_o = torch.randn(B, L, H, D, device=dev, generator=gen).bfloat16()
    got = []
    for pool in (False, True):
        out, lmk = pkg.norm_rope_pool(x, w, cos, sin, 64, pool=pool)
        z = [] if lmk is None or not lmk.numel() else [torch.zeros_like(lmk)]
        got.append([out, *torch.autograd.grad([out, *([lmk] if z else [])], [x, w], [g_o, *z])])
    (o1, dx1, dw1), (o2, dx2, dw2) = got
    assert torch.equal(o1, o2) and torch.equal(dx1, dx2)
    assert (dw1.float() - dw2.float()).abs().max() <= 2.0 ** -7 * dw2.float().abs().max()
