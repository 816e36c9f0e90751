"""A query or key that is not a number shows in the local branch's output, whichever kernel the shape runs on; a query's
reaches its own gradient and those of the keys, not those of the values, whichever tile it lies in."""
import pytest
import torch

from util import note

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("HQ,H,D,Dv", [(4, 4, 64, 64), (16, 2, 128, 128), (8, 1, 64, 128)])
@pytest.mark.parametrize("B,L,training", [(1, 96, True), (1, 3, False), (2, 3000, True)])  # rows of a few blocks, a step, tiles
def test_nan_shows(pkg, dev, HQ, H, D, Dv, B, L, training):
    note(f"local branch with a NaN, B{B} L{L} heads {HQ}/{H} x {D}/{Dv}")
    gen = torch.Generator(device=dev).manual_seed(L)
    Lk = L if training else L + 200
    r = lambda *s: torch.randn(*s, generator=gen, device=dev).bfloat16()
    q, k, v = r(B, L, HQ, D), r(B, Lk, H, D), r(B, Lk, H, Dv)
    o0, lse0 = pkg.flex_attn_tl(q, k, v, 64, 64, training=training)
    bad = q.clone()
    bad[B - 1, L - 1, 1, 5] = float("nan")
    o, lse = pkg.flex_attn_tl(bad, k, v, 64, 64, training=training)
    hit = torch.zeros(B, L, HQ, dtype=torch.bool, device=dev)
    hit[B - 1, L - 1, 1] = True
    assert o.isnan().all(-1).equal(hit) and o.isnan().any(-1).equal(hit)
    assert torch.equal(o[~hit], o0[~hit]) and torch.equal(lse[~hit], lse0[~hit])
    bad = k.clone()
    bad[0, Lk - 2, 0, 7] = float("nan")
    o, _ = pkg.flex_attn_tl(q, bad, v, 64, 64, training=training, mask_lmk=False)
    G = HQ // H
    assert o[0, L - 1, :G].isnan().all() and not o[0, L - 1, G:].isnan().any()


# the window split between two wavefronts (few blocks, a long window): the share that has the key, or only one of the two
# sees anything
@pytest.mark.parametrize("B,L,HQ,H,D,Dv", [(1, 1999, 16, 2, 64, 64), (1, 1024, 32, 8, 128, 128), (1, 1203, 16, 16, 64, 64)])
@pytest.mark.parametrize("t", [0, 70, 700, 1000])
def test_nan_shows_in_a_split_window(pkg, dev, B, L, HQ, H, D, Dv, t):
    note(f"split window with a NaN at {t}, L{L} heads {HQ}/{H} x {D}")
    gen = torch.Generator(device=dev).manual_seed(t)
    r = lambda *s: torch.randn(*s, generator=gen, device=dev).bfloat16()
    q, k, v = r(B, L, HQ, D), r(B, L, H, D), r(B, L, H, Dv)
    o0, lse0 = pkg.flex_attn_tl(q, k, v, 512, 64, mask_lmk=False)
    bad = q.clone()
    bad[0, t, 1, 5] = float("nan")
    o, lse = pkg.flex_attn_tl(bad, k, v, 512, 64, mask_lmk=False)
    hit = torch.zeros(B, L, HQ, dtype=torch.bool, device=dev)
    hit[0, t, 1] = True
    assert o.isnan().all(-1).equal(hit) and o.isnan().any(-1).equal(hit)
    assert torch.equal(o[~hit], o0[~hit]) and torch.equal(lse[~hit], lse0[~hit])
    bad = k.clone()
    bad[0, t, 0, 7] = float("nan")
    o, _ = pkg.flex_attn_tl(q, bad, v, 512, 64, mask_lmk=False)
    G = HQ // H
    last = min(L - 1, t // 64 * 64 + 63 + 511)  # the window of 512 begins in t's chunk and grows to its start
    sees = torch.zeros(L, dtype=torch.bool, device=dev)
    sees[t:last + 1] = True
    assert o[0, :, :G].isnan().any(-1).any(-1)[sees].all() and not o[0, :, G:].isnan().any()
    assert not o[0, ~sees, :G].isnan().any()


@pytest.mark.parametrize("HQ,H,D,Dv", [(8, 2, 64, 64), (8, 2, 128, 128), (4, 4, 128, 128), (16, 1, 64, 128), (4, 2, 128, 64)])
@pytest.mark.parametrize("W,mask_lmk", [(512, False), (300, True), (64, False)])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_gradients_of_a_query_that_is_no_number(pkg, dev, HQ, H, D, Dv, W, mask_lmk, bad):
    note(f"local branch backward, a query with {bad}, heads {HQ}/{H} x {D}/{Dv} window {W} mask {mask_lmk}")
    gen = torch.Generator(device=dev).manual_seed(W + D)
    B, L, t = 2, 901, 700
    r = lambda *s: torch.randn(*s, generator=gen, device=dev).bfloat16()
    q, k, v, d_o = r(B, L, HQ, D), r(B, L, H, D), r(B, L, H, Dv), r(B, L, HQ, Dv)

    def grads(q, d_o):
        ins = [x.clone().requires_grad_() for x in (q, k, v)]
        o, _ = pkg.flex_attn_tl(*ins, W, 64, mask_lmk=mask_lmk)
        return torch.autograd.grad(o, ins, d_o)

    without = d_o.clone()
    without[1, t, 1] = 0  # nothing but 0 comes from this row
    q0, k0, v0 = grads(q, without)
    q[1, t, 1, 5] = bad
    q1, k1, v1 = grads(q, d_o)
    assert torch.equal(v1, v0)
    hit = torch.zeros(B, L, HQ, dtype=torch.bool, device=dev)
    hit[1, t, 1] = True
    assert q1.isnan().any(-1).equal(hit) and torch.equal(q1[~hit], q0[~hit])
    assert torch.equal(k1[0], k0[0]) and k1[1, t, 1 // (HQ // H)].isnan().any()
