"""The prefill attention kernel's fixed-point sums at the ends of their range: NaNs and infinities show in the output as
the oracle's do, and a column whose V is small beside the largest |V| keeps its precision."""
import pytest
import torch

from util import assert_close_bf16, note, rand_indices

pytestmark = pytest.mark.gpu

SHAPES = [(4, 4, 64, 64), (8, 2, 128, 128), (16, 1, 64, 128), (4, 2, 128, 64)]


def _inputs(HQ, H, D, Dv, seed, B=2, L=130, N=7, K=4):
    gen = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=gen).bfloat16()
    q, k, v = r(B, L, HQ, D), r(B, N * 64, H, D), r(B, N * 64, H, Dv)
    idx = rand_indices(B, L, H, K, 64, gen, causal=False, n_chunks=N)
    w = torch.softmax(torch.randn(B, L, HQ, K, generator=gen), -1).bfloat16()
    return q, k, v, w, idx


def _same_with_nans(o, ref):
    o, ref = o.float().cpu(), ref.float()
    assert torch.equal(o.isnan(), ref.isnan()), "NaNs in other places"
    assert torch.equal(o.isinf(), ref.isinf()) and torch.equal(o[o.isinf()], ref[ref.isinf()])
    fin = ref.isfinite()
    assert_close_bf16(o[fin], ref[fin], "the finite part")


@pytest.mark.parametrize("HQ,H,D,Dv", SHAPES)
@pytest.mark.parametrize("where", ["v_nan", "v_inf", "k_nan", "q_nan", "w_nan", "v_huge"])
def test_non_finite_inputs_show(pkg, orc, dev, HQ, H, D, Dv, where):
    note(f"sparse attention with {where}, heads {HQ}/{H} x {D}/{Dv}")
    q, k, v, w, idx = _inputs(HQ, H, D, Dv, 11)
    if where == "v_nan":
        v[0, 64 + 5, 0, 3] = v[1, 6 * 64 + 62, H - 1, Dv - 1] = float("nan")
    elif where == "v_inf":
        v[0, 64 + 5, 0, 3], v[0, 2 * 64, 0, 7] = float("inf"), float("-inf")
    elif where == "k_nan":
        k[0, 3 * 64 + 9, H - 1, 4] = float("nan")
    elif where == "q_nan":
        q[0, 17, HQ - 1, 5] = q[1, 129, 0, 0] = float("nan")
    elif where == "w_nan":
        w[0, 40, 1, 2] = float("nan")
    else:  # past what the fixed-point scale is made for
        v[0, 64 + 5, 0, :] *= 1e30
    ref = orc.sparse_attn(q, k, v, w, idx, chunk_size=64)
    o = pkg.HiLS_block_M_head(q.to(dev), k.to(dev), v.to(dev), w.to(dev), idx.to(dev), is_training=False)
    if where == "v_huge":  # rows beside the huge ones are held to their own size
        big = ref.abs().amax(-1) > 1e3
        assert big.any() and not big.all()
        assert_close_bf16(o.cpu().float()[~big], ref[~big], "rows without a huge V")
        assert_close_bf16(o.cpu().float()[big] / 1e30, ref[big] / 1e30, "rows with one")
    else:
        _same_with_nans(o, ref)


@pytest.mark.parametrize("HQ,H,D", [(4, 4, 64), (8, 4, 128), (8, 2, 64), (16, 2, 128)])
def test_small_columns_beside_an_outlier(pkg, orc, dev, HQ, H, D):
    """One value of 3e4 per chunk, on the variant that decode_step uses: the other columns' error is that of the bf16
    probabilities, as without it.  (The sums' unit is 2^-29 of sum|w| max|V| or less, 6e-5 here; with 20 bits it is 0.03, a
    third of a typical output.)"""
    from hils_attention_amd.ops import _cabi
    note(f"sparse attention with an outlier in V, heads {HQ}/{H} x {D}")
    q, k, v, w, idx = _inputs(HQ, H, D, D, 12)
    v[:, 10::64, :, 0] = 3e4
    ref = orc.sparse_attn(q, k, v, w, idx, chunk_size=64)
    B, L, Lkv, K = 2, 130, k.shape[1], idx.shape[-1]
    args = [x.to(dev) for x in (q, k, v, w, idx)]
    o = torch.empty(q.shape, dtype=torch.bfloat16, device=dev)
    ws = _cabi.sparse_attn_fwd_workspace(dev, B, L, Lkv, HQ, H, D, D, K, HQ, 1, 64, 0.0)
    assert ws is not None
    _cabi.call("hils_sparse_attn_fwd_fine", *map(_cabi.ptr, args), _cabi.ptr(o), _cabi.ptr(ws), _cabi.nbytes(ws), B, L, Lkv,
               HQ, H, D, D, K, K, 64, D ** -0.5, 1)
    assert_close_bf16(o[..., 1:], ref[..., 1:], "the other columns")
    assert_close_bf16(o[..., :1], ref[..., :1], "the outliers' column")


def test_decode_step_with_many_queries_shows_a_nan(pkg, orc, dev):
    """A NaN in a cached V shows in the rows that selected its chunk, in its column, whichever kernels run."""
    gen = torch.Generator().manual_seed(13)
    B, Lkv, HQ, H, D, K, N = 1, 4096, 4, 4, 64, 8, 64
    r = lambda *s: torch.randn(*s, generator=gen).bfloat16().to(dev)
    k, v, lmk = r(B, Lkv, H, D), r(B, Lkv, H, D), r(B, N, H, D)
    v[0, 20 * 64 + 3, 2, 5] = float("nan")
    for Lq in (512, 8):  # the prefill kernels, the one-launch kernel
        note(f"decode_step, {Lq} queries, NaN in V")
        q, lse = r(B, Lq, HQ, D), torch.randn(B, Lq, HQ, generator=gen).to(dev) + 2
        o, w, idx, _ = pkg.decode_step(q, lmk, k, v, lse, K, 64, 1, q_offset=Lkv - Lq)
        hit = (idx == 20).any(-1)
        hit[:, :, [0, 1, 3]] = False
        assert hit.any()
        want = torch.zeros_like(o, dtype=torch.bool)
        want[..., 5] = hit
        assert torch.equal(o.isnan(), want)
