"""The LDS of a decode step's row, at the longest contexts of each layout: every shape the one-launch step covers has
to fit a compute unit, and the longest ones have to run."""
import pytest
import torch

from util import assert_close_bf16, note

LDS = 160 * 1024  # of a compute unit


def _covered(lib, n, HQ, H, D, prior):
    return bool(lib.hils_decode_step_covers(1, 1, n, HQ, H, D, 32, 64, int(prior)))


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("G", range(1, 9))
@pytest.mark.parametrize("prior", [False, True])
def test_covered_rows_fit_the_lds(pkg, D, G, prior):
    from hils_attention_amd.ops import _cabi
    lib = _cabi.load()
    longest = 0
    for n in range(1, 4097):
        if not _covered(lib, n, G, 1, D, prior):
            continue
        longest = n
        for paged in (0, 1):
            need = lib.hils_decode_step_lds(n, G, 1, D, int(prior), paged)
            assert 0 < need <= LDS, f"{n} chunks: {need} bytes"
    assert longest >= 2048, "contexts of 128K tokens are covered"


@pytest.mark.gpu
@pytest.mark.parametrize("HQ,H,D,prior,paged_keys,n", [
    (32, 4, 128, True, False, 1472), (32, 4, 128, True, False, 1409),  # eight heads, the bias beside the logits
    (32, 4, 128, False, True, 2496), (40, 8, 128, True, True, 2433),   # ... with keys per page
    (32, 8, 128, True, True, 2624), (32, 8, 128, True, True, 2561),    # four heads, keys per page
    (32, 4, 64, True, False, 0), (16, 2, 128, True, False, 0), (4, 4, 128, True, True, 0),  # 0: the longest that is covered
])
def test_longest_rows_run(pkg, orc, dev, HQ, H, D, prior, paged_keys, n):
    from hils_attention_amd.ops import _cabi
    lib = _cabi.load()
    if n == 0:
        n = max(c for c in range(1, 4097) if _covered(lib, c, HQ, H, D, prior))
    assert _covered(lib, n, HQ, H, D, prior)
    note(f"decode_step {n} chunks HQ{HQ} H{H} D{D} prior={prior} paged_keys={paged_keys}")
    gen = torch.Generator().manual_seed(n)
    B, K, G, S = 2, 32, HQ // H, 64
    L = n * S
    q = torch.randn(B, 1, HQ, D, generator=gen).bfloat16()
    pages = B * n
    kp = torch.randn(pages, H, S, D, generator=gen).bfloat16()
    vp = torch.randn(pages, H, S, D, generator=gen).bfloat16()
    table = torch.randperm(pages, generator=gen).view(B, n)
    k = kp[table].permute(0, 1, 3, 2, 4).reshape(B, L, H, D)
    v = vp[table].permute(0, 1, 3, 2, 4).reshape(B, L, H, D)
    lmk_pages = torch.randn(pages, H, D, generator=gen).bfloat16()
    pb_pages = torch.randn(pages, HQ, generator=gen) if prior else None
    lse = torch.randn(B, 1, HQ, generator=gen) + 4
    lmk, pb = lmk_pages[table], None if pb_pages is None else pb_pages[table]
    to = lambda x: None if x is None else x.to(dev)
    dbg = {}
    if paged_keys:
        o, w, idx = pkg.paged_hils_attend(to(q), to(kp), to(vp), to(lmk_pages), to(table.int()), to(lse), L, K, 1,
                                          prior_pages=to(pb_pages), _debug=dbg)
    else:
        o, w, idx, dbg["scores"] = pkg.decode_step(to(q), to(lmk), to(k), to(v), to(lse), K, S, 1, q_offset=L - 1,
                                                   prior_b=to(pb), _debug=dbg)
    lim = orc.causal_chunk_limit(1, L - 1, 1, S)
    assert torch.equal(idx.cpu(), orc.topk_select(dbg["sel_logits"].cpu(), dbg["lse_total"].cpu(), lim, K))
    ref_w = orc.inter_chunk_softmax(dbg["scores"].cpu(), lse, None if pb is None else pb.bfloat16(),
                                    None if pb is None else idx.cpu())
    assert_close_bf16(w, ref_w, "weights", max_abs=8e-3)
    assert_close_bf16(o, orc.sparse_attn(q, k, v, w.cpu(), idx.cpu(), chunk_size=S), "output")
