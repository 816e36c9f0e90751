"""Which kernels a step of many queries per sequence runs on."""
import math

import pytest
import torch

from util import note


@pytest.mark.parametrize("B,L,ctx,HQ,H,D,K,perq,prefill", [
    # measured, us, one launch / prefill kernels
    (1, 2048, 65500, 32, 8, 128, 32, 0, 1),   # 2160 / 625
    (1, 512, 65536, 32, 8, 128, 32, 0, 1),    # 529 / 312
    (1, 128, 65536, 32, 8, 128, 32, 0, 0),    # 144 / 209
    (1, 163, 35000, 16, 2, 64, 32, 0, 0),     # 23 / 55
    (1, 512, 4133, 4, 4, 64, 8, 0, 1),        # 72 / 49
    (1, 2048, 49200, 32, 4, 128, 32, 1, 1),   # more than 512 chunks, a key for each of eight heads
    (1, 128, 49200, 32, 4, 128, 32, 1, 0),
    (1, 63, 65536, 32, 8, 128, 32, 0, 0),     # the prefill kernels start at 64 queries
    # one head per KV head on short caches
    (1, 96, 8192, 16, 16, 64, 8, 0, 1),       # 56 / 50
    (1, 64, 8192, 32, 32, 128, 16, 0, 1),     # 154 / 104
    (1, 320, 8192, 4, 4, 64, 8, 0, 1),        # 46 / 43
    (1, 256, 8192, 4, 4, 64, 8, 0, 0),        # 38 / 40
    # no prefill attention kernel for these groups: the shape-generic one is ten times as slow as the one-launch step
    (1, 512, 16400, 40, 8, 128, 32, 0, 0), (1, 2048, 65536, 12, 4, 64, 32, 0, 0), (1, 1024, 16400, 48, 8, 128, 8, 0, 0),
    (1, 1024, 16400, 28, 4, 64, 8, 0, 0),
])
def test_the_rule(pkg, B, L, ctx, HQ, H, D, K, perq, prefill):
    from hils_attention_amd.ops import _cabi
    assert _cabi.load().hils_decode_step_prefill_ahead(B, L, ctx // 64, ctx, HQ, H, D, K, perq) == prefill


@pytest.mark.gpu
@pytest.mark.parametrize("L,ctx,HQ,H,D", [(300, 8229, 40, 8, 128), (200, 4133, 12, 4, 64)])
def test_uneven_groups_stay_on_the_one_launch_kernel(pkg, dev, L, ctx, HQ, H, D):
    from hils_attention_amd.ops import _cabi
    note(f"decode_step {L} queries at {ctx}, heads {HQ}/{H} x {D}")
    gen = torch.Generator(device=dev).manual_seed(L)
    r = lambda *s: torch.randn(*s, generator=gen, device=dev).bfloat16()
    N, K, scale = ctx // 64, 16, 1 / math.sqrt(D)
    q, lmk, k, v = r(1, L, HQ, D), r(1, N, H, D), r(1, ctx, H, D), r(1, ctx, H, D)
    lse = torch.randn(1, L, HQ, generator=gen, device=dev) + 3
    out = pkg.decode_step(q, lmk, k, v, lse, K, 64, 1, q_offset=ctx - L)
    o, w, idx, sc = (torch.empty_like(x) for x in out)
    _cabi.call("hils_decode_step", *map(_cabi.ptr, (q, lmk, k, v, lse, None, idx, sc, w, o)), None, None, 1, L, ctx, N, HQ, H,
               D, K, 64, 1, ctx - L, scale, scale, 1, 0, N, 0)
    for a, b in zip(out, (o, w, idx, sc)):
        assert torch.equal(a, b)
