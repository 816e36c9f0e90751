"""Precision of the per-chunk log-sum-exp against 64 bits where neighbouring chunks' sums lie far apart."""
import math

import pytest
import torch

from util import note

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("HQ,H,D", [(4, 4, 64), (8, 2, 128), (8, 1, 64)])
def test_small_sums_between_large_ones(pkg, dev, HQ, H, D):
    """Every other chunk's log sum is 40 (58 in log2 units) above its neighbours', which are near zero: these must not be
    rounded at the neighbours' size.  Bound: the scores (32 before scaling, summed in fp32: half a unit in the last
    place 2e-6 times the scale 1/8 or less, averaged over the chunk) and the exponents' arguments (up to 8: 2.4e-7 each)
    stay under 1e-6 together; exponents and logs taken 58 away are rounded at 2e-6 each."""
    note(f"log Z, alternating chunks, heads {HQ}/{H} x {D}")
    gen = torch.Generator().manual_seed(17)
    L = 1024
    q = torch.randn(1, L, HQ, D, generator=gen) * 0.25
    k = torch.randn(1, L, H, D, generator=gen) * 0.25
    scale = 1 / math.sqrt(D)
    q[..., 0] = 1 / scale
    k[..., 0] = -4
    k.view(1, L // 64, 64, H, D)[:, 1::2, :, :, 0] = 36
    q, k = q.bfloat16().to(dev), k.bfloat16().to(dev)
    z = pkg.exact_chunk_log_z_tl(q, k, chunk_size=64, window_size=64)
    for h in range(HQ):
        s = torch.matmul(q[0, :, h].double(), k[0, :, h // (HQ // H)].double().t().contiguous()) * scale
        ref = torch.logsumexp(s.view(L, L // 64, 64), -1)
        seen = torch.isfinite(z[0, :, h])
        seen[:, 1::2] = False
        err = (z[0, :, h].double() - ref)[seen].abs()
        assert seen.sum() > 1000 and err.max().item() <= 1e-6, f"head {h}: {err.max().item():.2e}"
