"""Selection among 513 to 1024 chunks with queries enough for the two-pass kernel, and a bf16 lse beside an fp32 one."""
import pytest
import torch

from test_gpu_topk_1024 import test_topk_many_chunks as _check_selection
from util import note

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,N,h_kv,G,D,topk,perq,bias", [
    (4200, 600, 4, 4, 128, 32, False, False), (4501, 700, 4, 3, 64, 7, False, True), (5000, 1000, 8, 2, 64, 32, False, False),
    (4100, 777, 4, 5, 64, 32, True, True), (9001, 640, 4, 8, 64, 32, True, True), (6000, 1024, 4, 6, 128, 13, True, False),
])
def test_many_queries_many_chunks(pkg, orc, dev, L, N, h_kv, G, D, topk, perq, bias):
    note(f"selection L{L} N{N} h{h_kv} G{G} D{D} top-{topk} perq={perq} bias={bias}")
    _check_selection(pkg, orc, dev, L, N, h_kv, G, D, topk, perq, bias)


@pytest.mark.parametrize("N", [512, 600])
def test_bf16_lse_on_both_sides_of_the_line(pkg, dev, N):
    gen = torch.Generator(device=dev).manual_seed(N)
    L, HQ, H, D = 4200, 16, 4, 128
    q = torch.randn(1, L, HQ, D, device=dev, generator=gen).bfloat16()
    lmk = torch.randn(1, N, H, D, device=dev, generator=gen).bfloat16()
    lse = (torch.randn(1, L, HQ, device=dev, generator=gen) + 3).bfloat16()
    a = pkg.topk_chunk_weights(q, lmk, lse, 32, 64, 64, q_offset=N * 64 - L)
    b = pkg.topk_chunk_weights(q, lmk, lse.float(), 32, 64, 64, q_offset=N * 64 - L)
    for x, y in zip(a, b):
        assert torch.equal(x, y)
