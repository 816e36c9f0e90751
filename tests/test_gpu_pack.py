"""The packed K and V of the sparse attention, word by word, against the layout by indexing."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Lkv,H,D,Dv", [(1, 64, 1, 64, 64), (2, 200, 3, 128, 64), (1, 333, 2, 64, 128), (1, 127, 2, 128, 128)])
def test_pack_kv_chunks(pkg, dev, B, Lkv, H, D, Dv):
    from hils_attention_amd.ops import _cabi
    lib, N = _cabi.load(), Lkv // 64
    gen = torch.Generator(device=dev).manual_seed(Lkv)
    k, v = (torch.randn(B, Lkv, H, d, device=dev, generator=gen).bfloat16() for d in (D, Dv))
    v[0, 5, 0, 3] = float("inf")   # a chunk that is not all numbers: the sign bit, infinities count and NaNs do not
    v[-1, 9, H - 1, Dv - 1] = float("nan")
    up = lambda n: (n + 255) // 256 * 256
    sizes = [up(B * H * N * 64 * Dv * 2), up(B * H * N * 64 * D * 2), up(B * H * N * 4)]
    ws = torch.zeros(sum(sizes), dtype=torch.uint8, device=dev)
    rc = lib.hils_pack_kv_chunks(_cabi.ptr(k), _cabi.ptr(v), _cabi.ptr(ws), ws.numel(), B, Lkv, H, D, Dv,
                                 torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    kc, vc = (x[:, :N * 64].view(B, N, 64, H, -1).permute(0, 3, 1, 2, 4).contiguous() for x in (k, v))
    lane = torch.arange(64, device=dev)
    m, j, e = (lane & 15).view(-1, 1), (lane >> 4).view(-1, 1), torch.arange(8, device=dev)
    blk = lambda n: torch.arange(n, device=dev).view(-1, 1, 1, 1)
    tok_k, d_k = blk(4) * 16 + m, blk(D // 32).view(1, -1, 1, 1) * 32 + j * 8 + e
    tok_v = blk(2).view(1, 2, 1, 1) * 32 + 16 * (e >> 2) + 4 * j + (e & 3)
    ref_k = kc[..., tok_k, d_k]
    ref_v = vc[..., tok_v, blk(Dv // 16) * 16 + m]
    bits = lambda x: x.contiguous().view(torch.int16).flatten()
    got_v = ws[:B * H * N * 64 * Dv * 2].view(torch.int16)
    got_k = ws[sizes[0]:sizes[0] + B * H * N * 64 * D * 2].view(torch.int16)
    assert torch.equal(got_v, bits(ref_v)) and torch.equal(got_k, bits(ref_k))
    top = vc.float().nan_to_num(0., float("inf"), -float("inf")).abs().flatten(3).amax(-1)
    top = torch.where(vc.float().isfinite().flatten(3).all(-1), top, -top)
    assert torch.equal(ws[sizes[0] + sizes[1]:][:B * H * N * 4].view(torch.float32), top.flatten())
