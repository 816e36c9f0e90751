"""CPU: scratch sizes of the training calls over the lengths they take."""
import pytest


@pytest.mark.parametrize("HQ,H,D,K", [(32, 8, 128, 32), (32, 4, 64, 32), (16, 2, 64, 8), (16, 1, 64, 64), (16, 16, 64, 32)])
@pytest.mark.parametrize("B,L", [(1, 8192), (8, 8192), (1, 32768), (2, 32768), (1, 131072), (2, 131072)])
def test_backward_workspace_is_linear_in_the_length(pkg, B, L, HQ, H, D, K):
    from hils_attention_amd.ops import _cabi
    got = _cabi.load().hils_sparse_attn_bwd_workspace(B, L, L, HQ, H, D, D, K, HQ, 1, 64, 0.0)
    chunks, pairs, partial = B * H * (L // 64), B * L * H * K, 64 * 2 * D * 4
    # pairs, K and V packed, the partial results of at most twice 2049 segments, and of ranges of queries 1 GiB at most;
    # 64 MiB for the counters and items
    assert got > 0 and got <= 4 * pairs + chunks * 64 * 3 * D * 2 + 2 * 2049 * partial + (1 << 30) + (64 << 20)
    # past 32K tokens a range's cells are too small for any of it
    if L >= 32768:
        assert got <= 4 * pairs + chunks * (64 * 3 * D * 2 + 64) + 2 * 2049 * partial + (1 << 20)


# walks of dK: many segments only where they are long (a block's partial results are 128 D floats each)
@pytest.mark.parametrize("B,L,HQ,H,D,most", [(1, 4096, 16, 2, 64, 25), (2, 2048, 32, 8, 128, 6), (1, 8192, 32, 8, 128, 8),
                                             (1, 5000, 32, 4, 128, 16)])
def test_log_z_segments(pkg, B, L, HQ, H, D, most):
    from hils_attention_amd.ops import _cabi
    got = _cabi.load().hils_chunk_logz_bwd_dk_workspace(B, L, HQ, H, D, 64, 64)
    blocks = B * H * ((L // 64 + 2) // 2 if L % 128 else L // 128)
    assert 1 < got // (blocks * 128 * D * 4) <= most


# a row of d_weight per workgroup: per chunk with a chunk mean, without one per 64 tokens or fewer up to 256 workgroups
@pytest.mark.parametrize("B,L,H,D,S,rows", [(2, 1024, 16, 64, 64, 256), (2, 1024, 2, 64, 64, 128), (1, 300, 4, 128, 64, 75),
                                            (8, 8192, 16, 64, 64, 2048), (1, 100, 2, 64, 8, 13)])
def test_norm_rope_backward_workspace_goes_by_the_shape(pkg, B, L, H, D, S, rows):
    from hils_attention_amd.ops import _cabi
    assert _cabi.load().hils_norm_rope_pool_bwd_workspace(B, L, H, D, S) == rows * D * 4
