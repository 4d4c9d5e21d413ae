"""What a fp32 MultiHeadAttention block asks for behind what it keeps from forward to backward: room for dS where the
backward makes use of it, nothing where it does not."""
import ctypes

import pytest


def kept(B, H, E, D, Sq, Skv):
    """Projections, context, log-sum-exp, delta and the gradients of the first two, 256-byte aligned each."""
    q, k, stats = B * H * Sq * D, B * H * Skv * D, B * H * Sq
    regions = (q + 2 * k, q, stats, stats, q, q + 2 * k)
    return sum((4 * n + 255) // 256 * 256 for n in regions)


@pytest.mark.parametrize("B,H,Sq,Skv,pairs", [
    (1, 1, 1, 1, 1), (8, 8, 512, 512, 64), (3, 5, 97, 130, 15),  # all pairs fit
    (2, 64, 1024, 1024, 128), (2, 65, 1024, 1024, 128),         # 512 MB to the byte, and two pairs more than fit
    (8, 128, 512, 512, 512), (4, 200, 512, 500, 512),           # parts of 512 pairs, four workgroups each
    (1, 64, 2048, 2016, 32), (1, 64, 2100, 2000, 0),            # 32 pairs of 16 workgroups fill the chip twice, 31 do not
    (4, 8, 2500, 2500, 0), (6, 32, 2200, 2200, 0), (4, 32, 4096, 4096, 0), (1, 8, 5000, 5000, 0),
    (64, 16, 4096, 64, 512), (64, 16, 5000, 60, 0),             # one workgroup a pair
    (1, 1, 20000, 20000, 0),                                    # not even one pair fits
    (1, 1, 1, 1 << 23, 1), (1, 1, 1, 1 << 24, 0), (1, 1, 10, 9 << 20, 1), (1, 1, 10, 11 << 20, 0),  # a tile's rows past 4 GB
])
def test_room_for_scores_is_asked_for_where_it_is_used(ffk, B, H, Sq, Skv, pairs):
    E, D = 64, 32
    desc = ffk.mha_desc(B, H, E, E, E, D, D, D, E, Sq, Skv)
    asked = ffk.lib().ffk_mha_reserve_bytes(ctypes.byref(desc), ffk.FLOAT) - kept(B, H, E, D, Sq, Skv)
    assert asked == pairs * Sq * ((Skv + 31) // 32 * 32) * 4
    assert ffk.lib().ffk_mha_backward_workspace_bytes(ctypes.byref(desc), ffk.FLOAT) == asked
    assert ffk.lib().ffk_mha_backward_workspace_bytes(ctypes.byref(desc), ffk.BF16) == 0
    # in parts: two workgroups of 128 rows a CU, in half a GB
    most = (512 << 20) // (Sq * ((Skv + 31) // 32 * 32) * 4)
    if (Sq + 96) * ((Skv + 31) // 32 * 32) * 4 > 1 << 32:  # offsets of 32 bits
        most = 0
    assert pairs == (B * H if most >= B * H else most if most * (-(-min(Sq, Skv) // 128)) >= 512 else 0)
