"""Where the tiled GEMM kernels copy the chunks of an operand from (sapphire_amd/csrc/sph_copy_offsets.h,
reached through the host harness): no copy of any slab reaches past the operand, whatever its width
and depth; no device is needed."""
import ctypes

import pytest

from tests import host_layer as hl


def reach(name, *args):
    out = ctypes.c_longlong()
    assert getattr(hl.lib(), name)(*args, ctypes.byref(out)) == 0
    return out.value


# fp32 kernels: (K step, tile edge)
@pytest.mark.parametrize("bk,tile", [(32, 64), (32, 32), (16, 128)])
def test_fp32_quads_end_with_the_operand(bk, tile):
    for limit in [4, 5, 6, 7, 8, 9, 31, 33, 61, 63, 64, 65, 66, 67, 127, 128, 129, 130, 131, 255]:
        for K in [16, 17, 19, 31, 32, 33, 47, 48, 63, 64, 65, 95, 96, 97, 100]:
            got = reach("sphh_quad_copies_reach", K, limit, bk, tile, 1)
            # exactly to the end: the last row's last chunk is there
            assert got == 0, (limit, K)
            if limit % 4 == 0:  # the kernels without a last step of its own
                assert reach("sphh_quad_copies_reach", K, limit, bk, tile, 0) == 0, (limit, K)


# an operand stored with K contiguous: a last slab of every number of values, one to three among them
@pytest.mark.parametrize("bk", [16, 32])
def test_fp32_row_chunks_end_with_the_operand(bk):
    for K in list(range(16, 100)) + [1025, 1026, 1027]:
        for rows in [1, 3]:
            assert reach("sphh_row_chunks_reach", K, rows, bk) == 0, (K, rows)


# few rows of an operand stored k-major: (values of k a round, most rows, pieces a round)
@pytest.mark.parametrize("wavefronts,rows", [(1, 4), (4, 4), (8, 4), (1, 8), (2, 8), (4, 8), (8, 8),
                                             (1, 16), (2, 16), (4, 16), (8, 16)])
def test_fp32_pieces_end_with_the_operand(wavefronts, rows):
    step = 256 * wavefronts
    for M in range(1, rows + 1):
        for K in [64, 65, 66, 67, 255, step - 1, step, step + 1, step + 2, step + 3, 2 * step + 1]:
            assert reach("sphh_pieces_reach", K, M, step, rows * 64 * wavefronts) <= 0, (K, M)


# fp16 kernels: (K step, tile edge, fewest slabs of broken rows)
@pytest.mark.parametrize("bk,tile", [(64, 64), (32, 128)])
def test_fp16_chunks_end_with_the_operand(bk, tile):
    for limit in list(range(8, 26)) + [57, 63, 64, 65, 121, 127, 128, 129, 135, 255]:
        for K in [2 * bk, 2 * bk + 1, 3 * bk - 1, 3 * bk, 3 * bk + 7, 5 * bk + 33]:
            assert reach("sphh_chunk_copies_reach", K, limit, bk, tile) == 0, (limit, K)
