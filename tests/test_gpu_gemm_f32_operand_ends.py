"""fp32 products whose operands end with their allocations: nothing behind the last value is read.

Bar: against 64 bits, |gpu - exact| <= (K + 5) 2^-24 sum_k |a_ik b_kj| (K products and additions in any
order).
"""
import numpy as np
import pytest

from sapphire_amd import capi, synth
from tests import helpers as h

pytestmark = pytest.mark.gpu
TA, TB, OVERWRITE = capi.SPH_GEMM_TRANS_A, capi.SPH_GEMM_TRANS_B, capi.SPH_GEMM_OVERWRITE
UNIT = 2 << 20  # allocations are mapped in pieces of at most this


def at_the_end(x):
    """(buffer, address of x): x is the last of its allocation."""
    x = np.ascontiguousarray(x)
    before = -x.nbytes % UNIT
    buffer = capi.DeviceBuffer.from_array(
        np.concatenate([np.zeros(before // 4, np.float32), x.ravel()]))
    return buffer, buffer.at(before)


def check(M, N, K, flags):
    h.announce("sph_gemm_f32_ex operands at the end of their memory", (M, N, K), "flags", flags)
    A, B = synth.uniform(871, (M, K)), synth.uniform(872, (K, N))
    (dA, pA), (dB, pB) = (at_the_end(x.T if flags & f else x) for x, f in ((A, TA), (B, TB)))
    dC = capi.DeviceBuffer(4 * M * N)
    capi.call("sph_gemm_f32_ex", dC.ptr, pA, pB, M, N, K, 1, M * N, M * K, K * N, flags | OVERWRITE)
    got = dC.download(np.float32, (M, N))
    for d in (dA, dB, dC):
        d.release()
    A, B = A.astype(np.float64), B.astype(np.float64)
    assert np.all(np.abs(got - A @ B) <= (K + 5) * 2.0 ** -24 * (np.abs(A) @ np.abs(B)))


# (M, N, K): a last step of one, two and three values of k, on 64 x 64 tiles, 64 x 32 tiles with K
# split and 128 x 128 tiles; M and N no multiples of 4
@pytest.mark.parametrize("flags", [0, TA, TB, TA | TB])
@pytest.mark.parametrize("shape", [(1024, 1024, 257), (768, 640, 225), (2048, 2048, 289), (2048, 2048, 291),
                                   (1022, 1022, 258), (2046, 2046, 290), (1024, 1020, 1025)])
def test_last_step_of_less_than_a_chunk(dev, shape, flags):
    check(*shape, flags)


# few rows of an A stored K x M, and few columns of a B stored K x N: a last round of K that has less than
# four values
@pytest.mark.parametrize("shape", [(1, 1024, 2049), (2, 1024, 2049), (3, 1024, 4097), (1, 512, 2051),
                                   (1024, 1, 2049), (1024, 1, 2050), (512, 2, 2049), (1024, 3, 4097)])
def test_last_round_of_less_than_a_piece(dev, shape):
    for flags in (0, TA, TB, TA | TB):
        check(*shape, flags)
