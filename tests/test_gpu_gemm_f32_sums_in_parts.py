"""fp32 products with an M or N that is no multiple of 4: the error of their sums.

Bar: rounding a result costs at most 2^-24 of it, uniformly distributed over a mantissa that is
itself spread over [1, 2): 2.5e-8 of the result's root mean square.  A chain of n additions of
independent products of variance v rounds partial sums of variance v, 2 v, ..., n v: n^2 / 2 of
them in all; four chains of K / 4 make K^2 / 8, and adding up the parts and the old value less than
5 K more.  Relative to a sum of K products that is 2.5e-8 sqrt(K / 8 + 5); 12 % are added for
the sample.  (One chain has twice that, two chains 1.4 times.)  Last rows and columns, which feed
from broken chunks, and the rest are held to it separately.
"""
import numpy as np
import pytest

from sapphire_amd import capi, synth
from tests import helpers as h

pytestmark = pytest.mark.gpu
TA, TB, OVERWRITE = capi.SPH_GEMM_TRANS_A, capi.SPH_GEMM_TRANS_B, capi.SPH_GEMM_OVERWRITE

# (M, N, K): 64 x 64 tiles with a last step and without, K in whole 32-wide, in 16-wide and in
# broken steps; 64 x 32 tiles with K split; 128 x 128 tiles, K of a few steps and of many; few rows
# or columns of many
SHAPES = [(1001, 1003, 1000), (1001, 1024, 784), (1001, 1024, 768), (1024, 1001, 256),
          (16384, 10, 513), (65, 4096, 1024), (513, 514, 999), (3001, 2687, 129),
          (3001, 2687, 700), (2687, 3000, 1025)]


def relative(error, exact):
    return float(np.sqrt(np.mean(error ** 2) / np.mean(exact ** 2))) if error.size else 0.0


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("shape", SHAPES)
def test_error_of_four_parts(dev, shape, offset):
    M, N, K = shape
    A, B = synth.uniform(861, (M, K)), synth.uniform(862, (K, N))
    exact = A.astype(np.float64) @ B.astype(np.float64)
    bar = 1.12 * 2.5e-8 * np.sqrt(K / 8 + 5)
    first = None
    for flags in (0, TA | TB):
        h.announce("sph_gemm_f32_ex error of sums", shape, "flags", flags, "offset", offset)
        # offset: operands off a 16-byte boundary, the kernels that stage slabs in registers
        stored = [np.concatenate([np.zeros(offset, np.float32),
                                  np.ascontiguousarray(x.T if flags & f else x).ravel()])
                  for x, f in ((A, TA), (B, TB))]
        dA, dB = (capi.DeviceBuffer.from_array(x) for x in stored)
        dC = capi.DeviceBuffer(4 * M * N)
        capi.call("sph_gemm_f32_ex", dC.ptr, dA.ptr + 4 * offset, dB.ptr + 4 * offset, M, N, K, 1,
                  M * N, M * K, K * N, flags | OVERWRITE)
        got = dC.download(np.float32, (M, N))
        for d in (dA, dB, dC):
            d.release()
        error = got - exact
        rows, columns = M - M % 4, N - N % 4
        for part in (np.s_[:rows, :columns], np.s_[rows:, :], np.s_[:, columns:]):
            assert relative(error[part], exact[part]) <= bar, (flags, part)
        first = got if first is None else first
        assert np.array_equal(got.view(np.uint32), first.view(np.uint32)), "depends on the storage"
