"""fp16 products whose sizes are no multiples of 8: the error of their sums.

Bar: the matrix instructions of this kernel family round a sum once per 8 products of k.  Rounding
costs 2.5e-8 of the result's root mean square (at most 2^-24 of it, uniformly distributed, over a
mantissa spread over [1, 2)), and a chain of n additions of equal independent parts rounds partial
sums that grow like 1 .. n, so `chains` chains over K / 8 additions make
sqrt(K / 8 / (2 chains)); adding up the chains and the parts of a last, broken step is another
`chains` + 1 roundings.  15 % are added for the sample.
"""
import numpy as np
import pytest

from sapphire_amd import capi, synth
from tests import helpers as h

pytestmark = pytest.mark.gpu
TA, TB, OVERWRITE = capi.SPH_GEMM_TRANS_A, capi.SPH_GEMM_TRANS_B, capi.SPH_GEMM_OVERWRITE


def check(shape, chains):
    M, N, K = shape
    A = synth.normal(951, (M, K), K ** -0.5).astype(np.float16)
    B = synth.normal(952, (K, N), K ** -0.5).astype(np.float16)
    exact = A.astype(np.float64) @ B.astype(np.float64)
    bar = 1.15 * 2.5e-8 * np.sqrt(K / 16 / chains + chains + 1)
    rows, columns = M - M % 8, N - N % 8
    for flags in (0, TA, TB, TA | TB):
        h.announce("sph_gemm_f16f32 error of sums", shape, "flags", flags)
        stored = [np.ascontiguousarray(x.T if flags & f else x) for x, f in ((A, TA), (B, TB))]
        dA, dB = (capi.DeviceBuffer.from_array(x) for x in stored)
        dC = capi.DeviceBuffer(4 * M * N)
        capi.call("sph_gemm_f16f32", dC.ptr, dA.ptr, dB.ptr, M, N, K, 1, M * N, M * K, K * N,
                  flags | OVERWRITE)
        error = dC.download(np.float32, (M, N)) - exact
        for d in (dA, dB, dC):
            d.release()
        # the last rows and columns, which come from broken chunks of a k-major operand, apart
        parts = [np.s_[:rows, :columns], np.s_[rows:, :], np.s_[:, columns:]]
        for part in parts:
            if error[part].size:
                got = np.sqrt(np.mean(error[part] ** 2) / np.mean(exact[part] ** 2))
                assert got <= bar, (flags, part, got, bar)


@pytest.mark.parametrize("shape", [(402, 502, 702), (401, 501, 1501), (401, 501, 301),
                                   (130, 1000, 1001), (900, 901, 903)])
def test_64_tiles(dev, shape):
    check(shape, 4)


@pytest.mark.parametrize("shape", [(2048, 1533, 1024), (2001, 1507, 999)])
def test_128_tiles_eight_wavefronts(dev, shape):
    check(shape, 4)


@pytest.mark.parametrize("shape", [(2561, 1701, 1001), (2500, 1803, 640)])
def test_128_tiles_four_wavefronts(dev, shape):
    check(shape, 2)
