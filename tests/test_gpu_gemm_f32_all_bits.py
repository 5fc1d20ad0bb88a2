"""fp32 products use every bit of every operand, and an element of the result depends on its own row
and column alone, at sizes from one round of 64 x 64 tiles to several of 128 x 128.

Bars.  A sum with one product in it that is not zero is that product rounded once, whatever the order of
the sum: at most 2^-24 of it away, and the product itself where it has at most 24 bits (a one or a zero
times a value, integers below 2^12).
"""
import numpy as np
import pytest

from sapphire_amd import capi, synth
from tests import helpers as h

pytestmark = pytest.mark.gpu
TA, TB, OW = capi.SPH_GEMM_TRANS_A, capi.SPH_GEMM_TRANS_B, capi.SPH_GEMM_OVERWRITE

# (M, N, K): one round of 64 x 64 tiles, with edges and without; two rounds; many tiles, a short K
SHAPES = [(1024, 1024, 1024), (1021, 1023, 1025), (1501, 1203, 1001), (2048, 2048, 352),
          (2046, 2045, 333)]
STORAGE = [0, TA, TB, TA | TB]


def bits(x):
    return np.ascontiguousarray(x).view(np.uint32)


def run(A, B, flags, C=None, offset=0):
    """A (M x K) times B (K x N), stored as the flags say, `offset` floats into their memory."""
    (M, K), N = A.shape, B.shape[1]
    pad = np.zeros(offset, np.float32)
    dA, dB = (capi.DeviceBuffer.from_array(np.concatenate(
        [pad, np.ascontiguousarray(x.T if flags & f else x).ravel()])) for x, f in ((A, TA), (B, TB)))
    start = np.full((M, N), np.nan, np.float32) if C is None else C
    dC = capi.DeviceBuffer.from_array(start)
    capi.call("sph_gemm_f32_ex", dC.ptr, dA.at(4 * offset), dB.at(4 * offset), M, N, K, 1, M * N, M * K,
              K * N, flags | (OW if C is None else 0))
    out = dC.download(np.float32, (M, N))
    for d in (dA, dB, dC):
        d.release()
    return out


def full(seed, shape, low=-3, high=0):
    """All 24 bits of the mantissa, signs, exponents spread evenly over low .. high."""
    rng = np.random.default_rng(seed)
    mantissa = rng.integers(2 ** 23, 2 ** 24, shape).astype(np.float64) * rng.choice([-1.0, 1.0], shape)
    return np.ldexp(mantissa, rng.integers(low - 23, high - 22, shape)).astype(np.float32)


def one_per_row(seed, rows, columns, values):
    """(matrix, columns): values[i] somewhere in row i, zeros elsewhere."""
    at = np.random.default_rng(seed).integers(0, columns, rows)
    x = np.zeros((rows, columns), np.float32)
    x[np.arange(rows), at] = values
    return x, at


def products(side, shape, ones, values):
    """(A, B, exact): one product per element, `ones` in the rows of A (side 0) or the columns of B."""
    M, N, K = shape
    if side == 0:
        A, at = one_per_row(971, M, K, ones(M))
        B = values((K, N))
        return A, B, A[np.arange(M), at].astype(np.float64)[:, None] * B[at]
    Bt, at = one_per_row(972, N, K, ones(N))
    A = values((M, K))
    return A, Bt.T, A[:, at] * Bt[np.arange(N), at].astype(np.float64)


@pytest.mark.parametrize("side", [0, 1], ids=["rows of A", "columns of B"])
@pytest.mark.parametrize("shape", SHAPES)
def test_gather(dev, shape, side):
    """A one per row (or column) picks rows (columns) of the other operand, bit for bit."""
    A, B, exact = products(side, shape, lambda n: np.ones(n, np.float32),
                           lambda s: full(973, s))
    C = full(974, exact.shape)
    for flags in STORAGE:
        for offset in (0, 1):
            h.announce("sph_gemm_f32_ex gather", shape, "side", side, "flags", flags, "offset", offset)
            assert np.array_equal(bits(run(A, B, flags, offset=offset)), bits(exact.astype(np.float32)))
    assert np.array_equal(bits(run(A, B, 0, C)), bits(C + exact.astype(np.float32)))


@pytest.mark.parametrize("side", [0, 1], ids=["rows of A", "columns of B"])
@pytest.mark.parametrize("spread", [0, 2, 15])
@pytest.mark.parametrize("shape", SHAPES)
def test_one_product(dev, shape, spread, side):
    """Full mantissas on both sides, over 1 to 31 binades."""
    def values(s):
        return full(977 + np.size(s), s, -spread, spread)
    A, B, exact = products(side, shape, values, values)
    for flags in (0, TA | TB):
        h.announce("sph_gemm_f32_ex one product", shape, "spread", spread, "side", side, "flags", flags)
        error = np.abs(run(A, B, flags) - exact)
        assert np.all(error <= 2.0 ** -24 * np.abs(exact)), \
            float(np.max(error / np.maximum(np.abs(exact), 1e-30)))


@pytest.mark.parametrize("shape", SHAPES)
def test_integers(dev, shape):
    """Integers of 12 bits each, one product per sum, and a few of 22 bits times ones and minus ones,
    whose sums stay below 2^24."""
    M, N, K = shape
    rng = np.random.default_rng(981)
    A, B, exact = products(0, shape, lambda n: rng.integers(-4095, 4096, n).astype(np.float32),
                           lambda s: rng.integers(-4095, 4096, s).astype(np.float32))
    S = np.zeros((M, K), np.float32)
    for _ in range(4):
        S[np.arange(M), rng.integers(0, K, M)] = rng.choice([-1.0, 1.0], M)
    V = rng.integers(-2 ** 22 + 1, 2 ** 22, (K, N)).astype(np.float32)
    for flags in (0, TA | TB):
        h.announce("sph_gemm_f32_ex integers", shape, "flags", flags)
        assert np.array_equal(run(A, B, flags), exact)
        assert np.array_equal(run(S, V, flags), S.astype(np.float64) @ V.astype(np.float64))


@pytest.mark.parametrize("value", [2.0 ** 60, 2.0 ** -60, np.inf, np.nan])
@pytest.mark.parametrize("shape", SHAPES[:1] + SHAPES[-1:])
def test_rows_and_columns_of_their_own(dev, shape, value):
    """What one row of A, or one column of B, holds changes no bit of the others."""
    M, N, K = shape
    A, B = synth.uniform(991, (M, K)), synth.uniform(992, (K, N))
    h.announce("sph_gemm_f32_ex one row differs", shape, value)
    want = bits(run(A, B, 0))
    A[37, 5::9] = value
    B[3::7, N - 30] = value
    got = bits(run(A, B, 0))
    rows, columns = np.arange(M) != 37, np.arange(N) != N - 30
    assert np.array_equal(got[rows][:, columns], want[rows][:, columns])
