"""fp32 products of one round of 64 x 64 tiles and more, by the values of their operands: exponents that
differ by row, by column, along K and everywhere, subnormal values, zeros, integers, infinities and NaN.

Bars, against 64 bits.  Of every element: |gpu - exact| / sum_k |a_ik b_kj| <= (K + 5) 2^-24, since a
term takes part in at most K + 3 roundings of partial sums that sum bounds, and the old value and the
product in one each.  Of a whole result of U(-1, 1) operands: a rounding costs 2^-24 at most, 2.5e-8 in the root
mean square (uniformly distributed over a mantissa that is itself spread over [1, 2)); a chain of K additions
rounds partial sums of variance v, 2 v, ..., K v, which makes 2.5e-8 sqrt(K / 2) of the result, and 5 K v are
left to the old value and the parts of a sum; 12 % are added for the sample.
"""
import numpy as np
import pytest

from oracle import pyoracle as po
from sapphire_amd import capi, synth
from tests import helpers as h

pytestmark = pytest.mark.gpu
TA, TB, OW = capi.SPH_GEMM_TRANS_A, capi.SPH_GEMM_TRANS_B, capi.SPH_GEMM_OVERWRITE

# (batch, M, N, K): many tiles, whole ones and edges that cut four columns, K of whole steps, of partial ones
# and within 4 values; a batch.  Then one round of 64 x 64 tiles, and two
SHAPES = [(1, 2048, 2048, 352), (1, 2046, 2045, 333), (1, 1921, 2047, 350), (16, 509, 511, 322),
          (1, 2048, 2047, 320), (1, 1024, 1024, 1024), (1, 1024, 1018, 992), (1, 1022, 961, 1007),
          (1, 1021, 1023, 1025), (3, 510, 509, 1050), (1, 1280, 1270, 1300)]
M, N, K = 2046, 2045, 333


@pytest.fixture(params=[(2046, 2045, 333), (1022, 1021, 1003)], ids=["many tiles", "one round"])
def sizes(request, monkeypatch):
    for name, value in zip("MNK", request.param):
        monkeypatch.setitem(globals(), name, value)


def bits(x):
    return np.ascontiguousarray(x).view(np.uint32)


def run(C, A, B, flags, offset=0):
    """A, B as they are multiplied; stored as the flags say, `offset` floats into their memory."""
    batch, m, k = A.shape
    n = B.shape[2]
    pad = np.zeros(offset, np.float32)
    dA, dB = (capi.DeviceBuffer.from_array(
        np.concatenate([pad, (x.swapaxes(1, 2) if flags & f else x).ravel()]))
        for x, f in ((A, TA), (B, TB)))
    guard = np.full(64, 7.0, np.float32)
    dC = capi.DeviceBuffer.from_array(np.concatenate([guard, C.ravel(), guard]))
    capi.call("sph_gemm_f32_ex", dC.at(256), dA.at(4 * offset), dB.at(4 * offset), m, n, k, batch,
              m * n, m * k, k * n, flags)
    out = dC.download(np.float32, (C.size + 128,))
    for d in (dA, dB, dC):
        d.release()
    assert np.all(out[:64] == 7.0) and np.all(out[-64:] == 7.0), "write outside out"
    return out[64:-64].reshape(C.shape)


def check(got, A, B, C=0.0):
    exact = A.astype(np.float64) @ B.astype(np.float64) + C
    size = np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64) + np.abs(C)
    bar = (A.shape[-1] + 5) * 2.0 ** -24
    error = np.abs(got - exact)
    assert np.all(error <= bar * size + 2.0 ** -149), float(np.max(error / np.maximum(size, 1e-300)))
    return float(np.sqrt(np.mean(error ** 2) / np.mean(exact ** 2)))


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("shape", SHAPES)
def test_storage_changes_no_bit(dev, shape, offset):
    batch, m, n, k = shape
    A, B = synth.uniform(901, (batch, m, k)), synth.uniform(902, (batch, k, n))
    C = synth.uniform(903, (batch, m, n))
    first = None
    for flags in (0, TA, TB, TA | TB):
        h.announce("sph_gemm_f32_ex", shape, "flags", flags, "offset", offset)
        got = run(C, A, B, flags, offset)
        if first is None:
            first = got
            relative = check(got, A, B, C)
            assert relative <= 1.12 * 2.5e-8 * np.sqrt(k / 2 + 5), relative
            assert np.array_equal(bits(run(np.full_like(C, np.nan), A, B, OW)),
                                  bits(run(np.zeros_like(C), A, B, 0)))
        assert np.array_equal(bits(got), bits(first)), flags


@pytest.mark.parametrize("shape", [(1921, 2047, 350), (2046, 1923, 333), (2042, 1954, 321), (961, 1023, 1001),
                                   (1022, 963, 1030)])
def test_large_neighbours_of_the_last_rows(dev, shape):
    """Rows and columns past a multiple of 32 next to others that are 2^20 larger."""
    m, n, k = shape
    A, B = synth.uniform(904, (1, m, k)), synth.uniform(905, (1, k, n))
    A[:, m // 32 * 32 - 4:m // 32 * 32] *= 2.0 ** 20
    B[:, :, n // 32 * 32 - 4:n // 32 * 32] *= 2.0 ** 20
    A[:, -1, ::3] *= 2.0 ** -12
    B[:, ::5, -1] *= 2.0 ** -12
    C = np.zeros((1, m, n), np.float32)
    first = None
    for flags in (0, TA, TB, TA | TB):
        h.announce("sph_gemm_f32_ex large neighbours", shape, "flags", flags)
        got = run(C, A, B, flags)
        if first is None:
            first = got
            check(got, A, B)
        assert np.array_equal(bits(got), bits(first)), flags


def spread(seed, shape, low, high):
    """Signs and mantissas of U(-1, 1), exponents spread evenly over low .. high."""
    e = np.random.default_rng(seed).integers(low, high + 1, shape)
    return np.ldexp(synth.uniform(seed, shape), e).astype(np.float32)


def rows_and_columns(low, high):
    """Every row of A and column of B with an exponent of its own."""
    rng = np.random.default_rng(911)
    return (np.ldexp(synth.uniform(912, (1, M, K)), rng.integers(low, high, (1, M, 1))),
            np.ldexp(synth.uniform(913, (1, K, N)), rng.integers(low, high, (1, 1, N))))


def balanced():
    """Column k of A large where row k of B is small: all products matter alike."""
    e = np.random.default_rng(914).integers(-30, 31, K)
    return (np.ldexp(synth.uniform(915, (1, M, K)), e[None, None, :]),
            np.ldexp(synth.uniform(916, (1, K, N)), -e[None, :, None]))


def growing():
    """Nothing for 40 values of k, then larger and larger values."""
    e = np.maximum(np.arange(K) - 40, 0) // 12
    A = np.ldexp(synth.uniform(917, (1, M, K)), e[None, None, :])
    A[:, :, :40] = 0
    return A, np.ldexp(synth.uniform(918, (1, K, N)), -e[None, :, None])


def a_few_small():
    """Rows and columns that hold nothing but one small value, next to ordinary ones."""
    A, B = synth.uniform(919, (1, M, K)), synth.uniform(920, (1, K, N))
    for i, (row, k) in enumerate([(5, 7), (6, 7), (130, 332), (M - 1, 331), (M - 2, 0), (64, 31)]):
        A[0, row] = 0
        A[0, row, k] = 2.0 ** -(30 + 3 * i) * 1.1
    for i, (col, k) in enumerate([(3, 7), (4, 7), (131, 332), (N - 1, 330), (N - 2, 1)]):
        B[0, :, col] = 0
        B[0, k, col] = -(2.0 ** -(31 + 3 * i)) * 1.3
    return A, B


def small_and_large(low, high):
    return spread(921, (1, M, K), low, high), spread(922, (1, K, N), low, high)


RANGES = {"rows and columns": lambda: rows_and_columns(-12, 13),
          "rows and columns, far apart": lambda: rows_and_columns(-40, 41),
          "balanced": balanced, "growing": growing, "a few small": a_few_small,
          "13 binades": lambda: small_and_large(-6, 6), "60 binades": lambda: small_and_large(-30, 30),
          "large": lambda: small_and_large(50, 58), "tiny": lambda: small_and_large(-70, -55),
          "subnormal": lambda: (spread(923, (1, M, K), -140, -130), spread(924, (1, K, N), 100, 110))}


@pytest.mark.parametrize("flags", [0, TA | TB])
@pytest.mark.parametrize("name", RANGES)
def test_ranges(dev, sizes, name, flags):
    h.announce("sph_gemm_f32_ex", name, (M, N, K), "flags", flags)
    A, B = (x.astype(np.float32) for x in RANGES[name]())
    check(run(np.zeros((1, M, N), np.float32), A, B, flags), A, B)


def test_zeros_and_ones(dev, sizes):
    """Small integers, and whole rows, columns and chunks of zeros: exact."""
    h.announce("sph_gemm_f32_ex integers")
    A, B = synth.small_integers(931, (1, M, K), span=9), synth.small_integers(932, (1, K, N), span=9)
    A[0, 64:160] = 0
    A[0, :, 32:96] = 0
    B[0, :, 700:900] = 0
    C = synth.small_integers(933, (1, M, N), span=100)
    want = (C + A.astype(np.float64) @ B.astype(np.float64)).astype(np.float32)
    assert np.array_equal(run(C, A, B, 0), want)
    assert np.array_equal(run(C, A, B, TA | TB), want)


@pytest.mark.parametrize("values", [(np.inf,), (-np.inf, np.nan), (3e38, -3e38), (np.nan,)])
def test_specials(dev, sizes, values):
    """Infinities, NaN and sums past the largest number, as the CPU loop has them."""
    h.announce("sph_gemm_f32_ex specials", values, (M, N, K))
    A, B = synth.uniform(941, (M, K)), synth.uniform(942, (K, N))
    for i, v in enumerate(values * 3):
        A[3 + 50 * i, 5 * i] = v
        B[332 - 7 * i, 9 + 40 * i] = v
    B[0] = 0.0
    B[0, 1] = 2.0
    with np.errstate(all="ignore"):
        ref = po.gemm_rows(np.zeros((320, N), np.float32), A[:320], B, 320, N, K, threads=8)
    got = run(np.zeros((1, M, N), np.float32), A[None], B[None], 0)[0][:320]
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    inf = np.isinf(ref)
    assert np.array_equal(got[inf], ref[inf]) and np.array_equal(np.isinf(got), inf)
    ok = np.isfinite(ref)
    scale = np.abs(np.where(np.isfinite(A[:320]), A[:320], 0)).astype(np.float64) @ \
        np.abs(np.where(np.isfinite(B), B, 0)).astype(np.float64)
    assert np.all(np.abs(got[ok].astype(np.float64) - ref[ok]) <= 1e-4 * scale[ok])


def test_linear_and_sgd_epilogues(dev, sizes):
    """Bias, ReLU and the optimizer's step after the same sums."""
    h.announce("sph_linear_forward_f32 and sph_gemm_f32_sgd", (M, N, K))
    x, W = synth.uniform(951, (M, K)), synth.uniform(952, (K, N))
    bias, old = synth.uniform(953, (N,)), synth.uniform(954, (M, N))
    dx, dW, db = (capi.DeviceBuffer.from_array(v) for v in (x, W, bias))
    dy, dz = capi.DeviceBuffer(4 * M * N), capi.DeviceBuffer.from_array(old)
    capi.call("sph_linear_forward_f32", dy.ptr, dx.ptr, dW.ptr, db.ptr, M, K, N,
              capi.SPH_LINEAR_RELU)
    capi.call("sph_gemm_f32_sgd", dz.ptr, dx.ptr, dW.ptr, M, N, K, 0.5, 0.25, 0)
    y, z = (d.download(np.float32, (M, N)) for d in (dy, dz))
    for d in (dx, dW, db, dy, dz):
        d.release()
    sums = run(np.zeros((1, M, N), np.float32), x[None], W[None], 0)[0]
    assert np.array_equal(bits(y), bits(np.maximum(np.float32(0) + bias + sums, np.float32(0))))
    assert np.array_equal(bits(z), bits(old - (sums * np.float32(0.5)) * np.float32(0.25)))
