"""fp32 products with few output columns: the few-row kernel with operands, rows and columns
changed over.  Bars and checks are those of the few rows (same chains of sums)."""
import numpy as np
import pytest

from sapphire_amd import synth
from tests import helpers as h
from tests import test_gpu_gemm_f32_few_rows as rows

pytestmark = pytest.mark.gpu

# edges of 4 and 8 columns, of 4 rows, of a lane's and a workgroup's share of K and of the two
# workgroup sizes, one column and one value of k past the rule, one and two workgroups per compute
# unit and past that, a batch
SHAPES = [(5, 2, 1024, 1), (5, 4, 1025, 1), (70, 1, 1333, 1), (7, 5, 1027, 1), (1023, 8, 1024, 1),
          (1025, 8, 1030, 1), (17, 9, 1024, 1), (130, 8, 1023, 1), (64, 3, 1026, 1),
          (33, 7, 2047, 1), (1028, 6, 2048, 1), (1028, 8, 2049, 1), (2048, 8, 4099, 1),
          (2049, 8, 1024, 1), (10, 6, 5000, 1), (9, 7, 1100, 5)]


@pytest.mark.parametrize("shape", SHAPES)
def test_few_columns_against_64_bits(dev, shape):
    rows.test_few_rows_against_64_bits(dev, shape)


@pytest.mark.parametrize("relu", [0, rows.capi.SPH_LINEAR_RELU])
@pytest.mark.parametrize("shape", [(1023, 8, 1024), (200, 3, 1100)])
def test_few_columns_bias_and_relu(dev, shape, relu):
    rows.test_few_rows_bias_and_relu(dev, shape, relu)


def test_few_columns_grouped(dev):
    """Units at different places of A, B and out (integers: every sum is exact)."""
    M, N, K = 70, 3, 1030
    A, B, C = (synth.small_integers(s, (2, x)) for s, x in ((861, M * K), (862, K * N), (863, M * N)))
    triples = [(0, M * K, K * N), (M * N, 0, K * N)]
    h.announce("sph_gemm_f32_grouped few columns", (M, N, K))
    got = h.gpu_gemm_grouped(C, A, B, M, N, K, triples).reshape(2, M, N)
    b = B[1].reshape(K, N)
    assert np.array_equal(got[0], C[0].reshape(M, N) + A[1].reshape(M, K) @ b)
    assert np.array_equal(got[1], C[1].reshape(M, N) + A[0].reshape(M, K) @ b)


@pytest.mark.parametrize("flags", [0, rows.TA, rows.TB, rows.TA | rows.TB])
@pytest.mark.parametrize("shape", [(1023, 7, 1030), (70, 3, 1024), (130, 8, 2049)])
def test_few_columns_optimizer_step(dev, shape, flags):
    """A weight of few outputs: scale and rate are powers of two, so the step adds no rounding of its
    own but that of the subtraction."""
    M, N, K = shape
    scale, rate = 0.25, 0.5
    h.announce("sph_gemm_f32_sgd few columns", shape, "flags", flags)
    A, B, W = synth.uniform(871, (M, K)), synth.uniform(872, (K, N)), synth.uniform(873, (M, N))
    stored = [np.ascontiguousarray(x.T) if flags & f else x
              for x, f in ((A, rows.TA), (B, rows.TB))]
    dW, dA, dB = (rows.capi.DeviceBuffer.from_array(v) for v in (W, *stored))
    rows.capi.call("sph_gemm_f32_sgd", dW.ptr, dA.ptr, dB.ptr, M, N, K, scale, rate, flags)
    got = dW.download(np.float32, (M, N))
    for d in (dW, dA, dB):
        d.release()
    a, b = A.astype(np.float64), B.astype(np.float64)
    assert np.all(np.abs(got - (W - scale * rate * (a @ b))) <= rows.bound(K, W, a, b))


@pytest.mark.parametrize("shared", ["A", "B"])
def test_few_columns_shared_operand(dev, shared):
    """One operand for all units of a batch: its stride is 0 (integers: every sum is exact)."""
    M, N, K, batch = 66, 5, 1029, 3
    h.announce("sph_gemm_f32_ex few columns, shared", shared)
    A = synth.small_integers(881, (1 if shared == "A" else batch, M, K), span=4)
    B = synth.small_integers(882, (1 if shared == "B" else batch, K, N), span=4)
    C = synth.small_integers(883, (batch, M, N), span=100)
    got = h.gpu_gemm_f32_ex(C, A, B, M, N, K, 0, batch=batch,
                            stride_a=0 if shared == "A" else None,
                            stride_b=0 if shared == "B" else None)
    assert np.array_equal(got, C + A @ B)
