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
