"""The few-row kernel where its wavefronts are split another way: K of one wavefront, of two, of four
and of eight, one group of rows and several.  Bars as for the other few-row products."""
import pytest

from tests.test_gpu_gemm_f32_few_rows import test_few_rows_against_64_bits as against_64_bits

pytestmark = pytest.mark.gpu

# (M, N, K, batch)
SHAPES = [(4, 9, 256, 1), (5, 10, 256, 1), (8, 33, 257, 1), (7, 1027, 255, 1), (8, 130, 512, 1),
          (6, 130, 513, 1), (9, 12, 256, 1), (16, 1026, 254, 1), (13, 14, 257, 1), (12, 33, 511, 2),
          (16, 130, 512, 1), (9, 130, 513, 1), (11, 70, 1023, 3), (15, 18, 1027, 1)]


@pytest.mark.parametrize("shape", SHAPES)
def test_splits_against_64_bits(dev, shape):
    against_64_bits(dev, shape)
