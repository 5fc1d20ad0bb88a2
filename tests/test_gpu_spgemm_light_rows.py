"""CSR x CSR, rows that are sorted in registers: which entry of A a product belongs to, and the line
between them and the strips on a product of two strips' width.  Bar: the CPU checker, bit for bit."""
import numpy as np
import pytest

from oracle import pyoracle as po
from sapphire_amd import synth
from tests import helpers as h
from tests.test_gpu_spgemm import bits, gpu_spgemm, gpu_spgemm_one_call

pytestmark = pytest.mark.gpu


def csr(lists):
    offsets = np.concatenate([[0], np.cumsum([len(c) for c in lists])]).astype(np.uint32)
    cols = np.concatenate([np.asarray(c, np.int64) for c in lists]).astype(np.uint32)
    return synth.uniform(int(offsets[-1]), (len(cols),)), cols, offsets


# columns; capacity per row on both sides of the line for two strips, and past them (any capacity);
# 2^23 columns take keys of 64 bits
@pytest.mark.parametrize("N,capacity_per_row", [(4097, 320), (4097, 321), (8192, 320), (8192, 321),
                                                (8193, 100), (1 << 23, 100)])
def test_products_find_their_entry_of_a(dev, N, capacity_per_row):
    h.announce("sph_spgemm_* products and their entries of A", (N, capacity_per_row))
    rng = np.random.default_rng(N + capacity_per_row)
    # row k of B has k entries up to 70, then empty rows, then single entries in one column
    b_rows = [rng.choice(N, size=k, replace=False) for k in range(71)]
    b_rows += [[] for _ in range(4)] + [[N - 1]] * 4
    empty, single = list(range(71, 75)), list(range(75, 79))
    a_rows = [
        empty, [0] + empty + [1], [64], [65], [63, 1], [64, 1], [32] * 4, [32] * 4 + [1],
        [64] * 4, [64] * 4 + [1], [64] * 8, [64] * 8 + [1],
        ([0, 1] * 32), ([1, 0] * 32), (empty * 16), (empty * 15 + [5, 6, 7, 8]),
        ([9, 8] + empty * 15), [70] * 7 + [0] * 57, single * 16, empty + single + empty, []]
    a_rows += [list(rng.choice(79, size=int(n))) for n in rng.integers(1, 65, 40)]
    A, B = csr(a_rows), csr(b_rows)
    M, K = len(a_rows), len(b_rows)
    wV, wC, wR = po.spgemm_csr(A, B, M, K, N)
    V, COL, ROW = gpu_spgemm(A, B, M, K, N)
    assert np.array_equal(ROW, wR) and np.array_equal(COL, wC)
    assert np.array_equal(bits(V), bits(wV))
    total = int(wR[M])
    for capacity in (capacity_per_row * M, total // 2, M):
        V, COL, ROW, nnz = gpu_spgemm_one_call(A, B, M, K, N, capacity)
        kept = min(capacity, total)
        assert nnz == total and np.array_equal(ROW, wR)
        assert np.array_equal(COL[:kept], wC[:kept])
        assert np.array_equal(bits(V[:kept]), bits(wV[:kept]))
