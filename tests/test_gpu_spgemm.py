"""CSR x CSR -> CSR on the device (C ABI and the C++ layer), bit-exact against the CPU checker."""
import ctypes

import numpy as np
import pytest

from oracle import pyoracle as po
from sapphire_amd import capi, synth
from tests import helpers as h
from tests import host_layer as hl

pytestmark = pytest.mark.gpu


def bits(x):
    return np.ascontiguousarray(x).view(np.uint32)


def sparse_dense(seed, shape, density):
    vals = synth.uniform(seed, shape)
    keep = synth.uniform(seed + 1, shape, 0.0, 1.0) < density
    return np.where(keep, vals, np.float32(0)).astype(np.float32)


def _dev(a, dtype):
    return capi.DeviceBuffer.from_array(a if a.size else np.zeros(1, dtype))


def gpu_spgemm(A, B, M, K, N):
    VA, CA, RA = A
    VB, CB, RB = B
    bufs = [_dev(VA, np.float32), _dev(CA, np.uint32), _dev(RA, np.uint32),
            _dev(VB, np.float32), _dev(CB, np.uint32), _dev(RB, np.uint32)]
    dRow = capi.DeviceBuffer(4 * (M + 1))
    nnz = ctypes.c_uint32(0xDEADBEEF)
    capi.call("sph_spgemm_row_offsets_f32", dRow.ptr, *[b.ptr for b in bufs], M, K, N,
              ctypes.byref(nnz))
    ROW = dRow.download(np.uint32, (M + 1,))
    assert ROW[M] == nnz.value
    guard = 4
    dV = capi.DeviceBuffer.from_array(np.full(nnz.value + guard, -77.0, np.float32))
    dCol = capi.DeviceBuffer.from_array(np.full(nnz.value + guard, 0xABCDEF, np.uint32))
    capi.call("sph_spgemm_fill_f32", dV.ptr, dCol.ptr, dRow.ptr, *[b.ptr for b in bufs], M, K, N)
    V = dV.download(np.float32, (nnz.value + guard,))
    COL = dCol.download(np.uint32, (nnz.value + guard,))
    assert np.all(V[nnz.value:] == -77.0) and np.all(COL[nnz.value:] == 0xABCDEF)
    for d in bufs + [dRow, dV, dCol]:
        d.release()
    return V[:nnz.value], COL[:nnz.value], ROW


def gpu_spgemm_one_call(A, B, M, K, N, capacity):
    """(V, COL, ROW, nnz) through sph_spgemm_f32 with room for `capacity` entries; the words past
    the capacity must come back untouched."""
    VA, CA, RA = A
    VB, CB, RB = B
    bufs = [_dev(VA, np.float32), _dev(CA, np.uint32), _dev(RA, np.uint32),
            _dev(VB, np.float32), _dev(CB, np.uint32), _dev(RB, np.uint32)]
    dRow = capi.DeviceBuffer.from_array(np.full(M + 1, 0xFFFFFFFF, np.uint32))
    guard = 8
    dV = capi.DeviceBuffer.from_array(np.full(capacity + guard, -77.0, np.float32))
    dCol = capi.DeviceBuffer.from_array(np.full(capacity + guard, 0xABCDEF, np.uint32))
    nnz = ctypes.c_uint32(0xDEADBEEF)
    capi.call("sph_spgemm_f32", dV.ptr, dCol.ptr, dRow.ptr, capacity, *[b.ptr for b in bufs],
              M, K, N, ctypes.byref(nnz))
    ROW = dRow.download(np.uint32, (M + 1,))
    V = dV.download(np.float32, (capacity + guard,))
    COL = dCol.download(np.uint32, (capacity + guard,))
    assert np.all(V[capacity:] == -77.0) and np.all(COL[capacity:] == 0xABCDEF)
    for d in bufs + [dRow, dV, dCol]:
        d.release()
    return V[:capacity], COL[:capacity], ROW, nnz.value


def check_one_call(A, B, M, K, N, want):
    """sph_spgemm_f32 against the result of the two calls: with room to spare, exactly enough,
    half of it (then the first half of the entries), and so little that the staging slots of
    the longer rows overflow and those rows are multiplied a second time."""
    wV, wC, wR = want
    total = int(wR[M])
    for capacity in (total + 3, total, total // 2, min(total, M)):
        V, COL, ROW, nnz = gpu_spgemm_one_call(A, B, M, K, N, capacity)
        assert nnz == total and np.array_equal(ROW, wR), capacity
        kept = min(capacity, total)
        assert np.array_equal(COL[:kept], wC[:kept]), capacity
        assert np.array_equal(bits(V[:kept]), bits(wV[:kept])), capacity
        if capacity > total:
            assert np.all(V[total:] == -77.0)


# M, K, N, density of A, density of B: single entries, rows of A and of B longer than 64
# entries, empty operands, a width that needs two strips, widths that are not multiples of 64
CASES = [(1, 1, 1, 1.0, 1.0), (5, 7, 3, 0.5, 0.5), (40, 60, 33, 0.1, 0.2), (64, 300, 200, 0.05, 0.05),
         (30, 200, 70, 1.0, 0.3), (20, 50, 700, 0.3, 0.5), (25, 25, 25, 0.0, 0.5),
         (25, 25, 25, 0.5, 0.0), (300, 400, 9000, 0.02, 0.01), (2000, 2000, 2000, 0.004, 0.004)]


@pytest.mark.parametrize("case", CASES)
def test_product_matches_checker(dev, case):
    M, K, N, da, db = case
    h.announce("sph_spgemm_* M K N dA dB =", case)
    dA = sparse_dense(3000 + M, (M, K), da)
    dB = sparse_dense(4000 + N, (K, N), db)
    A, B = po.csr_from_dense(dA), po.csr_from_dense(dB)
    wV, wC, wR = po.spgemm_csr(A, B, M, K, N)
    V, COL, ROW = gpu_spgemm(A, B, M, K, N)
    assert np.array_equal(ROW, wR)
    assert np.array_equal(COL, wC)
    assert np.array_equal(bits(V), bits(wV))
    check_one_call(A, B, M, K, N, (wV, wC, wR))


def test_cancelling_sums_are_dropped_and_unsorted_b_rows_are_accepted(dev):
    h.announce("sph_spgemm_* cancellation / unsorted rows of B")
    A = (np.array([1, -1, 3], np.float32), np.array([0, 1, 2], np.uint32),
         np.array([0, 2, 3], np.uint32))
    B = (np.array([2, 5, 2, 7, 4], np.float32), np.array([1, 3, 1, 0, 2], np.uint32),
         np.array([0, 2, 4, 5], np.uint32))
    V, COL, ROW = gpu_spgemm(A, B, 2, 3, 4)
    assert ROW.tolist() == [0, 2, 3] and COL.tolist() == [0, 3, 2]
    assert V.tolist() == [-7.0, 5.0, 12.0]


def test_equals_dense_product_of_the_densified_operands(dev):
    """Against the dense path of this library's own checker: densify, dense leaf, back to CSR."""
    M, K, N = 96, 128, 80
    h.announce("sph_spgemm_* against densify + dense leaf", (M, K, N))
    dA = sparse_dense(5000, (M, K), 0.08)
    dB = sparse_dense(5002, (K, N), 0.08)
    dense = po.naive_gemm(np.zeros((M, N), np.float32), dA, dB, M, N, K)
    wV, wC, wR = po.csr_from_dense(dense)
    V, COL, ROW = gpu_spgemm(po.csr_from_dense(dA), po.csr_from_dense(dB), M, K, N)
    assert np.array_equal(ROW, wR) and np.array_equal(COL, wC) and np.array_equal(bits(V), bits(wV))


@pytest.mark.parametrize("case", [(7, 9, 5, 0.5), (130, 90, 300, 0.05)])
def test_host_layer_sparse_sparse_gemm(dev, case):
    M, K, N, density = case
    h.announce("Sparse::Cuda::Gemm (sparse x sparse)", case)
    dA = sparse_dense(6000 + M, (M, K), density)
    dB = sparse_dense(6100 + N, (K, N), density)
    wV, wC, wR = po.spgemm_csr(po.csr_from_dense(dA), po.csr_from_dense(dB), M, K, N)
    V, COL, ROW = hl.sparse_sparse_gemm(dA, dB, capacity=wV.size + 16)
    assert np.array_equal(ROW, wR) and np.array_equal(COL, wC) and np.array_equal(bits(V), bits(wV))


@pytest.mark.parametrize("case", [(7, 9, 5, 0.5, 0.5), (130, 90, 300, 0.05, 0.2),
                                  (40, 33, 64, 0.0, 0.5), (64, 64, 64, 0.3, 0.0)])
def test_load_distribution_records(dev, case):
    """Per entry of A the number of entries in the row of B it selects (the reference's
    LoadDistMatrix), through GetLoadDist / CallLoadDist and every LoadDistMatrix copy overload of
    the C++ layer; the C ABI call with and without the load array."""
    M, K, N, da, db = case
    h.announce("load distribution M K N dA dB =", case)
    dA = sparse_dense(7100 + M, (M, K), da)
    dB = sparse_dense(7200 + N, (K, N), db)
    VA, CA, RA = po.csr_from_dense(dA)
    VB, CB, RB = po.csr_from_dense(dB)
    want = np.diff(RB.astype(np.int64))[CA].astype(np.uint32)
    load, col, row, products = hl.load_dist(dA, dB)
    assert np.array_equal(load, want) and np.array_equal(col, CA) and np.array_equal(row, RA)
    assert products == int(want.sum())
    # the products bound the entries of the product
    assert int(po.spgemm_csr((VA, CA, RA), (VB, CB, RB), M, K, N)[2][M]) <= products
    dCol, dRow = _dev(CA, np.uint32), _dev(RB, np.uint32)
    dLoad = capi.DeviceBuffer.from_array(np.full(max(len(CA), 1), 0xFFFFFFFF, np.uint32))
    total = ctypes.c_uint64(123)
    capi.call("sph_spgemm_load_u32", dLoad.ptr, dCol.ptr, dRow.ptr, len(CA), K, ctypes.byref(total))
    assert total.value == int(want.sum())
    assert np.array_equal(dLoad.download(np.uint32, (max(len(CA), 1),))[:len(CA)], want)
    total = ctypes.c_uint64(123)
    capi.call("sph_spgemm_load_u32", None, dCol.ptr, dRow.ptr, len(CA), K, ctypes.byref(total))
    assert total.value == int(want.sum())
    for d in (dCol, dRow, dLoad):
        d.release()


@pytest.mark.parametrize("block", range(4))
def test_random_shapes_and_densities(dev, block):
    """Widths on both sides of the bit-map word, run and strip boundaries (32, 64, 4096, several
    strips), short and long rows, empty results."""
    rng = np.random.default_rng(4200 + block)
    widths = [1, 7, 31, 32, 33, 63, 64, 65, 100, 127, 128, 129, 500, 2047, 2048, 2049, 4095, 4096,
              4097, 5000, 8191, 8193, 12289]
    for it in range(10):
        M, K = int(rng.integers(1, 300)), int(rng.integers(1, 300))
        N = int(rng.choice(widths))
        da = float(rng.choice([0.01, 0.05, 0.2, 0.6]))
        db = float(rng.choice([0.002, 0.01, 0.05] if N > 3000 else [0.002, 0.01, 0.05, 0.3]))
        h.announce("sph_spgemm_* random M K N dA dB =", (M, K, N, da, db))
        dA = sparse_dense(100000 + 100 * block + it, (M, K), da)
        dB = sparse_dense(200000 + 100 * block + it, (K, N), db)
        A, B = po.csr_from_dense(dA), po.csr_from_dense(dB)
        wV, wC, wR = po.spgemm_csr(A, B, M, K, N)
        V, COL, ROW = gpu_spgemm(A, B, M, K, N)
        assert np.array_equal(ROW, wR) and np.array_equal(COL, wC)
        assert np.array_equal(bits(V), bits(wV))
        check_one_call(A, B, M, K, N, (wV, wC, wR))


def test_wide_product_mixes_sorted_rows_and_strip_rows(dev):
    """More than two strips of columns: rows with few products (at most 64 entries of A, at most
    512 products) are sorted in registers, the others stay with the strips.  The operands mix
    both kinds: rows of A that select rows of B longer than 64 entries, rows of A with more than 64
    entries, rows with more than 512 products, empty rows, and a pair of entries whose
    contributions cancel exactly."""
    M, K, N = 260, 300, 20000
    h.announce("sph_spgemm_* wide product with light and heavy rows", (M, K, N))
    rng = np.random.default_rng(77)
    dB = np.zeros((K, N), np.float32)
    for k in range(K):
        count = 100 if k < 10 else 10
        cols = rng.choice(N, size=count, replace=False)
        dB[k, cols] = synth.uniform(9000 + k, (count,))
    dB[21] = dB[20]  # rows 20 and 21 of B are equal: +1 and -1 times them cancel
    dA = np.zeros((M, K), np.float32)
    for m in range(M):
        kind = m % 5
        if kind == 0:    # one or two long rows of B: light, 100 or 200 products
            ks = rng.choice(10, size=1 + m % 2, replace=False)
        elif kind == 1:  # a handful of short rows of B: light
            ks = 10 + rng.choice(K - 10, size=6, replace=False)
        elif kind == 2:  # more than 64 entries: the strips' row
            ks = rng.choice(K, size=150, replace=False)
        elif kind == 3:  # few entries, 600 products: the strips' row
            ks = rng.choice(10, size=6, replace=False)
        else:            # empty
            ks = np.zeros(0, np.int64)
        dA[m, ks] = synth.uniform(9500 + m, (len(ks),))
    dA[1, :] = 0
    dA[1, 20], dA[1, 21], dA[1, 30] = 1.0, -1.0, 0.5  # cancelling pair plus one survivor
    A, B = po.csr_from_dense(dA), po.csr_from_dense(dB)
    wV, wC, wR = po.spgemm_csr(A, B, M, K, N)
    assert wR[2] - wR[1] == np.count_nonzero(dB[30])  # the cancelled columns are not stored
    V, COL, ROW = gpu_spgemm(A, B, M, K, N)
    assert np.array_equal(ROW, wR) and np.array_equal(COL, wC)
    assert np.array_equal(bits(V), bits(wV))
    check_one_call(A, B, M, K, N, (wV, wC, wR))


@pytest.mark.parametrize("N,capacity_per_row", [(4097, 128), (4097, 129), (8193, 600), ((1 << 23) - 1, 600),
                                                (1 << 23, 600)])
def test_light_rows_at_the_edges_of_their_sort(dev, N, capacity_per_row):
    """Rows of 63 .. 513 products (a lane sorts 1, 2, 4 or 8 of them, more go to the strips), of
    64 and 65 entries of A, with every product in one column, with columns that cancel, with NaN,
    infinities and -0, and rows of B in descending column order; widths on both sides of the rule
    and of the 32-bit sort keys.  One more than the staged rows' workgroups hold rows."""
    h.announce("sph_spgemm_* light rows at the edges", (N, capacity_per_row))
    rng = np.random.default_rng(N)
    counts = [1, 2, 63, 64, 65, 127, 128, 129, 255, 256, 257, 511, 512, 513]
    lists = []  # rows of B: (columns, values)
    for n in counts:  # 0 .. 13: n entries, descending columns
        cols = np.sort(rng.choice(N, size=n, replace=False))[::-1]
        lists.append((cols, rng.uniform(-1, 1, n)))
    lists.append((np.array([N - 1]), np.array([0.5])))                        # 14: last column only
    lists.append((np.array([7, N - 1]), np.array([-0.5, -0.0])))              # 15
    lists.append((np.array([3, 5, 7]), np.array([np.nan, np.inf, -np.inf])))  # 16
    lists.append((np.array([], np.int64), np.array([])))                      # 17: empty
    for k in range(18, 90):
        cols = rng.choice(min(N, 40 + 60 * (k % 3)), size=1 + k % 8, replace=False)
        lists.append((cols, rng.uniform(-1, 1, len(cols))))
    K = len(lists)
    RB = np.concatenate([[0], np.cumsum([len(c) for c, _ in lists])]).astype(np.uint32)
    CB = np.concatenate([c for c, _ in lists]).astype(np.uint32)
    VB = np.concatenate([v for _, v in lists]).astype(np.float32)
    rows = [[i] for i in range(18)]                       # one row of B each
    rows += [[3, 17, 0], [3, 0, 1], [14] * 64, [14] * 65, [14, 14, 15], [15, 16, 15], [16, 5],
             [9, 9], [9, 9, 0], list(range(18, 82)), list(range(18, 83)), []]
    rows += [list(rng.choice(np.arange(18, 90), size=int(rng.integers(1, 64)))) for _ in range(60)]
    values = [rng.uniform(-1, 1, len(r)) for r in rows]
    values[22] = np.array([1.0, -1.0, 0.25])              # the last column cancels
    M = len(rows)
    RA = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.uint32)
    CA = np.concatenate([np.asarray(r, np.int64) for r in rows]).astype(np.uint32)
    VA = np.concatenate(values).astype(np.float32)
    A, B = (VA, CA, RA), (VB, CB, RB)
    wV, wC, wR = po.spgemm_csr(A, B, M, K, N)
    V, COL, ROW = gpu_spgemm(A, B, M, K, N)
    nan = np.isnan(wV)
    assert np.array_equal(ROW, wR) and np.array_equal(COL, wC)
    assert np.array_equal(np.isnan(V), nan) and np.array_equal(bits(V)[~nan], bits(wV)[~nan])
    total = int(wR[M])
    for capacity in (capacity_per_row * M, capacity_per_row * M + M - 1, total // 2, M):
        V, COL, ROW, nnz = gpu_spgemm_one_call(A, B, M, K, N, capacity)
        kept = min(capacity, total)
        assert nnz == total and np.array_equal(ROW, wR)
        assert np.array_equal(COL[:kept], wC[:kept])
        assert np.array_equal(np.isnan(V[:kept]), nan[:kept])
        assert np.array_equal(bits(V[:kept])[~nan[:kept]], bits(wV[:kept])[~nan[:kept]])


@pytest.mark.parametrize("M", [15, 16, 17, 8191, 8193, 131072, 131073])
def test_staged_rows_find_their_place(dev, M):
    """The offsets that every workgroup of the move adds up by itself: fewer rows than it has
    wavefronts, one more than whole groups of rows, the last number of rows and the first that is
    scanned by launches of its own; a row now and then overflows its slot."""
    h.announce("sph_spgemm_f32 rows", M)
    K = N = 300
    rng = np.random.default_rng(M)
    per = rng.integers(0, 4, M)
    RA = np.concatenate([[0], np.cumsum(per)]).astype(np.uint32)
    CA = rng.integers(0, K, int(RA[M])).astype(np.uint32)
    VA = rng.uniform(-1, 1, len(CA)).astype(np.float32)
    lengths = np.where(np.arange(K) == 5, 280, rng.integers(0, 3, K))
    RB = np.concatenate([[0], np.cumsum(lengths)]).astype(np.uint32)
    CB = np.concatenate([rng.choice(N, size=n, replace=False) for n in lengths]).astype(np.uint32)
    VB = rng.uniform(-1, 1, len(CB)).astype(np.float32)
    A, B = (VA, CA, RA), (VB, CB, RB)
    wV, wC, wR = po.spgemm_csr(A, B, M, K, N)
    total = int(wR[M])
    V, COL, ROW, nnz = gpu_spgemm_one_call(A, B, M, K, N, total + M)
    assert nnz == total and np.array_equal(ROW, wR) and np.array_equal(COL[:total], wC)
    assert np.array_equal(bits(V[:total]), bits(wV))


@pytest.mark.parametrize("N", [1, 300, 4097, 8192, 8193, 70000])
def test_no_rows(dev, N):
    """M = 0 through every entry point, on both sides of the widths that take other kernels:
    ROWC[0] and the count are 0, nothing behind ROWC, VC or COLC is touched."""
    h.announce("sph_spgemm_* without rows, N =", N)
    K = 3
    VB = np.array([0.5, -1.0, 2.0], np.float32)
    CB = np.array([0, N - 1, 0], np.uint32)
    RB = np.array([0, 1, 2, 3], np.uint32)
    bufs = [_dev(np.zeros(0, np.float32), np.float32), _dev(np.zeros(0, np.uint32), np.uint32),
            _dev(np.zeros(1, np.uint32), np.uint32), _dev(VB, np.float32), _dev(CB, np.uint32),
            _dev(RB, np.uint32)]
    operands = [b.ptr for b in bufs]
    guard = np.full(1025, 0xFFFFFFFF, np.uint32)
    dV, dCol = (capi.DeviceBuffer.from_array(guard) for _ in range(2))
    for entry, head in (("sph_spgemm_row_offsets_f32", []),
                        ("sph_spgemm_f32", [dV.ptr, dCol.ptr]),):
        for capacity in (0, 1000):
            dRow = capi.DeviceBuffer.from_array(guard)
            nnz = ctypes.c_uint32(0xDEADBEEF)
            tail = [capacity] if head else []
            capi.call(entry, *head, dRow.ptr, *tail, *operands, 0, K, N, ctypes.byref(nnz))
            ROW = dRow.download(np.uint32, guard.shape)
            assert nnz.value == 0 and ROW[0] == 0 and np.all(ROW[1:] == 0xFFFFFFFF), entry
            dRow.release()
    dRow = capi.DeviceBuffer.from_array(np.zeros(1, np.uint32))
    capi.call("sph_spgemm_fill_f32", dV.ptr, dCol.ptr, dRow.ptr, *operands, 0, K, N)
    for d in (dV, dCol):
        assert np.all(d.download(np.uint32, guard.shape) == 0xFFFFFFFF)
    for d in bufs + [dRow, dV, dCol]:
        d.release()


@pytest.mark.parametrize("N", [300, 9000])
@pytest.mark.parametrize("M", [1, 5, 2047, 7001, 14000, 40001, 300001])
def test_rows_that_a_pass_looks_for(dev, M, N):
    """Passes that take only some rows (those left to the strips in a wide product, those that
    overflowed their staging slot) with 1, 3, 6 and 8 rows per turn and more turns than one look
    of all wavefronts covers: scattered ones, a run of neighbours, the first and the last row;
    some of each kind overflow a slot of 67 entries."""
    h.announce("sph_spgemm_* rows looked for, M N", (M, N))
    K = 200
    rng = np.random.default_rng(M + N)
    lengths = np.where(np.arange(K) < 4, 90, rng.integers(0, 3, K))
    RB = np.concatenate([[0], np.cumsum(lengths)]).astype(np.uint32)
    CB = np.concatenate([rng.choice(N, size=n, replace=False) for n in lengths]).astype(np.uint32)
    VB = rng.uniform(-1, 1, len(CB)).astype(np.float32)
    kind = np.zeros(M, np.int64)                   # 0: one short row of B
    kind[rng.integers(0, M, M // 97 + 1)] = 1      # 1: 70 entries of A
    kind[rng.integers(0, M, M // 89 + 1)] = 2      # 2: two long rows of B, 180 products
    kind[M // 2:M // 2 + 20] = 1
    kind[[0, M - 1]] = 1, 2
    per = np.array([1, 70, 2])[kind]
    RA = np.concatenate([[0], np.cumsum(per)]).astype(np.uint32)
    CA = rng.integers(4, K, int(RA[M]))
    for row in np.nonzero(kind)[0]:
        low, high = (4, K) if kind[row] == 1 else (0, 4)
        CA[RA[row]:RA[row + 1]] = low + rng.choice(high - low, size=per[row], replace=False)
    CA = CA.astype(np.uint32)
    VA = rng.uniform(-1, 1, len(CA)).astype(np.float32)
    A, B = (VA, CA, RA), (VB, CB, RB)
    wV, wC, wR = po.spgemm_csr(A, B, M, K, N)
    V, COL, ROW = gpu_spgemm(A, B, M, K, N)
    assert np.array_equal(ROW, wR) and np.array_equal(COL, wC) and np.array_equal(bits(V), bits(wV))
    total = int(wR[M])
    for capacity in (M, total + 5):
        V, COL, ROW, nnz = gpu_spgemm_one_call(A, B, M, K, N, capacity)
        kept = min(capacity, total)
        assert nnz == total and np.array_equal(ROW, wR), capacity
        assert np.array_equal(COL[:kept], wC[:kept]), capacity
        assert np.array_equal(bits(V[:kept]), bits(wV[:kept])), capacity
