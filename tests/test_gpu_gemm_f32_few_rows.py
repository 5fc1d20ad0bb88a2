"""fp32 products with few output rows: 4 columns per workgroup, K split over its lanes.

Bars: the same sum in 64 bits -- an output element is a chain of at most 4 ceil(K / 1024) fused
multiply-adds, then 6 additions over the lanes, up to 7 over the wavefronts and the add of the old
value: |gpu - exact| <= (4 ceil(K / 1024) + 15) 2^-24 (|old| + sum_k |a_k b_kj|) to first order;
any way of storing the operands bit for bit the same; nothing written outside out.
"""
import numpy as np
import pytest

from sapphire_amd import capi, synth
from tests import helpers as h

pytestmark = pytest.mark.gpu

TA, TB, OVERWRITE = capi.SPH_GEMM_TRANS_A, capi.SPH_GEMM_TRANS_B, capi.SPH_GEMM_OVERWRITE

# (M, N, K, batch): edges of 4, 8 and 16 rows, of 4 columns, of 4 values of k, of a lane's, a
# wavefront's and a workgroup's share of K and of the two workgroup sizes; one row past the rule;
# one workgroup per compute unit, one more, two, and past that
SHAPES = [(2, 2, 64, 1), (4, 5, 65, 1), (5, 7, 67, 1), (8, 1023, 255, 1), (9, 1025, 257, 1),
          (16, 16, 1023, 1), (16, 17, 1024, 1), (16, 130, 1025, 1), (17, 130, 1025, 1),
          (3, 64, 1026, 1), (13, 33, 2047, 1), (16, 1028, 2048, 1), (16, 1028, 2049, 1),
          (8, 2048, 4099, 1), (8, 2049, 300, 1), (6, 10, 5000, 1), (7, 9, 100, 5), (1, 70, 333, 1)]


def bound(K, old, a, b):
    return (4 * -(-K // 1024) + 15) * 2.0 ** -24 * (np.abs(old) + np.abs(a) @ np.abs(b))


@pytest.mark.parametrize("shape", SHAPES)
def test_few_rows_against_64_bits(dev, shape):
    M, N, K, batch = shape
    A, B = synth.uniform(831, (batch, M, K)), synth.uniform(832, (batch, K, N))
    C = synth.uniform(833, (batch, M, N))
    padded = np.concatenate([np.full(64, 7.0, np.float32), C.ravel(), np.full(64, 7.0, np.float32)])
    a, b = A.astype(np.float64), B.astype(np.float64)
    for overwrite in (0, OVERWRITE):
        old = np.zeros_like(C) if overwrite else C
        first = None
        for flags in (0, TB, TA, TA | TB):
            h.announce("sph_gemm_f32_ex few rows", shape, "flags", flags | overwrite)
            stored_a = np.ascontiguousarray(A.transpose(0, 2, 1)) if flags & TA else A
            stored_b = np.ascontiguousarray(B.transpose(0, 2, 1)) if flags & TB else B
            dC, dA, dB = (capi.DeviceBuffer.from_array(x) for x in (padded, stored_a, stored_b))
            capi.call("sph_gemm_f32_ex", dC.ptr + 4 * 64, dA.ptr, dB.ptr, M, N, K, batch, M * N,
                      M * K, K * N, flags | overwrite)
            out = dC.download(np.float32, padded.shape)
            for d in (dC, dA, dB):
                d.release()
            assert np.all(out[:64] == 7.0) and np.all(out[-64:] == 7.0), "write outside out"
            got = out[64:-64].reshape(C.shape)
            assert np.all(np.abs(got - (old + a @ b)) <= bound(K, old, a, b)), flags
            if M > 1:  # (one row of a B stored K x N has a kernel of its own)
                first = got if first is None else first
                assert np.array_equal(got.view(np.uint32), first.view(np.uint32)), flags


@pytest.mark.parametrize("relu", [0, capi.SPH_LINEAR_RELU])
@pytest.mark.parametrize("shape", [(8, 1023, 784), (3, 10, 1100)])
def test_few_rows_bias_and_relu(dev, shape, relu):
    M, N, K = shape
    h.announce("sph_linear_forward_f32 few rows", shape, "flags", relu)
    x, W, bias = synth.uniform(841, (M, K)), synth.uniform(842, (K, N)), synth.uniform(843, (N,))
    dy, dx, dW, db = (capi.DeviceBuffer.from_array(v)
                      for v in (np.full((M, N), 5.0, np.float32), x, W, bias))
    capi.call("sph_linear_forward_f32", dy.ptr, dx.ptr, dW.ptr, db.ptr, M, K, N, relu)
    got = dy.download(np.float32, (M, N))
    for d in (dy, dx, dW, db):
        d.release()
    want = bias + x.astype(np.float64) @ W
    if relu:
        want = np.maximum(want, 0)
    assert np.all(np.abs(got - want) <= bound(K, bias, x.astype(np.float64), W))


def test_few_rows_optimizer_step(dev):
    """A weight of 5 rows: scale and rate are powers of two, so the step adds no rounding of its own
    but that of the subtraction."""
    M, N, K, scale, rate = 5, 130, 1030, 0.25, 0.5
    h.announce("sph_gemm_f32_sgd few rows", (M, N, K))
    x, dy, W = synth.uniform(851, (K, M)), synth.uniform(852, (K, N)), synth.uniform(853, (M, N))
    dW, dx, dd = (capi.DeviceBuffer.from_array(v) for v in (W, x, dy))
    capi.call("sph_gemm_f32_sgd", dW.ptr, dx.ptr, dd.ptr, M, N, K, scale, rate, TA)
    got = dW.download(np.float32, (M, N))
    for d in (dW, dx, dd):
        d.release()
    a, b = x.T.astype(np.float64), dy.astype(np.float64)
    assert np.all(np.abs(got - (W - scale * rate * (a @ b))) <= bound(K, W, a, b))
