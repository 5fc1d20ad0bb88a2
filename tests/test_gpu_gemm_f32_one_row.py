"""fp32 products with one output row (column sums, M = 1): 16 columns per workgroup from K = 321 on up
to half as many workgroups as compute units (2048 columns in all on this chip), 64 otherwise.

Bar: the same sum in 64 bits.  An output element is at most ceil(K / 16) + 3 fused multiply-adds in
one chain, then 2 + 15 + 2 additions of partial sums and the add of the old value, each rounded
once: |gpu - exact| <= (ceil(K / 16) + 23) 2^-24 (|old| + sum_k |a_k b_kj|) to first order.
"""
import numpy as np
import pytest

from sapphire_amd import capi, synth
from tests import helpers as h

pytestmark = pytest.mark.gpu

# (N, K, batch): edges of 16 and of 64 columns; K below, at and past whole rounds of 16 wavefronts
# with 4 rows at a time; both sides of the line between the two widths; batches at odd strides
SHAPES = [(1, 64, 1), (15, 65, 1), (16, 1024, 1), (17, 79, 1), (63, 1001, 1), (64, 4097, 1),
          (65, 127, 1), (1023, 1024, 1), (2048, 257, 1), (2049, 70, 1), (8255, 1001, 1),
          (37, 333, 3), (128, 130, 16), (129, 130, 16), (65, 66, 25), (65, 66, 26),
          # past the short K: the edges of 16 columns, of 4 rows at a time, of the two widths
          (1, 320, 1), (1, 321, 1), (15, 337, 1), (17, 383, 1), (65, 385, 1), (2048, 321, 1),
          (2049, 321, 1), (128, 322, 16), (129, 322, 16), (65, 324, 25), (65, 324, 26)]


@pytest.mark.parametrize("flags", [0, capi.SPH_GEMM_OVERWRITE])
@pytest.mark.parametrize("shape", SHAPES)
def test_one_row_against_64_bits(dev, shape, flags):
    N, K, batch = shape
    h.announce("sph_gemm_f32_ex one row", shape, "flags", flags)
    A = synth.uniform(811, (batch, 1, K))
    B = synth.uniform(812, (batch, K, N))
    C = synth.uniform(813, (batch, 1, N))
    padded = np.concatenate([C.ravel(), np.full(64, 7.0, np.float32)])
    dC, dA, dB = (capi.DeviceBuffer.from_array(x) for x in (padded, A, B))
    capi.call("sph_gemm_f32_ex", dC.ptr, dA.ptr, dB.ptr, 1, N, K, batch, N, K, K * N, flags)
    out = dC.download(np.float32, padded.shape)
    for d in (dC, dA, dB):
        d.release()
    assert np.all(out[C.size:] == 7.0), "write past the row"
    got = out[:C.size].reshape(C.shape).astype(np.float64)
    old = np.zeros_like(C) if flags else C
    a, b = A.astype(np.float64), B.astype(np.float64)
    bound = ((K + 15) // 16 + 23) * 2.0 ** -24 * (np.abs(old) + np.abs(a) @ np.abs(b))
    assert np.all(np.abs(got - (old + a @ b)) <= bound)


@pytest.mark.parametrize("K", [130, 330])
@pytest.mark.parametrize("relu", [0, capi.SPH_LINEAR_RELU])
def test_one_row_bias_and_relu(dev, relu, K):
    N = 77
    h.announce("sph_linear_forward_f32 one row, flags", relu)
    x, W, bias = synth.uniform(821, (1, K)), synth.uniform(822, (K, N)), synth.uniform(823, (N,))
    dy, dx, dW, db = (capi.DeviceBuffer.from_array(v)
                      for v in (np.zeros(N, np.float32), x, W, bias))
    capi.call("sph_linear_forward_f32", dy.ptr, dx.ptr, dW.ptr, db.ptr, 1, K, N, relu)
    got = dy.download(np.float32, (1, N))
    for d in (dy, dx, dW, db):
        d.release()
    want = bias + x.astype(np.float64) @ W
    bound = ((K + 15) // 16 + 23) * 2.0 ** -24 * (np.abs(bias) + np.abs(x) @ np.abs(W))
    if relu:
        want = np.maximum(want, 0)
    assert np.all(np.abs(got - want) <= bound)
