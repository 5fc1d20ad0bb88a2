"""fp32 products of fewer tiles than compute units: the last M % 4 rows and N % 4 columns are strips
on compute units that have no tile, where that leaves the tiled kernel whole rows and steps.

Integer-valued operands make every partial sum exact: out bit for bit that of the CPU loop,
whichever way the operands are stored and wherever they start.
"""
import numpy as np
import pytest

from oracle import pyoracle as po
from sapphire_amd import capi, synth
from tests import helpers as h

pytestmark = pytest.mark.gpu
TA, TB = capi.SPH_GEMM_TRANS_A, capi.SPH_GEMM_TRANS_B

# (M, N, K, batch): K-split tiles with both strips, with none (every compute unit has a tile or a
# strip already; a K in broken steps); 64-tiles with both, with one (both would leave whole tiles,
# which are walked without strips), with none that would help; a batch
SHAPES = [(513, 515, 96, 1), (577, 515, 64, 1), (641, 643, 64, 1), (513, 515, 70, 1),
          (131, 4097, 48, 1), (769, 770, 32, 1), (1025, 515, 128, 1), (66, 4097, 64, 1),
          (1025, 515, 40, 1), (131, 133, 64, 8)]


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("flags", [0, TA, TB, TA | TB])
@pytest.mark.parametrize("shape", SHAPES)
def test_exact_on_integers(dev, shape, flags, offset):
    M, N, K, batch = shape
    h.announce("sph_gemm_f32_ex strips on idle compute units", shape, "flags", flags, offset)
    A = synth.small_integers(871, (batch, M, K), span=4)
    B = synth.small_integers(872, (batch, K, N), span=4)
    C = synth.small_integers(873, (batch, M, N), span=100)
    ref = po.gemm_rows(C.copy(), A, B, M, N, K, batch=batch, threads=8)
    pad = np.zeros(offset, np.float32)
    stored = [np.concatenate([pad, (x.swapaxes(-1, -2) if flags & f else x).ravel()])
              for x, f in ((A, TA), (B, TB))]
    dA, dB = (capi.DeviceBuffer.from_array(x) for x in stored)
    guard = np.full(64, 7.0, np.float32)
    dC = capi.DeviceBuffer.from_array(np.concatenate([guard, C.ravel(), guard]))
    capi.call("sph_gemm_f32_ex", dC.at(256), dA.at(4 * offset), dB.at(4 * offset), M, N, K, batch,
              M * N, M * K, K * N, flags)
    out = dC.download(np.float32, (C.size + 128,))
    for d in (dA, dB, dC):
        d.release()
    assert np.all(out[:64] == 7.0) and np.all(out[-64:] == 7.0), "write outside out"
    assert np.array_equal(out[64:-64].reshape(C.shape), ref)
