"""fp16-input GEMM on the 64- and 128-tile kernels with rows that are no whole number of 8 halves:
the last chunk of a k-major operand's last row is copied early and moved to its place.

Integer-valued operands make every product and partial sum exact, so the result is compared bit
for bit with the CPU loop; out lies between guard words, and in one test NaN behind the operands.
That no copy reaches past an operand is not visible here (what it would bring feeds no output):
test_copy_offsets_cpu.py checks the offsets.
"""
import numpy as np
import pytest

from oracle import pyoracle as po
from sapphire_amd import capi, synth
from tests import helpers as h

pytestmark = pytest.mark.gpu
TA, TB, OW = capi.SPH_GEMM_TRANS_A, capi.SPH_GEMM_TRANS_B, capi.SPH_GEMM_OVERWRITE

# (M, N, K, batch).  64 x 64 tiles: every remainder of 8, the smallest rows with one chunk and a
# piece, K of whole steps, one more and one less, the fewest steps; 128 x 128 tiles with four and
# eight wavefronts, whole steps and not; few-tile shapes on both sides of the rule; a batch.
SHAPES = ([(704 - r, 640 + r, 256 + r, 1) for r in range(8)] +
          [(521, 523, 128, 1), (521, 523, 127, 1), (521, 523, 129, 1), (521, 523, 192, 1),
           (2100, 9, 320, 1), (9, 2100, 320, 1), (1201, 1203, 64, 1), (1201, 1203, 65, 1),
           (1201, 1203, 96, 1), (1201, 1205, 95, 1), (2100, 2101, 64, 1), (2100, 2103, 100, 1),
           (401, 501, 255, 1), (401, 501, 256, 1), (401, 501, 1537, 1), (333, 335, 300, 3)])


@pytest.mark.parametrize("flags", [0, TA, TB, TA | TB])
@pytest.mark.parametrize("shape", SHAPES)
def test_exact_on_integers(dev, shape, flags):
    M, N, K, batch = shape
    h.announce("sph_gemm_f16f32 any width", shape, "flags", flags)
    A = synth.small_integers(861, (batch, M, K), span=4).astype(np.float16)
    B = synth.small_integers(862, (batch, K, N), span=4).astype(np.float16)
    C = synth.small_integers(863, (batch, M, N), span=100)
    ref = po.gemm_rows(C.copy(), A.astype(np.float32), B.astype(np.float32), M, N, K,
                       batch=batch, threads=8)
    stored = [np.ascontiguousarray(x.swapaxes(-1, -2)) if flags & f else x
              for x, f in ((A, TA), (B, TB))]
    dA, dB = (capi.DeviceBuffer.from_array(x) for x in stored)
    padded = np.concatenate([np.full(64, 7.0, np.float32), C.ravel(), np.full(64, 7.0, np.float32)])
    for overwrite in (0, OW):
        dC = capi.DeviceBuffer.from_array(padded)
        capi.call("sph_gemm_f16f32", dC.ptr + 4 * 64, dA.ptr, dB.ptr, M, N, K, batch, M * N, M * K,
                  K * N, flags | overwrite)
        out = dC.download(np.float32, padded.shape)
        dC.release()
        assert np.all(out[:64] == 7.0) and np.all(out[-64:] == 7.0), "write outside out"
        want = ref - C if overwrite else ref
        assert np.array_equal(out[64:-64].reshape(C.shape), want), overwrite
    for d in (dA, dB):
        d.release()


@pytest.mark.parametrize("flags", [0, TA])
def test_what_follows_a_row_does_not_reach_the_result(dev, flags):
    """The halves behind the last row of an operand are NaN: none of them may reach out."""
    M, N, K = 661, 663, 200
    h.announce("sph_gemm_f16f32 any width, NaN behind the operands", flags)
    A = synth.small_integers(871, (M, K), span=4).astype(np.float16)
    B = synth.small_integers(872, (K, N), span=4).astype(np.float16)
    ref = po.gemm_rows(np.zeros((M, N), np.float32), A.astype(np.float32), B.astype(np.float32),
                       M, N, K, threads=8)
    tail = np.full(64, np.nan, np.float16)
    dA, dB = (capi.DeviceBuffer.from_array(np.concatenate([x.ravel(), tail]))
              for x in (np.ascontiguousarray(A.T) if flags & TA else A, B))
    dC = capi.DeviceBuffer(4 * M * N)
    capi.call("sph_gemm_f16f32", dC.ptr, dA.ptr, dB.ptr, M, N, K, 1, M * N, M * K, K * N, flags | OW)
    got = dC.download(np.float32, (M, N))
    for d in (dA, dB, dC):
        d.release()
    assert np.array_equal(got, ref)
