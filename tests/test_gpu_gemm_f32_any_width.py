"""fp32 GEMM on the straight-to-LDS kernels with rows that are no whole number of 4 floats: the
last chunk of a k-major operand's last row is copied early and its values are read from there.

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

# (M, N, K, batch).  64 x 64 tiles: every remainder of 4, K of whole steps, one more and one less,
# one step only, rows of one chunk and a piece; 64 x 32 tiles with K split (65 to 128 tiles of 64);
# 128 x 128 tiles; a batch.
SHAPES = ([(704 - r, 999 + r, 128 + r, 1) for r in range(4)] +
          [(701, 999, 64, 1), (701, 999, 63, 1), (701, 999, 48, 1), (701, 999, 16, 1),
           (701, 999, 17, 1), (701, 999, 33, 1), (8501, 5, 65, 1), (6, 8501, 32, 1),
           (513, 515, 64, 1), (513, 515, 65, 1), (522, 521, 95, 1), (66, 2103, 96, 1),
           (3001, 2687, 48, 1), (3001, 2686, 37, 1), (333, 335, 100, 7)])


@pytest.mark.parametrize("flags", [0, TA, TB, TA | TB])
@pytest.mark.parametrize("shape", SHAPES)
def test_exact_on_integers(dev, shape, flags):
    M, N, K, batch = shape
    h.announce("sph_gemm_f32_ex any width", shape, "flags", flags)
    A = synth.small_integers(881, (batch, M, K), span=4)
    B = synth.small_integers(882, (batch, K, N), span=4)
    C = synth.small_integers(883, (batch, M, N), span=100)
    ref = po.gemm_rows(C.copy(), A, B, M, N, K, batch=batch, threads=8)
    stored = [np.ascontiguousarray(x.swapaxes(-1, -2)) if flags & f else x
              for x, f in ((A, TA), (B, TB))]
    dA, dB = (capi.DeviceBuffer.from_array(x) for x in stored)
    padded = np.concatenate([np.full(64, 7.0, np.float32), C.ravel(), np.full(64, 7.0, np.float32)])
    for overwrite in (0, OW):
        dC = capi.DeviceBuffer.from_array(padded)
        capi.call("sph_gemm_f32_ex", dC.ptr + 4 * 64, dA.ptr, dB.ptr, M, N, K, batch, M * N, M * K,
                  K * N, flags | overwrite)
        out = dC.download(np.float32, padded.shape)
        dC.release()
        assert np.all(out[:64] == 7.0) and np.all(out[-64:] == 7.0), "write outside out"
        want = ref - C if overwrite else ref
        assert np.array_equal(out[64:-64].reshape(C.shape), want), overwrite
    for d in (dA, dB):
        d.release()


@pytest.mark.parametrize("flags", [0, TA])
@pytest.mark.parametrize("shape", [(702, 1001, 96), (523, 513, 100)])
def test_what_follows_a_row_does_not_reach_the_result(dev, shape, flags):
    """The floats behind the last row of an operand are NaN: none of them may reach out."""
    M, N, K = shape
    h.announce("sph_gemm_f32_ex any width, NaN behind the operands", shape, flags)
    A = synth.small_integers(891, (M, K), span=4)
    B = synth.small_integers(892, (K, N), span=4)
    ref = po.gemm_rows(np.zeros((M, N), np.float32), A, B, M, N, K, threads=8)
    tail = np.full(64, np.nan, np.float32)
    dA, dB = (capi.DeviceBuffer.from_array(np.concatenate([x.ravel(), tail]))
              for x in (np.ascontiguousarray(A.T) if flags & TA else A, B))
    dC = capi.DeviceBuffer(4 * M * N)
    capi.call("sph_gemm_f32_ex", dC.ptr, dA.ptr, dB.ptr, M, N, K, 1, M * N, M * K, K * N, flags | OW)
    got = dC.download(np.float32, (M, N))
    for d in (dA, dB, dC):
        d.release()
    assert np.array_equal(got, ref)


@pytest.mark.parametrize("shape", [(702, 1001, 96), (1001, 1203, 37), (701, 1002, 48)])
def test_storage_does_not_change_a_bit(dev, shape):
    M, N, K = shape
    h.announce("sph_gemm_f32_ex any width, storage", shape)
    A, B, C = (synth.uniform(s, x) for s, x in ((895, (1, M, K)), (896, (1, K, N)),
                                                (897, (1, M, N))))
    plain = h.gpu_gemm_f32_ex(C, A, B, M, N, K, 0, batch=1)
    for flags in (TA, TB, TA | TB):
        As = np.ascontiguousarray(A.swapaxes(-1, -2)) if flags & TA else A
        Bs = np.ascontiguousarray(B.swapaxes(-1, -2)) if flags & TB else B
        got = h.gpu_gemm_f32_ex(C, As, Bs, M, N, K, flags, batch=1)
        assert np.array_equal(got.view(np.uint32), plain.view(np.uint32)), flags
