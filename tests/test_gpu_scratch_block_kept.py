"""The scratch block that stays with a thread's own stream: taken again without an allocation, replaced
when it is too small, not used for a stream that the program has set, given back by a trim."""
import ctypes
import threading

import numpy as np
import pytest

from oracle import pyoracle as po
from sapphire_amd import capi, synth
from tests import helpers as h

pytestmark = pytest.mark.gpu


class Product:
    """A x A of `n` rows with four entries each, whose staging takes n * (3 * 17 + 64) * 8 bytes."""

    def __init__(self, n, seed):
        self.n, self.capacity = n, 17 * n
        self.A = synth.csr_matrix(seed, n, n, 100.0 * 4 / n)
        self.want = po.spgemm_csr(self.A, self.A, n, n, n)

    def run(self):
        bufs = [capi.DeviceBuffer.from_array(x) for x in self.A]
        V, COL = (capi.DeviceBuffer(4 * self.capacity) for _ in range(2))
        ROW = capi.DeviceBuffer(4 * (self.n + 1))
        before = allocations()
        capi.call("sph_spgemm_f32", V.ptr, COL.ptr, ROW.ptr, self.capacity, *[b.ptr for b in bufs],
                  *[b.ptr for b in bufs], self.n, self.n, self.n, None)
        made = allocations() - before
        capi.sync()
        v, col, row = self.want
        assert np.array_equal(ROW.download(np.uint32, (self.n + 1,)), row)
        count = int(row[-1])
        assert count <= self.capacity
        assert np.array_equal(COL.download(np.uint32, (self.capacity,))[:count], col)
        assert np.array_equal(V.download(np.float32, (self.capacity,))[:count].view(np.uint32),
                              v.view(np.uint32))
        for d in bufs + [V, COL, ROW]:
            d.release()
        return made


def allocations():
    count = ctypes.c_uint64(0)
    capi.call("sph_allocation_count", ctypes.byref(count))
    return count.value


def test_taken_again_and_replaced(dev):
    h.announce("scratch block of a stream, two sizes in turn")
    small, large = Product(3000, 61), Product(12000, 62)
    capi.call("sph_mem_pool_trim")
    assert [small.run(), small.run(), large.run(), small.run(), large.run()] == [1, 0, 1, 0, 0]
    capi.call("sph_mem_pool_trim")
    assert [small.run(), small.run()] == [1, 0]


def test_every_thread_has_its_own(dev):
    h.announce("scratch blocks of four threads at once")
    products = [Product(2000 + 500 * t, 63 + t) for t in range(4)]
    made, errors = [None] * 4, []

    def work(t):
        try:
            capi.call("sph_set_device", 0)
            capi.call("sph_mem_pool_trim")
            # (other threads allocate at the same time: only what the results are is looked at)
            for _ in range(10):
                products[t].run()
        except BaseException as exc:  # noqa: BLE001 - reported by the main thread
            errors.append((t, repr(exc)))

    # twice: the second set takes over the streams, and the blocks, of the first
    for _ in range(2):
        threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
        for th in threads:
            th.start()
        for th in threads:
            th.join()
    assert not errors, errors


def test_not_for_a_stream_of_the_programs(dev):
    h.announce("scratch blocks on a stream that the program has set")
    product = Product(3000, 67)
    product.run()
    stream = ctypes.c_void_p()
    assert capi.lib().hipStreamCreateWithFlags(ctypes.byref(stream), 1) == 0
    try:
        capi.call("sph_set_stream", stream)
        assert [product.run(), product.run()] == [1, 1]
    finally:
        capi.call("sph_set_stream", None)
    assert product.run() == 0
    assert capi.lib().hipStreamDestroy(stream) == 0
