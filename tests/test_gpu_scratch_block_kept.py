"""The scratch block that stays with a thread's own stream: taken again without an allocation, replaced
when it is too small, not used for a stream that the program has set, given back by a trim of any
thread, and together no more than the library's pool keeps."""
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


def free_memory():
    free, total = ctypes.c_size_t(0), ctypes.c_size_t(0)
    assert capi.lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def settles(buffer, holds):
    """True once `holds()`: the runtime keeps a block that its last commands used until some others
    have followed.  (Nothing is freed here: hipFree empties the pools.)"""
    for _ in range(200):
        if holds():
            return True
        capi.call("sph_fill_f32", buffer.ptr, 0.0, 4)
        capi.sync()
    return False


class Threads:
    """Threads that are alive until the end of the block, each with a stream of its own."""

    def __init__(self, count):
        self.gates = [[threading.Semaphore(0), threading.Semaphore(0)] for _ in range(count)]
        self.jobs, self.results, self.errors = [None] * count, [None] * count, []
        self.threads = [threading.Thread(target=self.work, args=(t,)) for t in range(count)]

    def work(self, t):
        capi.call("sph_set_device", 0)
        while True:
            self.gates[t][0].acquire()
            if self.jobs[t] is None:
                return
            try:
                self.results[t] = self.jobs[t]()
            except BaseException as exc:  # noqa: BLE001 - reported by the main thread
                self.errors.append((t, repr(exc)))
            self.gates[t][1].release()

    def run(self, t, job):
        """job() on thread t, waited for."""
        self.jobs[t] = job
        self.gates[t][0].release()
        self.gates[t][1].acquire()
        assert not self.errors, self.errors
        return self.results[t]

    def __enter__(self):
        for th in self.threads:
            th.start()
        return self

    def __exit__(self, *_):
        for t in range(len(self.threads)):
            self.jobs[t] = None
            self.gates[t][0].release()
        for th in self.threads:
            th.join()


def test_a_trim_gives_back_what_other_threads_keep(dev):
    """Threads that are alive and idle, and threads that have ended."""
    h.announce("scratch blocks of other threads, trimmed")
    product, count = Product(24000, 68), 4
    block, slack = 24000 * (3 * 17 + 64) * 8, 16 << 20
    buffer = capi.DeviceBuffer(1 << 20)

    def given_back(before):
        capi.call("sph_mem_pool_trim")
        return settles(buffer, lambda: before - free_memory() <= slack)

    with Threads(count) as threads:
        for t in range(count):  # (streams and what they hold are made once)
            threads.run(t, product.run)
        capi.call("sph_mem_pool_trim")
        before = free_memory()
        for _ in range(2):
            assert [threads.run(t, product.run) for t in range(count)] == [1] * count
            assert [threads.run(t, product.run) for t in range(count)] == [0] * count
            assert before - free_memory() >= count * block - slack
            assert given_back(before)
        for t in range(count):
            threads.run(t, product.run)
    assert before - free_memory() >= count * block - slack
    assert given_back(before)
    buffer.release()


def test_a_trim_leaves_a_stream_under_capture_alone(dev):
    h.announce("scratch block of a stream under capture")
    product, n = Product(3000, 69), 1000
    out = capi.DeviceBuffer.from_array(np.zeros(n, np.float32))
    graph = ctypes.c_void_p()

    def record():
        capi.call("sph_fill_f32", out.ptr, 3.0, n)
        capi.call("sph_graph_end_capture", ctypes.byref(graph))

    def replay():
        capi.call("sph_fill_f32", out.ptr, 1.0, n)
        capi.call("sph_graph_launch", graph)
        capi.sync()
        return out.download(np.float32, (n,))

    with Threads(1) as threads:
        threads.run(0, product.run)
        threads.run(0, lambda: capi.call("sph_graph_begin_capture"))
        capi.call("sph_mem_pool_trim")
        threads.run(0, record)
        for _ in range(3):
            assert np.all(threads.run(0, replay) == 3.0)
            product.run()
            capi.call("sph_mem_pool_trim")
        threads.run(0, product.run)
        threads.run(0, lambda: capi.call("sph_graph_destroy", graph))
    out.release()


def test_all_of_them_together_are_bounded(dev):
    """32 MiB each, 512 MiB together: the first 16 of 20 threads keep theirs."""
    h.announce("scratch blocks of 20 threads")
    product, count = Product(32000, 70), 20
    with Threads(count) as threads:
        capi.call("sph_mem_pool_trim")
        for t in range(count):
            threads.run(t, product.run)
        assert [threads.run(t, product.run) for t in range(count)] == [0] * 16 + [1] * 4
        capi.call("sph_mem_pool_trim")
