"""Where the CSR calls take their scratch blocks from: a pool of the library's own that keeps up to
512 MiB of freed blocks.  The release threshold of the device's default pool is the program's and
stays as the program set it; a default pool that keeps at least as much is used instead."""
import ctypes

import numpy as np
import pytest

from sapphire_amd import capi
from tests import helpers as h

pytestmark = pytest.mark.gpu

KEPT = 512 << 20
THRESHOLD, RESERVED = 4, 5  # hipMemPoolAttrReleaseThreshold, hipMemPoolAttrReservedMemCurrent


def hip(name, *args):
    assert getattr(capi.lib(), name)(*args) == 0, name


def free_memory():
    free, total = ctypes.c_size_t(0), ctypes.c_size_t(0)
    hip("hipMemGetInfo", ctypes.byref(free), ctypes.byref(total))
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


class DefaultPool:
    def __init__(self):
        self.pool = ctypes.c_void_p()
        hip("hipDeviceGetDefaultMemPool", ctypes.byref(self.pool), 0)

    def get(self, what):
        value = ctypes.c_uint64(0)
        hip("hipMemPoolGetAttribute", self.pool, what, ctypes.byref(value))
        return value.value

    def set_threshold(self, value):
        hip("hipMemPoolSetAttribute", self.pool, THRESHOLD, ctypes.byref(ctypes.c_uint64(value)))


@pytest.fixture
def default_pool(dev):
    pool = DefaultPool()
    before = pool.get(THRESHOLD)
    yield pool
    pool.set_threshold(before)


class Conversion:
    """Dense -> CSR of M rows without an entry, with a capacity that asks for `scratch` bytes."""

    N, PER_ROW = 4096, 450

    def __init__(self, M):
        self.M, self.capacity = M, M * self.PER_ROW
        self.scratch = M * (2 * self.PER_ROW + 32) * 8
        self.dense = capi.DeviceBuffer(4 * M * self.N)
        capi.call("sph_fill_f32", self.dense.ptr, 0.0, M * self.N)
        self.V, self.COL = (capi.DeviceBuffer(4 * self.capacity) for _ in range(2))
        self.ROW = capi.DeviceBuffer(4 * (M + 1))

    def run(self):
        nnz = ctypes.c_uint32(7)
        capi.call("sph_csr_from_dense_f32", self.V.ptr, self.COL.ptr, self.ROW.ptr, self.capacity,
                  self.dense.ptr, self.M, self.N, self.N, ctypes.byref(nnz))
        capi.sync()
        assert nnz.value == 0

    def release(self):
        for d in (self.dense, self.V, self.COL, self.ROW):
            d.release()


@pytest.mark.parametrize("value", [0, 1 << 20, KEPT - 1, KEPT, 2 * KEPT])
def test_the_programs_threshold_survives(default_pool, value):
    h.announce("scratch blocks beside a threshold of", value)
    default_pool.set_threshold(value)
    COL = capi.DeviceBuffer.from_array(np.zeros(4, np.uint32))
    ROW = capi.DeviceBuffer.from_array(np.arange(5, dtype=np.uint32))
    problems = ctypes.c_uint32(1)
    capi.call("sph_csr_validate_u32", COL.ptr, ROW.ptr, 4, 1, 4, ctypes.byref(problems))
    case = Conversion(8192)
    case.run()
    assert problems.value == 0 and default_pool.get(THRESHOLD) == value
    for d in (COL, ROW, case):
        d.release()


def test_blocks_are_kept_up_to_the_bound_and_given_back(default_pool):
    h.announce("scratch blocks kept and trimmed")
    default_pool.set_threshold(0)
    slack = 16 << 20
    for M in (32768, 131072):  # 244 and 977 MB of staging
        case = Conversion(M)
        capi.call("sph_mem_pool_trim")
        capi.DeviceBuffer(1 << 20).release()
        reserved, before = default_pool.get(RESERVED), free_memory()
        case.run()
        if case.scratch < KEPT:
            assert before - free_memory() >= case.scratch - slack  # there for the next call
            case.run()
            assert before - free_memory() <= case.scratch + slack  # which takes no more
        assert default_pool.get(RESERVED) == reserved  # not the program's pool
        assert settles(case.dense, lambda: before - free_memory() <= KEPT + slack)
        capi.call("sph_mem_pool_trim")
        assert settles(case.dense, lambda: before - free_memory() <= slack)
        case.release()


def test_a_pool_that_keeps_as_much_is_used(default_pool):
    h.announce("scratch blocks from the default pool")
    default_pool.set_threshold(2**64 - 1)
    case = Conversion(32768)
    capi.call("sph_mem_pool_trim")
    reserved = default_pool.get(RESERVED)
    case.run()
    assert default_pool.get(RESERVED) - reserved >= case.scratch
    capi.call("sph_mem_pool_trim")
    assert default_pool.get(RESERVED) == reserved
    case.release()
