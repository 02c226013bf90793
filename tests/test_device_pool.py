"""CPU: the pool of device blocks that a context keeps between runs
(csrc/devpool.h) over counted stand-in memory: what it keeps, what it gives
out again, and what it gives back."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MB, GB = 1 << 20, 1 << 30
LIMIT = 20 * GB


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("pool") / "pool.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-pthread", "-o", so,
                    os.path.join(ROOT, "tests", "harness", "pool_cpu.cpp")], check=True)
    H = C.CDLL(so)
    H.pool_new.restype = C.c_void_p
    H.pool_get.restype = H.pool_held.restype = C.c_longlong
    for f, a in (("pool_new", [C.c_longlong]), ("pool_delete", [C.c_void_p]), ("mem_set", [C.c_longlong]),
                 ("pool_get", [C.c_void_p, C.c_longlong]), ("pool_put", [C.c_void_p, C.c_longlong]),
                 ("pool_trim", [C.c_void_p]), ("pool_held", [C.c_void_p]), ("mem_counts", [C.POINTER(C.c_longlong)]),
                 ("pool_stress", [C.c_void_p, C.c_int, C.c_int])):
        getattr(H, f).argtypes = a
    return H


class Pool:
    def __init__(self, H, limit=LIMIT, memory=288 * GB):
        self.H, self.h = H, H.pool_new(limit)
        H.mem_set(memory)
        self.before = self.counts()

    def counts(self):
        c = (C.c_longlong * 4)()
        self.H.mem_counts(c)
        return list(c)

    @property
    def allocs(self):
        return self.counts()[1] - self.before[1]

    @property
    def live(self):
        return self.counts()[0]

    def run(self, *sizes):
        """One run: every block taken, then every block given back."""
        blocks = [self.H.pool_get(self.h, n) for n in sizes]
        assert all(blocks) and len(set(blocks)) == len(blocks)
        for b in blocks:
            self.H.pool_put(self.h, b)
        return blocks

    def close(self):
        self.H.pool_delete(self.h)
        c = self.counts()
        assert c[0] == 0 and c[1] == c[2] and c[3] == 0     # all memory back, nothing freed twice


@pytest.fixture
def pool(harness):
    p = Pool(harness)
    yield p
    p.close()


def test_repeated_run_allocates_once(pool):
    sizes = (100, 4 * MB, 9 * GB, 300, 40 * MB)
    first = pool.run(*sizes)
    n = pool.allocs
    for _ in range(3):
        assert sorted(pool.run(*sizes)) == sorted(first)
    assert pool.allocs == n == len(sizes)


def test_runs_of_other_sizes_after_a_large_one_do_not_allocate(pool):
    """A 16 GiB block of an earlier run serves later ones of 4 to 8 GiB, which
    otherwise find no room beside it and allocate on every call."""
    pool.run(16 * GB, 4 * MB)
    n = pool.allocs
    for size in (6, 4, 8, 7, 5, 16, 6):
        pool.run(size * GB, 4 * MB)
    assert pool.allocs == n and pool.live <= LIMIT


def test_returned_block_is_kept_and_others_make_room(pool):
    pool.run(9 * GB)
    pool.run(12 * GB)            # does not fit beside the 9 GiB
    n = pool.allocs
    pool.run(12 * GB)
    assert pool.allocs == n
    pool.run(10 * GB)
    assert pool.allocs == n and pool.H.pool_held(pool.h) <= LIMIT


def test_small_arrays_leave_the_large_block_alone(pool):
    pool.run(16 * GB)
    b = [pool.H.pool_get(pool.h, n) for n in (100, 40 * MB, 255 * MB)]
    n = pool.allocs
    pool.run(16 * GB)
    assert pool.allocs == n
    for q in b:
        pool.H.pool_put(pool.h, q)


@pytest.mark.parametrize("n,kept", [(3 * MB, True), (3 * MB // 2, True), (3 * MB // 2 - 256, False), (300, False)])
def test_reuse_up_to_twice_the_size(n, kept, pool):
    pool.run(3 * MB)
    pool.run(n)
    assert pool.allocs == (1 if kept else 2)


def test_limit_is_never_exceeded(pool):
    for size in (19 * GB, 20 * GB, 21 * GB, 1, 20 * GB + 1, 3 * GB, 18 * GB, 500 * MB):
        pool.run(size, 70 * MB)
        assert pool.H.pool_held(pool.h) <= LIMIT and pool.live == pool.H.pool_held(pool.h)


def test_no_limit_keeps_nothing(harness):
    p = Pool(harness, limit=0)
    p.run(100, 5 * GB)
    assert p.live == 0
    p.close()


def test_trim_gives_idle_blocks_back(pool):
    out = pool.H.pool_get(pool.h, 2 * GB)
    pool.run(5 * GB, 3 * MB)
    pool.H.pool_trim(pool.h)
    assert pool.live == 2 * GB and pool.H.pool_held(pool.h) == 0
    pool.H.pool_put(pool.h, out)
    assert pool.H.pool_held(pool.h) == 2 * GB


def test_failed_allocation_leaves_the_pool_usable(harness):
    p = Pool(harness, memory=10 * GB)
    assert p.H.pool_get(p.h, 11 * GB) == 0
    p.run(6 * GB)
    assert p.H.pool_get(p.h, 7 * GB) == 0       # the caller's allocator trims and tries again
    p.H.pool_trim(p.h)
    p.run(7 * GB)
    p.close()


def test_threads(harness):
    p = Pool(harness, limit=64 * MB)
    assert harness.pool_stress(p.h, 8, 3000) == 0
    assert p.H.pool_held(p.h) <= 64 * MB
    p.close()
