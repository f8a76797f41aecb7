"""The device memory pool (ferric_amd/csrc/memory.hip) on the CPU, over a runtime that only hands out addresses: what has to be refused, what may
be handed out again, and what a capture on one thread means for the others."""
import ctypes as C
import os
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

from conftest import ROOT

KIB, MIB, GIB = 1 << 10, 1 << 20, 1 << 30


@pytest.fixture(scope="module")
def library(tmp_path_factory):
    d = tmp_path_factory.mktemp("pool")
    obj = str(d / "pool.o")
    subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "--offload-host-only", "--offload-arch=gfx950", "-x", "hip", "-std=c++17", "-O1", "-fPIC", "-c",
                    os.path.join(ROOT, "tests", "pool_harness.cpp"), "-o", obj], check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    return obj


class Pool:
    def __init__(self, obj, path):
        subprocess.run(["g++", "-shared", "-Wl,-Bsymbolic", "-o", path, obj, "-lpthread"], check=True)
        self.c = C.CDLL(path)
        for name, res, args in (("h_malloc", C.c_int, [C.c_size_t, C.c_void_p]), ("h_free", C.c_int, [C.c_void_p]), ("h_range", C.c_size_t, [C.c_void_p]),
                                ("h_stream", C.c_void_p, []), ("h_stream_destroy", C.c_int, [C.c_void_p]), ("h_begin", None, [C.c_void_p, C.c_int]),
                                ("h_end", C.c_int, [C.c_void_p]), ("h_bytes", C.c_size_t, []), ("h_text", C.c_char_p, []), ("h_trim", None, [])):
            getattr(self.c, name).restype, getattr(self.c, name).argtypes = res, args

    def malloc(self, n):
        """(return code, address)"""
        p = C.c_void_p(1)
        rc = self.c.h_malloc(n, C.byref(p))
        return rc, p.value

    def new(self, n):
        rc, p = self.malloc(n)
        assert rc == 0 and p
        return p


@pytest.fixture
def pool(library, tmp_path):
    return Pool(library, str(tmp_path / "pool.so"))       # a copy of its own: the pool is as old as the library


@pytest.mark.parametrize("n", [0, 100, 5000, 3 * MIB, 900 * MIB])
def test_a_second_free_is_refused(pool, n):
    """Also of a block that has been clean for a while, and of one too large to be kept. Nothing is given to two owners afterwards."""
    p = pool.new(n)
    assert pool.c.h_range(p) == n + 256
    assert pool.c.h_free(p) == 0 and pool.c.h_range(p) == 0
    held = pool.c.h_bytes()
    assert pool.c.h_free(p) != 0
    for _ in range(300):
        assert pool.c.h_free(pool.new(n + 8)) == 0        # of the same class; has waited for the device meanwhile
    assert pool.c.h_free(p) != 0 and pool.c.h_bytes() >= held
    mine = [pool.new(n) for _ in range(5)]
    assert len(set(mine)) == 5 and all(pool.c.h_range(q) == n + 256 for q in mine)
    assert [pool.c.h_free(q) for q in mine] == [0] * 5


def test_a_block_is_handed_out_again_only_after_the_device_was_idle(pool):
    for n in (2000, 700 * KIB, 300 * MIB):
        freed_under_work = set()
        for _ in range(600):
            p = pool.new(n)
            if not pool.c.h_busy():
                freed_under_work.clear()
            assert p not in freed_under_work
            pool.c.h_work()
            freed_under_work.add(p)
            pool.c.h_free(p)
        assert pool.c.h_waits() > 0


def test_cached_memory_is_found_beside_a_capture(pool):
    """With nothing left to allocate (8 GiB: eleven blocks of 704 MiB and one of 448), not even what the wait needs."""
    s = pool.c.h_stream()
    blocks = [pool.new(704 * MIB - 256) for _ in range(11)] + [pool.new(448 * MIB - 256)]
    assert pool.c.h_bytes() == 8 * GIB
    with ThreadPoolExecutor(1) as other:
        pool.c.h_begin(s, 1)
        for p in blocks[:2]:
            pool.c.h_free(p)
        assert other.submit(pool.malloc, 704 * MIB - 256).result()[0] == 0
        assert pool.c.h_end(s) == 0


def test_cached_memory_is_bounded_and_given_back(pool):
    blocks = [pool.new(100 * MIB + k) for k in range(40)]
    for p in blocks:
        assert pool.c.h_free(p) == 0
    assert pool.c.h_bytes() <= 2 * GIB
    assert all(pool.c.h_free(p) != 0 for p in blocks)     # the cached ones and those the runtime has back
    pool.c.h_trim()
    assert pool.c.h_bytes() == 0
    big = [pool.new(6 * GIB), pool.new(GIB)]               # what the pool holds back is not what is missing
    pool.c.h_free(big[0])
    pool.new(500 * MIB)
    pool.c.h_free(pool.new(700 * MIB))
    pool.new(6 * GIB)


@pytest.mark.parametrize("n", [9 * GIB, 1 << 60, (1 << 63) + 5, (1 << 64) - (1 << 60), (1 << 64) - (1 << 60) - 256, (1 << 64) - 1000, (1 << 64) - 257, (1 << 64) - 256, (1 << 64) - 1])
def test_a_size_that_no_device_has_is_refused(pool, n):
    """Among them negative counts cast to size_t; none may come out as a small class or a null pointer."""
    for _ in range(2):
        rc, p = pool.malloc(n)
        assert rc != 0 and not p and pool.c.h_bytes() == 0


@pytest.mark.parametrize("n", [0, 1, 768, 769, 1024, 1025, 64 * KIB - 256, 64 * KIB - 255, MIB, 512 * MIB - 256, 512 * MIB - 255, 768 * MIB - 257, 768 * MIB - 256, 768 * MIB - 255])
def test_a_block_holds_what_was_asked_for(pool, n):
    p = pool.new(n)
    assert n + 256 <= pool.c.h_bytes() <= max(1024, (n + 256) * 9 // 8) and pool.c.h_range(p) == n + 256
    assert pool.c.h_range(p + n + 255) == 1


@pytest.mark.parametrize("through_library", [0, 1])
def test_a_thread_that_captures_gets_no_memory_and_loses_none(pool, through_library):
    """Cached blocks of the size or not. What it frees stays with the pool, past the bound too, and is given back later. A capture that
    the pool knows of stays valid."""
    cached, big = [pool.new(3000) for _ in range(3)], [pool.new(300 * MIB) for _ in range(9)]
    for p in cached:
        pool.c.h_free(p)
    for _ in range(300):
        pool.c.h_free(pool.new(9000))                      # has waited: the three are clean
    s = pool.c.h_stream()
    pool.c.h_begin(s, through_library)
    held = pool.c.h_bytes()
    for n in (3000, 300 * MIB, GIB):
        assert pool.malloc(n)[0] != 0
    for p in big:
        assert pool.c.h_free(p) == 0
    pool.c.h_trim()
    assert pool.c.h_bytes() == held
    assert pool.c.h_end(s) == (0 if through_library else 1)
    pool.c.h_free(pool.new(300 * MIB))
    assert pool.c.h_bytes() <= 2 * GIB
    pool.c.h_trim()
    assert pool.c.h_bytes() == 0
    assert pool.c.h_stream_destroy(s) == 0


def test_a_capture_ends_with_its_thread_or_its_stream(pool):
    a, b = pool.c.h_stream(), pool.c.h_stream()
    with ThreadPoolExecutor(1) as other:
        pool.c.h_begin(a, 1)
        assert other.submit(pool.c.h_end, a).result() == 2
        assert pool.malloc(100)[0] != 0 and other.submit(pool.malloc, 100).result()[0] == 0
        for _ in range(300):                               # the other thread's waits
            assert other.submit(pool.c.h_free, other.submit(pool.new, 5000).result()).result() == 0
        assert pool.c.h_waits() > 0 and pool.c.h_end(a) == 0
        pool.c.h_begin(a, 1)
        pool.c.h_begin(b, 1)
        assert pool.c.h_end(a) == 0 and pool.malloc(100)[0] != 0
        pool.c.h_stream_destroy(b)
        pool.new(100)
        pool.c.h_begin(a, 0)                               # through the runtime: the other thread goes on, whatever becomes of the capture
        for _ in range(300):
            assert other.submit(pool.c.h_free, other.submit(pool.new, 9000).result()).result() == 0
        pool.c.h_end(a)


@pytest.mark.parametrize("n", [0, 1000, 900 * MIB])
def test_a_copy_belongs_into_one_block_in_use(pool, n):
    """As far as it was asked for (and the slack behind it), whatever the class holds beyond; on its own device; not after the free."""
    p, place = pool.new(n), pool.c.h_place
    place.argtypes = [C.c_void_p, C.c_size_t, C.c_int]
    inside, outside, elsewhere = 0, 1, 2
    assert [place(*a) for a in ((p, n + 256, 0), (p + 100, n + 156, 0), (p + n + 255, 1, 0))] == [inside] * 3
    assert [place(*a) for a in ((p, n + 257, 0), (p + 100, n + 157, 0), (p + n + 255, 2, 0), (p, (1 << 64) - 1, 0), (p + 8, (1 << 64) - 8, 0))] == [outside] * 5
    assert [place(*a) for a in ((p - 1, 2, 0), (p, 1, 1), (4096, 1, 0), (p + 2 * GIB, 1, 0))] == [elsewhere] * 4
    pool.c.h_free(p)
    assert place(p, 1, 0) == (outside if n < GIB // 2 else elsewhere)       # still the pool's, or the runtime's again
