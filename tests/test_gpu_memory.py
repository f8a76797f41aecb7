"""Device memory and host copies of the library where they have to say no: stream captures, blocks freed twice, sizes and ranges that
no allocation has; and what they do beside each other on several threads and streams."""
import ctypes as C
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
KIB, MIB = 1 << 10, 1 << 20


def blocks_in_turn(F, nbytes, times=200):
    """How many different blocks `times` allocations get when each is freed before the next one."""
    lib, check, seen = F._lib.load(), F._lib.check, set()
    for _ in range(times):
        p = C.c_void_p()
        check(lib.fhip_malloc(C.byref(p), nbytes))
        seen.add(p.value)
        check(lib.fhip_free(p))
    return len(seen)


# ---- captures ----------------------------------------------------------------------------------------------------------------------

def test_a_capture_is_its_own_threads_whoever_tries_to_end_it(F):
    """The runtime refuses another thread; that thread's memory goes on as before (64 blocks of a small class, then a wait), and so does
    the capture."""
    lib, check = F._lib.load(), F._lib.check
    s, word = F.Stream(), F.Tensor.from_vec(np.zeros(4, np.float32), (4,))
    other = ThreadPoolExecutor(1)
    g = F.Graph.begin(s)
    check(lib.fhip_u32_add(word.buf.ptr, 1, 1, s.handle))
    h = C.c_void_p()
    assert other.submit(lib.fhip_graph_capture_end, s.handle, C.byref(h)).result() == F._lib.ERR_HIP
    check(lib.fhip_u32_add(word.buf.ptr, 1, 1, s.handle))
    g.end()
    for _ in range(3):
        g.launch()
    assert word.to_vec(s).view(np.uint32)[0] == 6
    assert other.submit(blocks_in_turn, F, 9000).result() <= 64
    assert blocks_in_turn(F, 9000) <= 64


def test_a_stream_destroyed_while_it_captures_ends_the_capture(F):
    s = F.Stream()
    F.Graph.begin(s)
    handle, s.handle = s.handle, None
    F._lib.check(F._lib.load().fhip_stream_destroy(handle))
    assert blocks_in_turn(F, 11000) <= 64
