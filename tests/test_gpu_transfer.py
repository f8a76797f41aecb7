"""Copies through the library's pinned slots and the pool behind fhip_malloc, at the sizes where they change course: whole copies
against the bytes that went in, host dequantization against the oracle, freed memory that is still in use."""
import ctypes as C
import threading

import numpy as np
import pytest

from conftest import bits

pytestmark = pytest.mark.gpu
KIB, MIB = 1 << 10, 1 << 20


# one byte, tails of the 16-byte units, a slot's way up (640 KiB) and way down (1 MiB) and one byte on either side, more chunks
# than a copy holds slots (12); a copy back is made in parts from 96 KiB on (64 + offset bytes are added to n)
@pytest.mark.parametrize("n", [1, 3, 15, 17, 4096, 64 * KIB + 5, 96 * KIB - 65, 96 * KIB - 64, 96 * KIB + 1, 640 * KIB - 1, 640 * KIB, 640 * KIB + 1, MIB - 65, MIB - 64, MIB - 63, 2 * MIB + 1,
                               6 * MIB + 7, 21 * MIB + 4])
@pytest.mark.parametrize("offset", [0, 1, 4])
def test_round_trip(F, n, offset):
    lib, check = F._lib.load(), F._lib.check
    a = np.random.default_rng(n).integers(0, 256, n, np.uint8)
    buf = F.DeviceBuffer(n + offset + 64)
    check(lib.fhip_memset(buf.ptr, 0xA5, n + offset + 64, None))
    src = a.copy()
    check(lib.fhip_memcpy_h2d(C.c_void_p(buf.ptr.value + offset), src.ctypes.data, n, None))
    if n <= F.qmatrix.H2D_STAGED:
        src[:] = 0                                # has been read
    out = np.empty(n + offset + 64, np.uint8)
    check(lib.fhip_memcpy_d2h(out.ctypes.data, buf.ptr, out.size, None))
    assert np.array_equal(out[offset:offset + n], a)
    assert (out[:offset] == 0xA5).all() and (out[offset + n:] == 0xA5).all()


# two and three slots that the host empties by itself, and one byte more (64 + offset bytes are added to n)
@pytest.mark.parametrize("n", [MIB + 200, 2 * MIB - 64, 2 * MIB - 63, 3 * MIB - 65, 3 * MIB - 64, 3 * MIB - 63])
@pytest.mark.parametrize("offset", [0, 1, 4])
def test_copies_back_of_two_and_three_slots(F, n, offset):
    test_round_trip(F, n, offset)


# the runtime's, in two chunks, in as many as there are slots, the runtime's again; to an idle stream and behind other work
@pytest.mark.parametrize("n", [1280 * KIB, 1280 * KIB + 1, 2 * MIB, 2 * MIB + 3, 7 * MIB + 260, 12 * MIB, 12 * MIB + 1])
@pytest.mark.parametrize("offset", [0, 1, 4])
def test_uploads_have_read_their_source(F, n, offset):
    lib, check = F._lib.load(), F._lib.check
    a = np.random.default_rng(n).integers(0, 256, n, np.uint8)
    buf, other, s = F.DeviceBuffer(n + offset + 64), F.DeviceBuffer(64 * MIB), F.Stream()
    for busy in (False, True):
        check(lib.fhip_memset(buf.ptr, 0xA5, n + offset + 64, s.handle))
        if busy:
            for _ in range(4):
                check(lib.fhip_memset(other.ptr, 1, 64 * MIB, s.handle))
        else:
            s.synchronize()
        src = a.copy()
        check(lib.fhip_upload(C.c_void_p(buf.ptr.value + offset), src.ctypes.data, n, s.handle))
        src[:] = 0
        out = np.empty(n + offset + 64, np.uint8)
        check(lib.fhip_memcpy_d2h(out.ctypes.data, buf.ptr, out.size, s.handle))
        assert np.array_equal(out[offset:offset + n], a) and (out[:offset] == 0xA5).all() and (out[offset + n:] == 0xA5).all(), busy


@pytest.mark.parametrize("n", [640 * KIB + 1, MIB, MIB + 1, 7 * MIB + 260, 12 * MIB, 12 * MIB + 1])
def test_a_long_upload_may_be_used_on_another_stream(F, n):
    """From an idle stream and behind other work: it has arrived when the call returns, also where the other stream has read what was there before."""
    lib, check = F._lib.load(), F._lib.check
    buf, copy, other, s, s2 = F.DeviceBuffer(n), F.DeviceBuffer(n), F.DeviceBuffer(64 * MIB), F.Stream(), F.Stream()
    for k in range(6):
        a = np.random.default_rng(n + k).integers(0, 256, n, np.uint8)
        for _ in range(2 * (k % 3)):
            check(lib.fhip_memset(other.ptr, 1, 64 * MIB, s.handle))
        check(lib.fhip_upload(buf.ptr, a.ctypes.data, n, s.handle))
        check(lib.fhip_memcpy_d2d(copy.ptr, buf.ptr, n, s2.handle))
        out = np.empty(n, np.uint8)
        check(lib.fhip_memcpy_d2h(out.ctypes.data, (copy if k % 2 else buf).ptr, n, s2.handle))
        assert np.array_equal(out, a), k


# a destination whose pages are made while its stream is busy: in parts, two and three slots, the workers; nothing around it is written
@pytest.mark.parametrize("n", [20 * KIB, 608 * KIB, MIB + 5, 2 * MIB + 4097, 3 * MIB, 5 * MIB + 3])
@pytest.mark.parametrize("fills", [1, 40])
def test_copies_back_into_fresh_memory_behind_other_work(F, n, fills):
    import mmap
    lib, check = F._lib.load(), F._lib.check
    a = np.random.default_rng(n).integers(0, 256, n, np.uint8)
    buf, other, s = F.DeviceBuffer(n), F.DeviceBuffer(64 * MIB), F.Stream()
    check(lib.fhip_upload(buf.ptr, a.ctypes.data, n, s.handle))
    for offset in (0, 4000):
        whole = np.frombuffer(mmap.mmap(-1, n + 8192), np.uint8)
        for k in range(fills):
            check(lib.fhip_memset(other.ptr, k, 64 * MIB, s.handle))
        check(lib.fhip_memcpy_d2h(whole[offset:].ctypes.data, buf.ptr, n, s.handle))
        assert np.array_equal(whole[offset:offset + n], a) and not whole[:offset].any() and not whole[offset + n:].any()


# who empties the slots goes by whether the destination's pages are there: none of them, all, all but the first or the last
@pytest.mark.parametrize("n", [3 * MIB // 2, 3 * MIB // 2 + 1, 2 * MIB + 4097, 3 * MIB])
@pytest.mark.parametrize("touched", ["none", "all", "not the first", "not the last"])
def test_copies_back_into_fresh_memory(F, n, touched):
    import mmap
    a = np.random.default_rng(n).integers(0, 256, n, np.uint8)
    buf = F.DeviceBuffer(n)
    F._lib.check(F._lib.load().fhip_upload(buf.ptr, a.ctypes.data, n, None))
    for offset in (0, 4000):                      # (a range that does not begin with a page)
        out = np.frombuffer(mmap.mmap(-1, n + 8192), np.uint8)[offset:offset + n]
        if touched != "none":
            out[8192 if touched == "not the first" else 0:-8192 if touched == "not the last" else None] = 1
        F._lib.check(F._lib.load().fhip_memcpy_d2h(out.ctypes.data, buf.ptr, n, None))
        assert np.array_equal(out, a)


@pytest.mark.parametrize("ty,block", [(8, 32), (12, 256), (14, 256), (7, 32), (39, 32)])
@pytest.mark.parametrize("values", [32 * 8, MIB // 4 - 256, MIB // 4, MIB // 4 + 256, 2 * MIB // 4 + 256, 17 * MIB // 4 + 512])
def test_host_dequantization_in_chunks(F, O, ty, block, values):
    from ferric_amd.synth import synth_weights
    raw = synth_weights(ty, 1, values // block * block, values)
    assert np.array_equal(bits(F.deq_raw(raw, values, ty)), bits(O.deq_raw(raw, values, ty)))


def test_copies_from_several_threads_and_streams(F):
    """More small copies in flight than there are slots, and chunked ones beside them."""
    wrong = []

    def work(seed):
        rng, s = np.random.default_rng(seed), F.Stream()
        lib, check = F._lib.load(), F._lib.check
        for i in range(40):
            n = int(rng.integers(1, 600 * KIB)) if i % 10 else 5 * MIB + seed
            a = rng.integers(0, 256, n, np.uint8)
            d = F.DeviceBuffer(n)
            check(lib.fhip_memcpy_h2d(d.ptr, a.ctypes.data, n, s.handle))
            b = np.empty(n, np.uint8)
            check(lib.fhip_memcpy_d2h(b.ctypes.data, d.ptr, n, s.handle))
            if not np.array_equal(a, b):
                wrong.append((seed, i, n))

    ts = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not wrong


def test_freed_memory_is_not_handed_out_while_work_uses_it(F):
    """Long copies enqueued on one stream out of buffers that are freed at once; buffers of the same size are made and overwritten
    on another stream straight away."""
    lib, check = F._lib.load(), F._lib.check
    n, s1, s2 = 64 * MIB, F.Stream(), F.Stream()
    outs = []
    for k in range(12):
        src, dst = F.DeviceBuffer(n), F.DeviceBuffer(n)
        check(lib.fhip_memset(src.ptr, k + 1, n, s1.handle))
        for _ in range(4):
            check(lib.fhip_memcpy_d2d(dst.ptr, src.ptr, n, s1.handle))
        del src
        other = F.DeviceBuffer(n)
        check(lib.fhip_memset(other.ptr, 0xFF, n, s2.handle))
        del other
        outs.append(dst)
    s1.synchronize()
    for k, d in enumerate(outs):
        got = np.empty(n, np.uint8)
        check(lib.fhip_memcpy_d2h(got.ctypes.data, d.ptr, n, s1.handle))
        assert (got == k + 1).all(), k


def test_a_wrapped_weight_must_fit_what_was_asked_for(F):
    raw = np.zeros(144 * 3, np.uint8)
    buf = F.DeviceBuffer(raw.size)
    F.QMatrix.wrap_device(buf, raw.size, F.Q4_K, 3, 256)
    with pytest.raises(F._lib.FerricHipError, match="must extend"):
        F.QMatrix.wrap_device(buf, 144 * 4, F.Q4_K, 4, 256)
