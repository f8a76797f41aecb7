"""Device memory and host copies of the library where they have to say no: stream captures, blocks freed twice, sizes and ranges that
no allocation has; and what they do beside each other on several threads and streams."""
import ctypes as C
import gc
import time
import weakref
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
KIB, MIB = 1 << 10, 1 << 20
KEPT = 64                 # freed blocks that a small class collects before an allocation waits for the device


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
    assert other.submit(blocks_in_turn, F, 9000).result() <= KEPT
    assert blocks_in_turn(F, 9000) <= KEPT


def test_a_stream_destroyed_while_it_captures_ends_the_capture(F):
    s = F.Stream()
    F.Graph.begin(s)
    handle, s.handle = s.handle, None
    F._lib.check(F._lib.load().fhip_stream_destroy(handle))
    assert blocks_in_turn(F, 11000) <= KEPT


def _allocating_calls(F):
    """Operators that allocate (their result, most of them scratch of their own too), each as a call on a stream."""
    from ferric_amd import decode, kvquant
    from ferric_amd.synth import synth_weights
    rng = np.random.default_rng(0)
    t = lambda *shape: F.Tensor.from_vec(rng.standard_normal(shape).astype(np.float32), shape)
    w = lambda ty, rows, cols: F.QMatrix.from_bytes(synth_weights(ty, rows, cols, rows), ty, rows, cols)
    x, x40, gu, down = t(8, 512), t(40, 512), w(F.Q4_K, 1024, 512), w(F.Q6_K, 512, 512)
    slab, sel, slots = w(F.Q4_K, 4 * 256, 512), F.Tensor.from_vec(np.array([[0.5, 0.5, 1, 3]], np.float32), (1, 4)), t(1, 2, 512)
    q, cache = t(1, 512), decode.KvCache(3000, 256).append2(t(3000, 256), t(3000, 256))
    kvq = [kvquant.QKvCache(kvquant.Q8_0, 3000, 256).append(t(3000, 256)) for _ in range(2)]
    return {
        "a buffer": lambda s: F.DeviceBuffer(5000),
        "matmul_q": lambda s: x.matmul_q(gu, s),
        "matmul_q_coop": lambda s: x40.matmul_q_coop(gu, s),
        "matmul_q_f16x2": lambda s: x.matmul_q_f16x2(gu, s),
        "ffn": lambda s: x.ffn(gu, down, s),
        "ffn_f16x2": lambda s: x.ffn_f16x2(gu, down, s),
        "ffn_coop": lambda s: x40.ffn_coop(gu, down, s),
        "matmul_q_id_wsum": lambda s: slots.matmul_q_id_wsum(slab, sel, 256, s),
        "rope": lambda s: decode.rope(q, 4, 128, 1e6, positions=[7], stream=s),
        "decode_attention": lambda s: decode.decode_attention(q, cache, 4, 2, stream=s),
        "decode_attention_kvq": lambda s: decode.decode_attention_kvq(q, *kvq, 4, 2, stream=s),
    }


@pytest.fixture(scope="module")
def allocating_calls(F):
    return _allocating_calls(F)


@pytest.mark.parametrize("name", ["a buffer", "matmul_q", "matmul_q_coop", "matmul_q_f16x2", "ffn", "ffn_f16x2", "ffn_coop", "matmul_q_id_wsum", "rope", "decode_attention",
                                  "decode_attention_kvq"])
def test_nothing_is_allocated_inside_a_capture(F, allocating_calls, name):
    """The graph would use the scratch again after the pool has given it to somebody else. The calls have run before, so that the pool
    holds blocks for all of it; the capture goes on after the refusal."""
    s, call = F.Stream(), allocating_calls[name]
    word = F.Tensor.from_vec(np.zeros(4, np.float32), (4,))
    for _ in range(2):
        call(s)
        blocks_in_turn(F, 13000)                 # has waited for the device: what the call freed can be handed out
    g = F.Graph.begin(s)
    with pytest.raises(F._lib.FerricHipError, match="captures a stream"):
        call(s)
    F._lib.check(F._lib.load().fhip_u32_add(word.buf.ptr, 1, 1, s.handle))
    g.end()
    for _ in range(3):
        g.launch()
        s.synchronize()
    assert word.to_vec(s).view(np.uint32)[0] == 3
    call(s)


def test_nothing_is_allocated_inside_a_capture_through_the_runtime(F):
    """hipMalloc refuses such a thread, and so does the pool, though it holds blocks of the size."""
    hip = C.CDLL("libamdhip64.so.7")
    s, graph = F.Stream(), C.c_void_p()
    blocks_in_turn(F, 15000)
    assert hip.hipStreamBeginCapture(s.handle, 1) == 0
    with pytest.raises(F._lib.FerricHipError):
        F.DeviceBuffer(15000)
    assert hip.hipStreamEndCapture(s.handle, C.byref(graph)) != 0       # the runtime invalidates what it refuses
    hip.hipGetLastError()                                               # (or the next launch would report it)
    F.DeviceBuffer(15000)


def test_cached_memory_and_copies_leave_a_global_capture_of_another_thread_alone(F):
    """The runtime invalidates such a capture when any thread calls hipMalloc; a block that the pool holds already needs no such call."""
    hip, s, graph = C.CDLL("libamdhip64.so.7"), F.Stream(), C.c_void_p()
    t = F.Tensor.from_vec(np.arange(5000, dtype=np.float32), (5000,))
    t.to_vec()
    blocks_in_turn(F, 19000)                     # the last wait was a few blocks ago: some are clean
    with ThreadPoolExecutor(1) as other:
        assert other.submit(hip.hipStreamBeginCapture, s.handle, 0).result() == 0
        F.DeviceBuffer(19000)
        assert np.array_equal(t.to_vec(), np.arange(5000, dtype=np.float32))
        assert other.submit(hip.hipStreamEndCapture, s.handle, C.byref(graph)).result() == 0
    hip.hipGraphDestroy(graph)


def test_other_threads_allocate_and_copy_while_one_captures(F):
    """Their waits for the device must leave the capture alone (hipDeviceSynchronize would fail and invalidate it)."""
    lib, check = F._lib.load(), F._lib.check
    s, word = F.Stream(), F.Tensor.from_vec(np.zeros(4, np.float32), (4,))
    g = F.Graph.begin(s)
    check(lib.fhip_u32_add(word.buf.ptr, 1, 1, s.handle))
    with ThreadPoolExecutor(1) as other:
        assert other.submit(blocks_in_turn, F, 17000).result() <= KEPT
        a = np.arange(3 * MIB, dtype=np.float32)
        assert np.array_equal(other.submit(lambda: F.Tensor.from_vec(a, a.shape).to_vec()).result(), a)
    check(lib.fhip_u32_add(word.buf.ptr, 1, 1, s.handle))
    g.end()
    for _ in range(3):
        g.launch()
        s.synchronize()
    assert word.to_vec(s).view(np.uint32)[0] == 6


def _small_decoder(F, stream):
    from ferric_amd import decode
    from ferric_amd.synth import synth_weights
    d, heads, kv, hd, ff = 512, 4, 2, 64, 1024
    rng = np.random.default_rng(1)
    w = lambda ty, rows, cols, seed: F.QMatrix.from_bytes(synth_weights(ty, rows, cols, seed), ty, rows, cols)
    n = lambda k: F.Tensor.from_vec(rng.uniform(0.5, 1.5, k).astype(np.float32), (k,))
    layer = decode.Qwen3Layer(n(d), w(F.Q4_K, (heads + 2 * kv) * hd, d, 1), w(F.Q8_0, d, heads * hd, 2), n(d), w(F.Q4_K, 2 * ff, d, 3), w(F.Q6_K, d, ff, 4), n(hd), n(hd))
    return decode.Qwen3Decoder(decode.Qwen3Cfg(d, heads, kv, hd, ff), [layer], max_len=64, stream=stream)


def test_host_copies_are_refused_inside_a_capture(F):
    """Reading back, setting a decoder's input or position, dequantizing to the host: on the captured stream and on others. The capture goes on, and so
    does what the refused calls would have set."""
    s, elsewhere = F.Stream(), F.Stream()
    dec = _small_decoder(F, s)
    x = np.random.default_rng(2).standard_normal((3, 512)).astype(np.float32)
    dec.set_pos(0)
    dec.set_input(x[0])
    dec.step()
    want, before = dec.hidden(), [c.len for c in dec.caches]
    t, big, raw = F.Tensor.from_vec(x, x.shape), np.zeros(1 << 20, np.float32), np.zeros(34 * 64, np.uint8)
    room = F.Tensor.empty(big.shape)
    assert F.deq_raw(raw, 32 * 64, F.Q8_0).size == 32 * 64
    dec.set_pos(0)
    g = F.Graph.begin(s)
    dec._enqueue_step()
    refused = [lambda: t.to_vec(s), lambda: t.to_vec(elsewhere), lambda: t.to_vec(), lambda: dec.hidden(), lambda: dec.set_pos(7), lambda: dec.set_input(x[1]),
               lambda: F.qmatrix._upload(room.buf, big, s), lambda: F.qmatrix._upload(room.buf, big, elsewhere), lambda: F.deq_raw(raw, 32 * 64, F.Q8_0),
               lambda: dec.prefill(x)]
    for call in refused:
        with pytest.raises(F._lib.FerricHipError, match="captur"):
            call()
    g.end()
    assert [c.len for c in dec.caches] == [0] != before
    for _ in range(3):
        dec.set_pos(0)
        dec.set_input(x[0])
        g.launch()
        assert np.array_equal(dec.hidden(), want)
    assert np.array_equal(t.to_vec(), x.reshape(-1))


def test_a_recorded_upload_reads_its_source_at_every_replay(F):
    lib, check = F._lib.load(), F._lib.check
    s, t, src = F.Stream(), F.Tensor.empty((1000,)), np.zeros(1000, np.float32)
    g = F.Graph.begin(s)
    check(lib.fhip_memcpy_h2d(t.buf.ptr, src.ctypes.data, src.nbytes, s.handle))
    g.end()
    for k in range(3):
        src[:] = k + 1
        g.launch()
        assert (t.to_vec(s) == k + 1).all()


def test_an_upload_has_read_its_source_whatever_its_size(F):
    lib, check, s = F._lib.load(), F._lib.check, F.Stream()
    for n in (1, 640 * KIB, 640 * KIB + 4, 40 * MIB):
        want = np.random.default_rng(n).integers(0, 256, n, np.uint8)
        d, src, got = F.DeviceBuffer(n), want.copy(), np.empty(n, np.uint8)
        check(lib.fhip_upload(d.ptr, src.ctypes.data, n, s.handle))
        src[:] = 0
        check(lib.fhip_memcpy_d2h(got.ctypes.data, d.ptr, n, s.handle))
        assert np.array_equal(got, want)


# ---- copies of what the library does not own -------------------------------------------------------------------------------------------

def test_copies_outside_the_librarys_blocks_go_to_the_runtime(F):
    """Device memory of somebody else's, device memory in the host's place, more bytes than a block has: copied by the runtime, which looks its
    pointers up, or refused, and never reached by a kernel that does not look."""
    lib, hip, s = F._lib.load(), C.CDLL("libamdhip64.so.7"), F.Stream()
    rng = np.random.default_rng(5)
    for n in (7, 100 * KIB, 640 * KIB, 3 * MIB):
        a, got = rng.integers(0, 256, n, np.uint8), np.zeros(n, np.uint8)
        foreign, own = C.c_void_p(), F.DeviceBuffer(n)
        assert hip.hipMalloc(C.byref(foreign), C.c_size_t(n)) == 0
        src = a.copy()
        F._lib.check(lib.fhip_upload(foreign, src.ctypes.data, n, s.handle))
        src[:] = 0
        F._lib.check(lib.fhip_memcpy_d2h(got.ctypes.data, foreign, n, s.handle))
        assert np.array_equal(got, a)
        F._lib.check(lib.fhip_upload(own.ptr, foreign, n, s.handle))               # device memory as the source
        got[:] = 0
        F._lib.check(lib.fhip_memcpy_d2h(got.ctypes.data, own.ptr, n, s.handle))
        assert np.array_equal(got, a)
        for name, call in (("to", lambda d, m: lib.fhip_memcpy_h2d(d, (C.c_char * m)(), m, s.handle)), ("from", lambda d, m: lib.fhip_memcpy_d2h((C.c_char * m)(), d, m, s.handle))):
            for at, m in ((0, n + 257), (n, 257), (0, n + 64 * MIB)):                 # past what was asked for, and its slack
                assert call(C.c_void_p(own.ptr.value + at), m) == F._lib.ERR_HIP, (name, at, m)
        assert hip.hipFree(foreign) == 0


@pytest.mark.parametrize("values", [32 * 40, 5 << 18])
def test_host_dequantization_takes_device_memory_on_either_side(F, values):
    from ferric_amd.synth import synth_weights
    lib, raw = F._lib.load(), synth_weights(F.Q8_0, 1, values, 8)
    want, t, got = F.deq_raw(raw, values, F.Q8_0), F.Tensor.empty((values,)), C.c_size_t()
    d = F.DeviceBuffer(raw.size)
    F._lib.check(lib.fhip_upload(d.ptr, raw.ctypes.data, raw.size, None))
    F._lib.check(lib.fhip_stream_sync(None))
    F._lib.check(lib.fhip_deq_raw(d.ptr, raw.size, values, F.Q8_0, t.buf.ptr, C.byref(got)))
    assert got.value == values and np.array_equal(t.to_vec(), want)


# ---- copies beside each other ------------------------------------------------------------------------------------------------------------

class Work:
    """Something for a stream to do for about the given time, in launches of some milliseconds that leave room on every CU."""

    def __init__(self, F):
        self.lib, self.check, self.sink, self.iters = F._lib.load(), F._lib.check, F.DeviceBuffer(64), 20000
        self.s = F.Stream()
        self.launch(self.s)
        self.s.synchronize()
        start = time.perf_counter()
        self.launch(self.s)
        self.s.synchronize()
        self.each = time.perf_counter() - start

    def launch(self, s):
        self.check(self.lib.fhip_debug_mfma_probe(self.iters, self.sink.ptr, None, s.handle))

    def enqueue(self, s, seconds):
        for _ in range(max(1, int(seconds / self.each))):
            self.launch(s)


@pytest.fixture(scope="module")
def work(F):
    return Work(F)


def _read(F, t, s):
    return F.Tensor.to_vec(t, s)


def test_a_long_readback_behind_work_holds_nobody_up(F, work):
    """2 MB behind half a second of work on one stream; 5 MB on an idle one and a dequantization in chunks come back meanwhile, and the wait costs one
    core at most."""
    busy, idle = F.Stream(), F.Stream()
    a = np.random.default_rng(3).standard_normal(5 << 18).astype(np.float32)
    t, raw = F.Tensor.from_vec(a, a.shape), np.zeros(34 << 16, np.uint8)
    small = F.Tensor.from_vec(a[:1 << 19], (1 << 19,))
    _read(F, t, idle), F.deq_raw(raw, 32 << 16, F.Q8_0)          # the slots and the workers are there
    with ThreadPoolExecutor(1) as other:
        work.enqueue(busy, 0.5)
        wall, cpu = time.perf_counter(), time.process_time()
        waiting = other.submit(_read, F, small, busy)
        time.sleep(0.02)
        assert np.array_equal(_read(F, t, idle), a) and not F.deq_raw(raw, 32 << 16, F.Q8_0).any()
        assert not waiting.done()
        assert np.array_equal(waiting.result(), a[:1 << 19])
        wall, cpu = time.perf_counter() - wall, time.process_time() - cpu
    assert wall > 0.2 and cpu < 2 * wall, (wall, cpu)


def test_many_readbacks_behind_work_leave_the_others_their_way(F, work):
    """More of them than there are pinned slots, behind half a second of work; copies in both directions of other streams come back meanwhile."""
    from ferric_amd.synth import synth_weights
    busy, idle = F.Stream(), F.Stream()
    a = np.random.default_rng(4).standard_normal(60000).astype(np.float32)
    t, long = F.Tensor.from_vec(a, a.shape), F.Tensor.from_vec(np.tile(a, 20), (1200000,))
    raw = synth_weights(F.Q8_0, 1, 32 << 16, 6)
    dense = F.deq_raw(raw, 32 << 16, F.Q8_0)
    with ThreadPoolExecutor(20) as other:
        work.enqueue(busy, 0.5)
        waiting = [other.submit(_read, F, t, busy) for _ in range(20)]
        time.sleep(0.02)
        assert np.array_equal(_read(F, t, idle), a) and np.array_equal(_read(F, long, idle)[-60000:], a)
        F.qmatrix._upload(t.buf, a, idle)
        assert np.array_equal(F.deq_raw(raw, 32 << 16, F.Q8_0), dense) and np.array_equal(F.deq_raw(raw[:3400], 3200, F.Q8_0), dense[:3200])
        assert not any(w.done() for w in waiting)
        assert all(np.array_equal(w.result(), a) for w in waiting)


# ---- the Python object ---------------------------------------------------------------------------------------------------------------------

def test_a_device_buffer_takes_attributes_and_weak_references(F):
    b = F.DeviceBuffer(100)
    b.owner, gone = "me", []
    ref = weakref.ref(b, gone.append)
    assert b.owner == "me" and vars(b) == {"owner": "me"} and ref() is b and b.nbytes == 100
    del b.owner
    with pytest.raises(AttributeError):
        b.owner
    assert weakref.WeakValueDictionary({1: b})[1] is b
    del b
    assert ref() is None and gone == [ref]

    class Mine(F.DeviceBuffer):
        pass
    cycle = [F.DeviceBuffer(100), Mine(100)]
    refs = [weakref.ref(c) for c in cycle]
    cycle[0].other, cycle[1].other = cycle[1], cycle[0]
    del cycle
    gc.collect()
    assert [r() for r in refs] == [None, None]


def test_matmul_q_takes_any_buffer_and_stream_with_an_address(F):
    """Objects that are not the library's own: a `ptr` and a `handle`, as ctypes pointers or as numbers, as the other operators take them."""
    from ferric_amd.synth import synth_weights

    class Address:
        def __init__(self, **kw):
            self.__dict__.update(kw)
    w = F.QMatrix.from_bytes(synth_weights(F.Q4_K, 256, 512, 3), F.Q4_K, 256, 512)
    x, s = F.Tensor.from_vec(np.random.default_rng(0).standard_normal((3, 512)).astype(np.float32), (3, 512)), F.Stream()
    want = x.matmul_q(w).to_vec()
    for ptr in (x.buf.ptr, x.buf.ptr.value):
        for handle in (s.handle, s.handle.value):
            other = F.Tensor(Address(ptr=ptr, nbytes=x.buf.nbytes), x.shape)
            for t in (other, x):
                assert np.array_equal(t.matmul_q(w, Address(handle=handle)).to_vec(s), want)
        assert np.array_equal(other.matmul_q(w).to_vec(), want)
    with pytest.raises(AttributeError):
        F.Tensor(Address(), x.shape).matmul_q(w)
