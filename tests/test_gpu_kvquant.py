"""The block-quantized KV cache through the C ABI against the oracle (oracle/kvquant_oracle.py): codes, scale bits and
dequantized values are integer / single-rounding work and must be bit-identical. Mirrors the reference's own tests of this
module (crates/ferric-tensor/src/kvquant.rs:1620-2130)."""
import ctypes as C

import numpy as np
import pytest

from conftest import bits
from test_oracle_kvquant import exact_case

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K():
    from oracle import kvquant_oracle
    return kvquant_oracle


@pytest.fixture(scope="module")
def Q(F):
    from ferric_amd import kvquant
    return kvquant


def packed(Q, K, cache):
    """(codes [nblk, words], scale halves) of the live rows, in the oracle's shapes."""
    c, s = cache.to_host()
    nblk = cache.len * cache.nblk_per_row()
    h = s.view(np.uint16)
    return c.reshape(nblk, K.CODE_WORDS[cache.fmt]), (h.reshape(nblk, 2) if cache.fmt == K.Q4_1 else h[:nblk])


def same_as_oracle(Q, K, cache, x):
    want = K.quantize(x, x.shape[0], x.shape[1], cache.fmt)
    c, s = packed(Q, K, cache)
    assert np.array_equal(c, want.codes), "codes"
    assert np.array_equal(s, want.scales), "scales"
    got = cache.dequantize().to_vec().reshape(x.shape)
    assert np.array_equal(bits(got), bits(want.dequantize_rows(0, x.shape[0]))), "dequantized values"


@pytest.mark.parametrize("fmt", [0, 1, 2])
def test_codes_fixed_by_construction_and_ties(F, Q, K, fmt):
    # kvquant.rs:1620 gpu_quantize_matches_the_exact_codes; :1559 ties away from zero
    x, want = exact_case(7, 96, fmt, 7)
    cache = Q.QKvCache.from_tensor(F.Tensor.from_vec(x, x.shape), fmt)
    ref = K.Cache(fmt, 7, 96)
    ref.codes, ref.scales = packed(Q, K, cache)
    for b in range(21):
        assert np.array_equal(K.codes_of(ref, b), want[b]), b
    assert np.array_equal(cache.dequantize().to_vec().reshape(7, 96), x)          # exactly representable data comes back exactly
    if fmt == K.Q8_0:
        t = np.zeros((1, 32), np.float32)
        t[0, 0] = 127.0
        t[0, 1:7] = [0.5, 1.5, 2.5, -0.5, -1.5, -2.5]
        cache = Q.QKvCache.from_tensor(F.Tensor.from_vec(t, t.shape), fmt)
        ref = K.Cache(fmt, 1, 32)
        ref.codes, ref.scales = packed(Q, K, cache)
        assert list(K.codes_of(ref, 0)[1:7]) == [1, 2, 3, -1, -2, -3]


@pytest.mark.parametrize("fmt", [0, 1, 2])
def test_heavy_tailed_and_special_values_bit_for_bit(F, Q, K, fmt):
    # kvquant.rs:1821 gpu_quantize_matches_the_cpu_reference_on_heavy_tailed_data, :1689 dequantize bit for bit
    rng = np.random.default_rng(40 + fmt)
    rows, width = 53, 160                                    # five blocks a row: scale pairs straddle rows
    x = (rng.standard_t(2, (rows, width)) * 10.0 ** rng.integers(-4, 4, (rows, 1))).astype(np.float32)
    x[3, 32:64] = 0.0                                        # d = 0
    x[4, 0:32] = -0.0
    x[5, 64:96] = 2.5                                        # a constant block (Q4_1: d = 0, min = 2.5)
    x[6, 7] = x[6, 20] = -np.abs(x[6, :32]).max() * 2        # equal extremes: the first wins
    x[7, 0:32] *= 1e-7                                       # scales in f16's subnormal range
    x[8, 0:32] *= 1e-10                                      # ... and below it: the scale rounds to zero
    x[9, 96:128] *= 1e7                                      # a scale beyond f16: infinity
    x[10, 3] = np.nan
    x[11, 40] = np.inf
    x[12, 70] = -np.inf
    x[13, 128:160] = np.nan
    x[14, 0:32] = np.float32(1e-42)                          # f32 subnormals
    cache = Q.QKvCache.from_tensor(F.Tensor.from_vec(x, x.shape), fmt)
    with np.errstate(all="ignore"):
        same_as_oracle(Q, K, cache, x)
    assert cache.len == rows and cache.width == width and cache.cap == 64


@pytest.mark.parametrize("fmt", [0, 1, 2])
def test_appends_growth_windows_and_copies(F, Q, K, fmt):
    rng = np.random.default_rng(50 + fmt)
    rows, width = 150, 96
    x = (rng.standard_normal((rows, width)) * 3).astype(np.float32)
    one_shot = Q.QKvCache.from_tensor(F.Tensor.from_vec(x, x.shape), fmt)
    same_as_oracle(Q, K, one_shot, x)
    # one row at a time (kvquant.rs:1908), through two doublings of the capacity (:2052): every earlier row survives
    grown = Q.QKvCache(fmt)
    for r in range(rows):
        grown.append(F.Tensor.from_vec(x[r:r + 1], (1, width)))
    assert grown.cap == 256 and grown.len == rows
    same_as_oracle(Q, K, grown, x)
    # rows in uneven batches, read as a window of wider rows (the key span of a fused qkv row, :2083)
    wide = rng.standard_normal((rows, 40 + width + 24)).astype(np.float32)
    wide[:, 40:40 + width] = x
    wt = F.Tensor.from_vec(wide, wide.shape)
    win = Q.QKvCache(fmt)
    at = 0
    for n in (1, 2, 60, 3, 84):
        part = F.Tensor.from_vec(wide[at:at + n], (n, wide.shape[1]))
        win.append(part, cols=(40, width))
        at += n
    same_as_oracle(Q, K, win, x)
    assert np.array_equal(bits(one_shot.dequantize_rows(17, 9).to_vec()), bits(K.quantize(x, rows, width, fmt).dequantize_rows(17, 9).reshape(-1)))
    # clone_prefix (:1861) and deep_clone (:2008): exactly those rows, and no shared memory
    pre = one_shot.clone_prefix(70)
    assert pre.len == 70 and pre.cap == 70 and pre.width == width
    same_as_oracle(Q, K, pre, x[:70])
    twin = one_shot.deep_clone()
    extra = (rng.standard_normal((5, width)) * 9).astype(np.float32)
    pre.append(F.Tensor.from_vec(extra, extra.shape))
    twin.append(F.Tensor.from_vec(-extra, extra.shape))
    same_as_oracle(Q, K, one_shot, x)                                      # untouched by either
    same_as_oracle(Q, K, pre, np.concatenate([x[:70], extra]))
    same_as_oracle(Q, K, twin, np.concatenate([x, -extra]))
    assert Q.QKvCache(fmt).clone_prefix(3).len == 0 and one_shot.clone_prefix(0).width == 0
    # what it costs (:2110): the advertised bits per value, up to the one shared scale word
    full = Q.QKvCache.from_tensor(F.Tensor.from_vec(x[:64], (64, width)), fmt)
    assert full.bytes() == full.live_bytes() == 64 * 3 * Q.BLOCK_BYTES[fmt] and full.f32_bytes() == 64 * width * 4
    assert Q.bits_per_value(fmt) == {0: 8.5, 1: 4.5, 2: 5.0}[fmt]


def test_positions_on_the_device_and_argument_checks(F, Q, K):
    """What a captured decode step uses: the row index read from a device word on both sides, the source row at that index of a
    full-length f32 staging cache, and a dequantize sized for the capacity that stops at the newest row."""
    lib = F._lib.load()
    rng = np.random.default_rng(60)
    cap, width, fmt = 12, 64, 0
    staging = (rng.standard_normal((cap, width)) * 2).astype(np.float32)
    st = F.Tensor.from_vec(staging, staging.shape)
    cache = Q.QKvCache(fmt, cap, width)
    pos = F.Tensor(F.DeviceBuffer(4), (1,), np.uint32)
    ref = K.Cache(fmt, cap, width)
    out = F.Tensor.from_vec(np.full((cap, width), 777.0, np.float32), (cap, width))
    for p in (0, 1, 2, 7):
        word = np.array([p], np.uint32)
        F._lib.check(lib.fhip_memcpy_h2d(pos.buf.ptr, word.ctypes.data, 4, None))
        F._lib.check(lib.fhip_kvq_append(fmt, st.buf.ptr, width, 1, width, pos.buf.ptr, 0, 1, cap, cache.codes.ptr, cache.scales.ptr, None))
        ref.quantize_into(staging[p], p)
        F._lib.check(lib.fhip_kvq_dequantize_rows(fmt, cache.codes.ptr, cache.scales.ptr, 0, cap, width, pos.buf.ptr, out.buf.ptr, None))
        got = out.to_vec().reshape(cap, width)
        assert np.array_equal(bits(got[p]), bits(ref.dequantize_rows(p, 1)[0])), p
        assert (got[p + 1:] == 777.0).all(), p                                  # rows past the position are not written
    # a position beyond the capacity is dropped, as fhip_kv_append2 drops it
    word = np.array([cap + 3], np.uint32)
    F._lib.check(lib.fhip_memcpy_h2d(pos.buf.ptr, word.ctypes.data, 4, None))
    before = cache.codes
    F._lib.check(lib.fhip_kvq_append(fmt, st.buf.ptr, width, 1, width, pos.buf.ptr, 0, 0, cap, cache.codes.ptr, cache.scales.ptr, None))
    F._lib.check(lib.fhip_stream_sync(None))
    # errors: the reference's width assert (kvquant.rs:470), unknown formats, rows past the capacity, NULL pointers
    assert lib.fhip_kvq_append(fmt, st.buf.ptr, 0, 1, 48, None, 0, 0, cap, cache.codes.ptr, cache.scales.ptr, None) != 0
    assert b"must be a multiple of 32" in lib.fhip_last_error()
    assert lib.fhip_kvq_append(9, st.buf.ptr, 0, 1, 64, None, 0, 0, cap, cache.codes.ptr, cache.scales.ptr, None) != 0
    assert lib.fhip_kvq_append(fmt, st.buf.ptr, 0, 5, 64, None, 10, 0, cap, cache.codes.ptr, cache.scales.ptr, None) != 0
    assert b"exceed the capacity" in lib.fhip_last_error()
    assert lib.fhip_kvq_append(fmt, None, 0, 1, 64, None, 0, 0, cap, cache.codes.ptr, cache.scales.ptr, None) != 0
    assert lib.fhip_kvq_dequantize_rows(fmt, cache.codes.ptr, cache.scales.ptr, 0, 1, 64, None, None, None) != 0
    assert lib.fhip_kvq_append(fmt, None, 0, 0, 64, None, 0, 0, cap, None, None, None) == 0              # nothing to do
    cw, sw = C.c_size_t(), C.c_size_t()
    for f in (0, 1, 2):
        assert lib.fhip_kvq_sizes(f, 7, 96, C.byref(cw), C.byref(sw)) == 0 and (cw.value, sw.value) == K.sizes(7, 96, f)
    with pytest.raises(AssertionError, match="past len"):
        cache.dequantize_rows(0, 1)


@pytest.mark.parametrize("fmt", [0, 1, 2])
def test_attention_over_the_blocks_is_attention_over_the_dequantized_rows(F, Q, K, fmt):
    """fhip_decode_attention_kvq dequantizes rows in registers by the dequantize kernel's own operations, so its output has the
    bits of fhip_decode_attention_ex over dequantize(); and it is the oracle's attention over the oracle's dequantized rows to the
    f32 attention's tolerance (1e-5 of the largest output)."""
    from types import SimpleNamespace
    from ferric_amd import decode as X
    from oracle import decode_oracle as D
    rng = np.random.default_rng(70 + fmt)
    # (heads, kv heads, head dim, rows, window, softcap): one split and many, both head sizes, every group size class, a
    # length that leaves the last split ragged, a window, a softcap
    cases = [(8, 2, 128, 7, 0, 0.0), (40, 8, 128, 300, 0, 0.0), (8, 8, 64, 129, 0, 0.0), (6, 2, 64, 1000, 0, 0.0), (16, 2, 128, 2100, 512, 0.0),
             (5, 1, 128, 260, 0, 30.0), (14, 2, 64, 33, 8, 50.0)]
    for nh, nkv, hd, rows, window, cap in cases:
        width = nkv * hd
        k = (rng.standard_normal((rows, width)) * 2).astype(np.float32)
        v = (rng.standard_t(3, (rows, width))).astype(np.float32)
        q = rng.standard_normal((1, nh * hd)).astype(np.float32)
        kq = Q.QKvCache.from_tensor(F.Tensor.from_vec(k, k.shape), fmt)
        vq = Q.QKvCache.from_tensor(F.Tensor.from_vec(v, v.shape), fmt)
        qt = F.Tensor.from_vec(q, q.shape)
        got = X.decode_attention_kvq(qt, kq, vq, nh, nkv, window=window, softcap=cap).to_vec()
        plain = SimpleNamespace(k=kq.dequantize(), v=vq.dequantize(), cap=rows, width=width, len=rows)
        same = X.decode_attention(qt, plain, nh, nkv, window=window, softcap=cap).to_vec()
        assert np.array_equal(bits(got), bits(same)), (nh, nkv, hd, rows)
        want = D.decode_attention(q[0], K.roundtrip(k, rows, width, fmt), K.roundtrip(v, rows, width, fmt), nh, nkv, window, cap)
        assert np.abs(got - want.reshape(-1)).max() <= 1e-5 * np.abs(want).max(), (nh, nkv, hd, rows)
        # a shorter length, and the length read from a device word (what a captured step does)
        n = max(1, rows // 3)
        word = F.Tensor(F.DeviceBuffer(4), (1,), np.uint32)
        last = np.array([n - 1], np.uint32)
        F._lib.check(F._lib.load().fhip_memcpy_h2d(word.buf.ptr, last.ctypes.data, 4, None))
        a = X.decode_attention_kvq(qt, kq, vq, nh, nkv, length=n, window=window, softcap=cap).to_vec()
        b = X.decode_attention_kvq(qt, kq, vq, nh, nkv, length=rows, last_pos=word, window=window, softcap=cap).to_vec()
        want = D.decode_attention(q[0], K.roundtrip(k[:n], n, width, fmt), K.roundtrip(v[:n], n, width, fmt), nh, nkv, window, cap).reshape(-1)
        assert np.abs(a - want).max() <= 1e-5 * np.abs(want).max() and np.abs(b - want).max() <= 1e-5 * np.abs(want).max()
    lib = F._lib.load()
    assert lib.fhip_decode_attention_kvq(fmt, qt.buf.ptr, kq.codes.ptr, kq.scales.ptr, vq.codes.ptr, vq.scales.ptr, 14, 2, 48, 5, None, 0, 0.0, None,
                                         qt.buf.ptr, None) != 0                      # 2 x 48 is a multiple of 32, the head size is not one the kernel takes
    assert b"head_dim must be 64 or 128" in lib.fhip_last_error()


@pytest.mark.parametrize("nh,nkv,hd,rows", [(32, 32, 128, 192), (32, 32, 128, 193), (8, 8, 128, 352), (32, 32, 128, 353), (2, 2, 128, 256), (40, 40, 64, 352), (40, 40, 64, 353),
                                           (40, 8, 128, 256), (40, 8, 128, 257), (16, 2, 128, 352), (16, 2, 128, 353), (2, 1, 128, 300), (24, 8, 64, 352), (24, 8, 64, 353)])
def test_about_the_end_of_the_short_caches(F, Q, K, nh, nkv, hd, rows):
    """One workgroup a head, or splits: heads of 128 dims from 257 rows on, from 193 with a KV head each; f32 and Q8_0 caches at the 1e-5 of the attention tests,
    the same bits from both; a launch without a workspace is taken up to 352 rows, as the one workgroup needs none."""
    from types import SimpleNamespace
    from ferric_amd import decode as X
    from oracle import decode_oracle as D
    lib, rng, width = F._lib.load(), np.random.default_rng(rows + nh), nkv * hd
    k, v = (rng.standard_normal((rows, width)).astype(np.float32) for _ in range(2))
    q = rng.standard_normal((1, nh * hd)).astype(np.float32)
    kq, vq = (Q.QKvCache.from_tensor(F.Tensor.from_vec(a, a.shape), Q.Q8_0) for a in (k, v))
    qt = F.Tensor.from_vec(q, q.shape)
    plain = SimpleNamespace(k=kq.dequantize(), v=vq.dequantize(), cap=rows, width=width, len=rows)
    want = D.decode_attention(q[0], K.roundtrip(k, rows, width, Q.Q8_0), K.roundtrip(v, rows, width, Q.Q8_0), nh, nkv)[0]
    a, b = X.decode_attention_kvq(qt, kq, vq, nh, nkv).to_vec(), X.decode_attention(qt, plain, nh, nkv).to_vec()
    assert np.array_equal(bits(a), bits(b)) and np.abs(b - want).max() <= 1e-5 * np.abs(want).max()
    out = F.Tensor.empty((1, nh * hd))
    rc = lib.fhip_decode_attention_ex(qt.buf.ptr, plain.k.buf.ptr, plain.v.buf.ptr, nh, nkv, hd, rows, None, 0, 0.0, None, out.buf.ptr, None)
    assert (rc == 0) == (rows <= 352)
    if rc == 0:
        assert np.abs(out.to_vec() - want).max() <= 1e-5 * np.abs(want).max()
    assert (lib.fhip_decode_attention_ws_bytes(nh, nkv, hd, rows) > 0) == (rows > (352 if hd == 64 else 192 if nh == nkv else 256))


@pytest.mark.parametrize("fmt", [0, 1])
@pytest.mark.parametrize("nh,nkv,hd,rows,lengths", [
    (5, 1, 64, 5121, (5121, 97, 1)),              # the smallest group and cache that take the kernel; splits of a few keys, of one, of none
    (16, 2, 64, 6150, (6150, 5000)), (10, 2, 64, 5200, (5200,)), (6, 1, 128, 5121, (5121, 33)), (8, 1, 128, 7000, (7000, 6999)),
    (7, 1, 128, 16384, (16384, 9001))])
def test_attention_over_long_caches_on_the_matrix_cores(F, Q, K, fmt, nh, nkv, hd, rows, lengths):
    """Group sizes and lengths at the edges of the long-cache kernel's rounds (32 keys a wave, eight waves, 41 to 128 splits), with the
    length on the device, a window and a softcap, against the oracle over the oracle's dequantized rows: the f32 attention's 1e-5
    of the largest output. Large scores (a query of magnitude 4) sharpen the softmax, where an error in a score would show."""
    from ferric_amd import decode as X
    from oracle import decode_oracle as D
    rng = np.random.default_rng(90 + fmt)
    width = nkv * hd
    k = (rng.standard_normal((rows, width)) + 0.5).astype(np.float32)
    v = rng.standard_t(3, (rows, width)).astype(np.float32)
    q = (rng.standard_normal((1, nh * hd)) * np.where(np.arange(nh * hd) < hd, 4.0, 1.0)).astype(np.float32)
    kq, vq = (Q.QKvCache.from_tensor(F.Tensor.from_vec(x, x.shape), fmt) for x in (k, v))
    kr, vr = K.roundtrip(k, rows, width, fmt), K.roundtrip(v, rows, width, fmt)
    qt = F.Tensor.from_vec(q, q.shape)
    word = F.Tensor(F.DeviceBuffer(4), (1,), np.uint32)
    for n in lengths:
        last = np.array([n - 1], np.uint32)
        F._lib.check(F._lib.load().fhip_memcpy_h2d(word.buf.ptr, last.ctypes.data, 4, None))
        for window, cap in ((0, 0.0), (301, 20.0)):
            got = X.decode_attention_kvq(qt, kq, vq, nh, nkv, length=rows, last_pos=word, window=window, softcap=cap).to_vec()
            want = D.decode_attention(q[0], kr[:n], vr[:n], nh, nkv, window, cap).reshape(-1)
            assert np.abs(got - want).max() <= 1e-5 * np.abs(want).max(), (n, window)


@pytest.mark.parametrize("fmt", [0, 1])
@pytest.mark.parametrize("nh,nkv,hd,rows,lengths", [
    (3, 1, 64, 5121, (5121, 257)), (4, 1, 128, 5377, (5377, 256)), (10, 2, 128, 9001, (9001, 33)), (15, 3, 64, 7001, (7001,)), (21, 3, 128, 5200, (5200,))])
def test_long_caches_by_cut_columns_and_by_query_columns(F, Q, K, fmt, nh, nkv, hd, rows, lengths):
    """Three to five query heads a KV head (a column holds one cut of a query's products) and seven, at the edges of eight waves' rounds."""
    test_attention_over_long_caches_on_the_matrix_cores(F, Q, K, fmt, nh, nkv, hd, rows, lengths)


@pytest.mark.parametrize("nh,nkv,hd,rows,lengths", [
    (5, 1, 64, 5121, (5121, 97, 1)), (16, 2, 64, 6150, (6150, 5000)), (8, 1, 128, 7000, (7000, 6999)), (10, 2, 128, 9001, (9001, 33)), (21, 3, 128, 5200, (5200,)), (3, 1, 64, 5121, (257,))])
def test_long_caches_of_blocks_with_a_minimum(F, Q, K, nh, nkv, hd, rows, lengths):
    """Q4_1 on the long-cache kernel, at the same edges and the same bar: rows off zero, where a block's minimum carries most of its values, and about it."""
    test_attention_over_long_caches_on_the_matrix_cores(F, Q, K, 2, nh, nkv, hd, rows, lengths)


@pytest.mark.parametrize("fmt", [0, 1])
@pytest.mark.parametrize("nkv,g,n", [(171, 3, 700), (300, 3, 511), (511, 3, 290), (171, 6, 257), (171, 8, 31)])
def test_long_caches_of_many_kv_heads_in_the_fewest_splits(F, Q, K, fmt, nkv, g, n):
    """Two splits of a cache that other kernels would cut into two or three: a wave's first round only, a second one partly filled, waves without a key. Rows behind
    the length on the device hold nothing. The bar is the one above."""
    from ferric_amd import decode as X
    from oracle import decode_oracle as D
    rng, hd, cap = np.random.default_rng(n + fmt), 64, 5121
    width = nkv * hd
    k, v = (rng.standard_normal((n, width)).astype(np.float32) for _ in range(2))
    q = rng.standard_normal((1, nkv * g * hd)).astype(np.float32)
    kq, vq = (Q.QKvCache(fmt, cap, width).append(F.Tensor.from_vec(x, x.shape)) for x in (k, v))
    word = F.Tensor.from_vec(np.array([n - 1], np.uint32).view(np.float32), (1,))
    got = X.decode_attention_kvq(F.Tensor.from_vec(q, q.shape), kq, vq, nkv * g, nkv, length=cap, last_pos=word).to_vec()
    want = D.decode_attention(q[0], K.roundtrip(k, n, width, fmt), K.roundtrip(v, n, width, fmt), nkv * g, nkv, 0, 0.0).reshape(-1)
    assert np.abs(got - want).max() <= 1e-5 * np.abs(want).max()


@pytest.mark.parametrize("nkv,g,n", [(171, 3, 700), (300, 3, 511), (171, 6, 257), (171, 8, 31)])
def test_long_caches_of_many_kv_heads_of_blocks_with_a_minimum(F, Q, K, nkv, g, n):
    test_long_caches_of_many_kv_heads_in_the_fewest_splits(F, Q, K, 2, nkv, g, n)


@pytest.mark.parametrize("off,every", [(3.0, 1), (12.0, 16)])
def test_blocks_with_a_minimum_whose_channels_lie_off_zero(F, Q, K, off, every):
    """Q4_1 rows whose channels, all or one in sixteen, lie several times the spread off zero: there a block's minimum and its codes cancel, unless the codes are taken from the one
    next to zero. At the bar above, and over all of it no further from f64 than attention over the dequantized rows."""
    from types import SimpleNamespace
    from ferric_amd import decode as X
    from oracle import decode_oracle as D
    rows, squares = 5200, np.zeros(2)
    for nh, nkv, hd in ((3, 1, 64), (5, 1, 128), (8, 1, 128)):
        for seed in range(6):
            rng, width = np.random.default_rng(seed), nkv * hd
            k, v = ((rng.standard_normal((rows, width)) + off * rng.standard_normal(width) * (rng.integers(0, every, width) == 0)).astype(np.float32) for _ in range(2))
            q = (rng.standard_normal((1, nh * hd)) * (4.0 if seed % 2 else 1.0)).astype(np.float32)
            kq, vq = (Q.QKvCache.from_tensor(F.Tensor.from_vec(x, x.shape), Q.Q4_1) for x in (k, v))
            plain, qt = SimpleNamespace(k=kq.dequantize(), v=vq.dequantize(), cap=rows, width=width, len=rows), F.Tensor.from_vec(q, q.shape)
            want = D.decode_attention(q[0], K.roundtrip(k, rows, width, Q.Q4_1), K.roundtrip(v, rows, width, Q.Q4_1), nh, nkv, 0, 0.0).reshape(-1)
            errors = [t.to_vec().reshape(-1) - want for t in (X.decode_attention_kvq(qt, kq, vq, nh, nkv), X.decode_attention(qt, plain, nh, nkv))]
            assert np.abs(errors[0]).max() <= 1e-5 * np.abs(want).max(), (nh, hd, seed)
            squares += [(e.astype(np.float64) ** 2).sum() / (want.astype(np.float64) ** 2).sum() for e in errors]
    assert squares[0] <= squares[1], np.sqrt(squares)


@pytest.mark.parametrize("fmt", [0, 1])
@pytest.mark.parametrize("nkv,g,hd,n", [(8, 5, 128, 33), (8, 3, 64, 1), (5, 8, 128, 8340), (171, 3, 64, 514), (171, 5, 128, 514), (171, 8, 128, 258), (300, 6, 128, 31)])
def test_the_token_s_row_at_the_edges_of_long_caches(F, Q, K, fmt, nkv, g, hd, n):
    """The token's row is the first of a wave's round, its first round or a later one, or the only row of its split; splits behind it are empty; two splits at both head sizes.
    With the post-processing inside the launch and in front of it: the same bits and the same row in the cache, the outputs at the bar above."""
    from ferric_amd import decode as X
    from oracle import decode_oracle as D
    rng, lib, cap, nh, width = np.random.default_rng(n + fmt), F._lib.load(), max(n, 5121), nkv * g, nkv * hd
    T = lambda a: F.Tensor.from_vec(a, a.shape)
    rows = [rng.standard_normal((n, width)).astype(np.float32) for _ in range(2)]
    raw = rng.standard_normal((1, (nh + 2 * nkv) * hd)).astype(np.float32)
    qkv, p, ws = T(raw), X._u32_tensor([n - 1]), F.DeviceBuffer(lib.fhip_decode_attention_ws_bytes(nh, nkv, hd, cap))
    got = []
    for one in (False, True):
        kc, vc = (Q.QKvCache(fmt, cap, width).append(T(r)) for r in rows)
        out, q = T(np.zeros((1, nh * hd), np.float32)), T(np.zeros((1, nh * hd), np.float32))
        where = (kc.codes.ptr, kc.scales.ptr, vc.codes.ptr, vc.scales.ptr)
        if one:
            F._lib.check(lib.fhip_qkv_post_attention_kvq(fmt, qkv.buf.ptr, None, None, None, p.buf.ptr, None, nh, nkv, hd, 0, 0, 1e-6, 1e6, *where, cap, cap, 0, 0.0, ws.ptr,
                                                         out.buf.ptr, None))
        else:
            F._lib.check(lib.fhip_qkv_post_kvq(fmt, qkv.buf.ptr, None, None, None, p.buf.ptr, None, 1, nh, nkv, hd, 0, 0, 1e-6, 1e6, q.buf.ptr, *where, cap, None))
            F._lib.check(lib.fhip_decode_attention_kvq(fmt, q.buf.ptr, *where, nh, nkv, hd, cap, p.buf.ptr, 0, 0.0, ws.ptr, out.buf.ptr, None))
        got.append([out.to_vec()] + [c.dequantize().to_vec() for c in (kc, vc)])
    for a, b in zip(*got):
        assert np.array_equal(bits(a), bits(b))
    for r, own in zip(rows, (raw[0, nh * hd:nh * hd + width], raw[0, nh * hd + width:])):
        r[n - 1] = own
    want = D.decode_attention(raw[0, :nh * hd], *(K.roundtrip(r, n, width, fmt) for r in rows), nh, nkv, 0, 0.0).reshape(-1)
    assert np.abs(got[1][0] - want).max() <= 1e-5 * np.abs(want).max()


@pytest.mark.parametrize("nkv,g,hd,n", [(8, 5, 128, 33), (8, 3, 64, 1), (5, 8, 128, 8340), (171, 3, 64, 514), (171, 8, 128, 258)])
def test_the_token_s_row_of_blocks_with_a_minimum(F, Q, K, nkv, g, hd, n):
    test_the_token_s_row_at_the_edges_of_long_caches(F, Q, K, 2, nkv, g, hd, n)



@pytest.mark.parametrize("nkv,g,hd,n", [(8, 5, 128, 33), (8, 3, 64, 1), (5, 8, 128, 8340), (171, 8, 128, 258), (300, 6, 128, 31)])
def test_the_token_s_row_of_blocks_with_a_minimum(F, Q, K, nkv, g, hd, n):
    """The same on a Q4_1 cache, fused and not."""
    test_the_token_s_row_at_the_edges_of_long_caches(F, Q, K, 2, nkv, g, hd, n)


def test_k_and_v_rows_stored_by_one_launch(F, Q, K):
    rng = np.random.default_rng(80)
    t, width, cap = 5, 256, 16
    k, v = rng.standard_normal((t, width)).astype(np.float32), (rng.standard_normal((t, width)) * 7).astype(np.float32)
    lib = F._lib.load()
    for fmt in (0, 1, 2):
        kq, vq = Q.QKvCache(fmt, cap, width), Q.QKvCache(fmt, cap, width)
        pos = F.Tensor(F.DeviceBuffer(4 * t), (t,), np.uint32)
        where = np.array([3, 0, 9, 15, 4], np.uint32)
        F._lib.check(lib.fhip_memcpy_h2d(pos.buf.ptr, where.ctypes.data, 4 * t, None))
        kt, vt = F.Tensor.from_vec(k, k.shape), F.Tensor.from_vec(v, v.shape)
        F._lib.check(lib.fhip_kvq_append2(fmt, kt.buf.ptr, vt.buf.ptr, 0, t, width, pos.buf.ptr, 0, cap, kq.codes.ptr, kq.scales.ptr, vq.codes.ptr,
                                          vq.scales.ptr, None))
        kq.len = vq.len = cap
        for cache, x in ((kq, k), (vq, v)):
            got = cache.dequantize().to_vec().reshape(cap, width)
            for i, r in enumerate(where):
                assert np.array_equal(bits(got[r]), bits(K.roundtrip(x[i], 1, width, fmt)[0])), (fmt, i)


@pytest.mark.parametrize("fmt", [0, 1, 2])
@pytest.mark.parametrize("nh,nkv,hd,n_rot,inter,norms", [(10, 2, 128, 128, 0, True), (4, 4, 64, 64, 1, True), (6, 3, 32, 16, 0, False), (5, 1, 96, 64, 0, True),
                                                         (2, 1, 256, 256, 0, True), (8, 2, 64, 0, 0, True)])
def test_post_processing_and_quantized_stores_in_one_launch(F, Q, fmt, nh, nkv, hd, n_rot, inter, norms):
    """fhip_qkv_post_kvq against fhip_qkv_post_packed followed by fhip_kvq_append2: the same query bits, codes and scales, for heads of one, one
    and a half and four halves of a wave; blocks of zeros of both signs, equal magnitudes, NaN and infinities; a position past the cache."""
    rng = np.random.default_rng(nh * hd + fmt)
    lib, t, cap, width = F._lib.load(), 5, 9, nkv * hd
    T = lambda a: F.Tensor.from_vec(a, a.shape)
    qkv = (rng.standard_normal((t, (nh + 2 * nkv) * hd)) * 3).astype(np.float32)
    v = qkv[:, (nh + nkv) * hd:]
    v[0, :32] = np.where(np.arange(32) % 2, 0.0, -0.0)
    v[1, :32] = np.where(np.arange(32) % 3, 2.5, -2.5)
    v[2, 3], v[2, 20], v[3, 5] = np.nan, np.inf, 1e-42
    v[3, 6:32] = np.abs(v[3, 6:32])
    bias, qn, kn = (rng.standard_normal(n).astype(np.float32) for n in (qkv.shape[1], hd, hd))
    bias[(nh + nkv) * hd:] = 0
    bt, qnt, knt = (T(bias), T(qn), T(kn)) if norms else (None, None, None)
    P = lambda x: x.buf.ptr if x is not None else None
    qt, pt = T(qkv), F.Tensor(F.DeviceBuffer(4 * t), (t,), np.uint32)
    where = np.array([3, 0, 8, 7, cap + 2], np.uint32)
    F._lib.check(lib.fhip_memcpy_h2d(pt.buf.ptr, where.ctypes.data, 4 * t, None))
    got = []
    for one in (True, False):
        kq, vq, qo = Q.QKvCache(fmt, cap, width), Q.QKvCache(fmt, cap, width), T(np.full((t, nh * hd), 7.0, np.float32))
        for c in (kq, vq):
            for b in (c.codes, c.scales):
                fill = np.full(b.nbytes, 0x5A, np.uint8)
                F._lib.check(lib.fhip_memcpy_h2d(b.ptr, fill.ctypes.data, b.nbytes, None))
        if one:
            F._lib.check(lib.fhip_qkv_post_kvq(fmt, qt.buf.ptr, P(bt), P(qnt), P(knt), pt.buf.ptr, None, t, nh, nkv, hd, n_rot, inter, 1e-6, 1e6, qo.buf.ptr,
                                               kq.codes.ptr, kq.scales.ptr, vq.codes.ptr, vq.scales.ptr, cap, None))
        else:
            k1, v1 = F.Tensor.empty((t, width)), F.Tensor.empty((t, width))
            F._lib.check(lib.fhip_qkv_post_packed(qt.buf.ptr, P(bt), P(qnt), P(knt), pt.buf.ptr, None, t, nh, nkv, hd, n_rot, inter, 1e-6, 1e6, qo.buf.ptr,
                                                  k1.buf.ptr, v1.buf.ptr, None))
            F._lib.check(lib.fhip_kvq_append2(fmt, k1.buf.ptr, v1.buf.ptr, 0, t, width, pt.buf.ptr, 0, cap, kq.codes.ptr, kq.scales.ptr, vq.codes.ptr,
                                              vq.scales.ptr, None))
        raw = [bits(qo.to_vec())]
        for b in (kq.codes, kq.scales, vq.codes, vq.scales):
            h = np.empty(b.nbytes, np.uint8)
            F._lib.check(lib.fhip_memcpy_d2h(h.ctypes.data, b.ptr, b.nbytes, None))
            raw.append(h)
        got.append(raw)
    for name, a, b in zip(("q", "k codes", "k scales", "v codes", "v scales"), *got):
        assert np.array_equal(a, b), (name, np.flatnonzero(a != b)[:8])
    c = kq
    assert lib.fhip_qkv_post_kvq(fmt, qt.buf.ptr, None, None, None, pt.buf.ptr, None, 1, 1, 1, 288, 0, 0, 1e-6, 1e6, qt.buf.ptr, c.codes.ptr, c.scales.ptr, c.codes.ptr,
                                 c.scales.ptr, cap, None) != 0 and b"multiple of 32" in lib.fhip_last_error()


@pytest.mark.parametrize("fmt", [0, 1, 2])
@pytest.mark.parametrize("nh,nkv,hd,n_rot,inter,norms,t,past", [
    # heads rotated whole, one a wave and eight (the last wave of a token with six, four, all); other rotations and head sizes
    (10, 2, 128, 128, 0, True, 5, 0), (5, 1, 64, 64, 0, True, 7, 33), (10, 2, 128, 128, 0, True, 600, 3), (8, 2, 64, 64, 0, False, 700, 130), (4, 2, 64, 64, 0, True, 1100, 0),
    (4, 4, 64, 64, 1, True, 5, 9), (6, 3, 32, 16, 0, False, 41, 1), (2, 1, 96, 96, 0, True, 3, 3), (8, 2, 128, 0, 0, True, 4, 1)])
def test_post_processing_stores_and_rows_in_one_launch(F, Q, fmt, nh, nkv, hd, n_rot, inter, norms, t, past):
    """fhip_qkv_post_kvq_rows against fhip_qkv_post_packed, fhip_kvq_append2 and fhip_kvq_dequantize_rows of both caches: the same bits everywhere, over blocks of zeros
    of both signs, equal magnitudes, NaN and infinities; a position past the rows' outputs is stored and leaves no row, one past the cache neither."""
    rng = np.random.default_rng(nh * hd + fmt)
    lib, width = F._lib.load(), nkv * hd
    n, cap = past + t - 1, past + t + 2
    T = lambda a: F.Tensor.from_vec(a, a.shape)
    qkv = (rng.standard_normal((t, (nh + 2 * nkv) * hd)) * 3).astype(np.float32)
    v = qkv[:, (nh + nkv) * hd:]
    v[0, :32] = np.where(np.arange(32) % 2, 0.0, -0.0)
    v[1, :32] = np.where(np.arange(32) % 3, 2.5, -2.5)
    v[2, 3], v[2, 20] = np.nan, np.inf
    bias, qn, kn = (rng.standard_normal(m).astype(np.float32) for m in (qkv.shape[1], hd, hd))
    bt, qnt, knt = (T(bias), T(qn), T(kn)) if norms else (None, None, None)
    P = lambda x: x.buf.ptr if x is not None else None
    where = past + rng.permutation(t).astype(np.uint32)
    where[where == past + 1] = cap + 2
    qt, pt = T(qkv), F.Tensor(F.DeviceBuffer(4 * t), (t,), np.uint32)
    F._lib.check(lib.fhip_memcpy_h2d(pt.buf.ptr, where.ctypes.data, 4 * t, None))
    old = [rng.standard_normal((cap, width)).astype(np.float32) for _ in range(2)]
    got = []
    for one in (True, False):
        kq, vq = (Q.QKvCache.from_tensor(T(o), fmt) for o in old)
        qo, rows = T(np.full((t, nh * hd), 7.0, np.float32)), [T(np.full((n, width), 7.0, np.float32)) for _ in range(2)]
        if one:
            F._lib.check(lib.fhip_qkv_post_kvq_rows(fmt, qt.buf.ptr, P(bt), P(qnt), P(knt), pt.buf.ptr, None, t, nh, nkv, hd, n_rot, inter, 1e-6, 1e6, qo.buf.ptr, kq.codes.ptr,
                                                    kq.scales.ptr, vq.codes.ptr, vq.scales.ptr, cap, rows[0].buf.ptr, rows[1].buf.ptr, n, past, None))
        else:
            k1, v1 = F.Tensor.empty((t, width)), F.Tensor.empty((t, width))
            F._lib.check(lib.fhip_qkv_post_packed(qt.buf.ptr, P(bt), P(qnt), P(knt), pt.buf.ptr, None, t, nh, nkv, hd, n_rot, inter, 1e-6, 1e6, qo.buf.ptr, k1.buf.ptr,
                                                  v1.buf.ptr, None))
            F._lib.check(lib.fhip_kvq_append2(fmt, k1.buf.ptr, v1.buf.ptr, 0, t, width, pt.buf.ptr, 0, cap, kq.codes.ptr, kq.scales.ptr, vq.codes.ptr, vq.scales.ptr, None))
            for c, r in zip((kq, vq), rows):
                F._lib.check(lib.fhip_kvq_dequantize_rows(fmt, c.codes.ptr, c.scales.ptr, 0, n, width, None, r.buf.ptr, None))
        r = [bits(x.to_vec()).reshape(n, width) for x in rows]
        if not one and past + 1 < n:
            for x in r:
                x[past + 1] = np.float32(7.0).view(np.uint32)    # the position that went past the cache
        got.append([bits(qo.to_vec())] + [x.view(np.uint8) for c in (kq, vq) for x in c.to_host()] + r)
    for name, a, b in zip(("q", "k codes", "k scales", "v codes", "v scales", "k rows", "v rows"), *got):
        assert np.array_equal(a, b), (name, np.flatnonzero(a.reshape(-1) != b.reshape(-1))[:8])
    call = lambda rows, n_rows, first: lib.fhip_qkv_post_kvq_rows(fmt, qt.buf.ptr, None, None, None, pt.buf.ptr, None, 1, nh, nkv, hd, n_rot, inter, 1e-6, 1e6, qo.buf.ptr, kq.codes.ptr,
                                                                  kq.scales.ptr, vq.codes.ptr, vq.scales.ptr, cap, rows, rows, n_rows, first, None)
    assert call(None, 1, 0) != 0 and call(rows[0].buf.ptr, cap + 1, 0) != 0 and call(rows[0].buf.ptr, 1, 2) != 0


@pytest.mark.parametrize("fmt", [0, 1, 2])
@pytest.mark.parametrize("nh,nkv,hd,cap,pos,norm,bias,inter,n_rot,window,cap_soft", [
    # one workgroup a query head: four waves, the first of sixteen, full, the last; a head of its own per KV head
    (10, 2, 128, 1, 0, True, False, False, 128, 0, 0.0), (8, 4, 64, 96, 95, True, True, False, 64, 0, 0.0), (8, 4, 64, 97, 64, False, False, True, 64, 0, 30.0),
    (40, 8, 128, 352, 351, True, False, False, 128, 100, 0.0), (4, 4, 128, 352, 200, True, True, False, 64, 0, 0.0),
    # a workgroup a query head and split; all heads of a KV head a workgroup, and the matrix kernel (three heads and more), whose first request waits for the row
    (8, 4, 128, 353, 352, True, False, False, 128, 0, 0.0), (40, 8, 128, 1500, 1300, True, True, False, 128, 0, 0.0), (4, 4, 64, 700, 699, True, False, False, 64, 0, 0.0),
    (8, 4, 128, 5300, 5299, True, False, False, 128, 0, 0.0), (10, 2, 64, 5300, 4000, True, True, False, 64, 0, 0.0), (16, 2, 128, 6000, 5999, True, False, True, 128, 300, 0.0),
    (16, 2, 64, 6000, 17, True, False, False, 32, 0, 20.0), (6, 2, 128, 5200, 5100, False, False, False, 0, 0, 0.0),
    # a position past the cache is attended up to the cache's end and appended nowhere
    (8, 4, 128, 300, 300, True, False, False, 128, 0, 0.0), (10, 2, 64, 5300, 6000, True, False, False, 64, 0, 0.0)])
def test_post_processing_inside_the_attention_launch(F, Q, fmt, nh, nkv, hd, cap, pos, norm, bias, inter, n_rot, window, cap_soft):
    # the two calls and the one leave the same bytes in the cache and the same outputs, bit for bit
    from ferric_amd import decode as X
    lib, rng = F._lib.load(), np.random.default_rng(cap + pos + fmt)
    T = lambda a: F.Tensor.from_vec(a, a.shape)
    width, row = nkv * hd, (nh + 2 * nkv) * hd
    qkv = T(rng.standard_normal((1, row)).astype(np.float32))
    b = T(rng.standard_normal(row).astype(np.float32)) if bias else None
    qn, kn = (T(rng.standard_normal(hd).astype(np.float32)) for _ in range(2)) if norm else (None, None)
    P = lambda t: t.buf.ptr if t is not None else None
    rows = [rng.standard_normal((cap, width)).astype(np.float32) for _ in range(2)]
    p = X._u32_tensor([pos])
    ws = F.DeviceBuffer(max(256, lib.fhip_decode_attention_ws_bytes(nh, nkv, hd, cap)))
    got = []
    for one in (False, True):
        kc, vc = (Q.QKvCache.from_tensor(T(r), fmt) for r in rows)
        out, q = T(np.zeros((1, nh * hd), np.float32)), T(np.zeros((1, nh * hd), np.float32))
        if one:
            F._lib.check(lib.fhip_qkv_post_attention_kvq(fmt, qkv.buf.ptr, P(b), P(qn), P(kn), p.buf.ptr, None, nh, nkv, hd, n_rot, int(inter), 1e-6, 1e6, kc.codes.ptr,
                                                         kc.scales.ptr, vc.codes.ptr, vc.scales.ptr, cap, cap, window, cap_soft, ws.ptr, out.buf.ptr, None))
        else:
            F._lib.check(lib.fhip_qkv_post_kvq(fmt, qkv.buf.ptr, P(b), P(qn), P(kn), p.buf.ptr, None, 1, nh, nkv, hd, n_rot, int(inter), 1e-6, 1e6, q.buf.ptr, kc.codes.ptr,
                                               kc.scales.ptr, vc.codes.ptr, vc.scales.ptr, cap, None))
            F._lib.check(lib.fhip_decode_attention_kvq(fmt, q.buf.ptr, kc.codes.ptr, kc.scales.ptr, vc.codes.ptr, vc.scales.ptr, nh, nkv, hd, cap, p.buf.ptr, window, cap_soft,
                                                       ws.ptr, out.buf.ptr, None))
        got.append([out.to_vec().view(np.uint32)] + [x.view(np.uint8) for c in (kc, vc) for x in c.to_host()])
    for a, c in zip(*got):
        assert np.array_equal(a, c)


def test_post_processing_inside_the_attention_launch_refuses(F, Q):
    lib = F._lib.load()
    t = F.Tensor.from_vec(np.zeros(1024, np.float32), (1024,))
    call = lambda fmt=0, qkv=t.buf.ptr, nh=2, nkv=1, hd=64, cap=4, n=4, soft=0.0, ws=t.buf.ptr: lib.fhip_qkv_post_attention_kvq(
        fmt, qkv, None, None, None, t.buf.ptr, None, nh, nkv, hd, 64, 0, 1e-6, 1e6, t.buf.ptr, t.buf.ptr, t.buf.ptr, t.buf.ptr, cap, n, 0, soft, ws, t.buf.ptr, None)
    for bad in (dict(fmt=7), dict(qkv=None), dict(nh=3, nkv=2), dict(nh=9), dict(hd=96), dict(n=5), dict(n=0), dict(soft=-1.0), dict(cap=6000, n=6000, ws=None)):
        assert call(**bad) != 0, bad
