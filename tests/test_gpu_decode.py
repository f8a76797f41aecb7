"""The decode-layer steps around the quantized matmuls, through the C ABI, against the f64 oracle (oracle/decode_oracle.py).
Floating-point kernels: tolerances are written at each comparison, relative to the largest expected magnitude; the
residual sum of add_rmsnorm, the pass-through dims of rope and cache appends are copies or single f32 adds and must be
bit-exact."""
import numpy as np
import pytest

from conftest import bits, dot_bar

pytestmark = pytest.mark.gpu
Q8_0, Q4_K, Q6_K = 8, 12, 14


@pytest.fixture(scope="module")
def D():
    from oracle import decode_oracle
    return decode_oracle


@pytest.fixture(scope="module")
def X(F):
    from ferric_amd import decode
    return decode


def close(got, want, rel):
    want = np.asarray(want, np.float64)
    return np.abs(np.asarray(got, np.float64).reshape(want.shape) - want).max() <= rel * max(1e-30, np.abs(want).max())


def test_rmsnorm_and_add_rmsnorm(F, X, D):
    rng = np.random.default_rng(0)
    for rows, d in [(1, 5120), (3, 4096), (40, 128), (7, 64), (1, 1), (5, 33), (2, 513), (1, 17408)]:
        x = (rng.standard_normal((rows, d)) * 3).astype(np.float32)
        y = rng.standard_normal((rows, d)).astype(np.float32)
        w = rng.standard_normal(d).astype(np.float32)
        xt, yt, wt = F.Tensor.from_vec(x, (rows, d)), F.Tensor.from_vec(y, (rows, d)), F.Tensor.from_vec(w, (d,))
        assert close(X.rmsnorm(xt, wt, 1e-6).to_vec(), D.rmsnorm(x, w, 1e-6), 2e-6), (rows, d)
        s, n = X.add_rmsnorm(xt, yt, wt, 1e-5)
        so, no = D.add_rmsnorm(x, y, w, 1e-5)
        assert np.array_equal(bits(s.to_vec()), bits(so.reshape(-1))), (rows, d)       # the next residual: exact f32 a + b
        assert close(n.to_vec(), no, 2e-6), (rows, d)
        assert np.array_equal(bits(X.add(xt, yt).to_vec()), bits((x + y).reshape(-1)))
    # the residual updated in place (sum written over a)
    lib = __import__("ferric_amd")._lib.load()
    a = F.Tensor.from_vec(x, x.shape); nrm = F.Tensor.empty(x.shape)
    F._lib.check(lib.fhip_add_rmsnorm(a.buf.ptr, yt.buf.ptr, wt.buf.ptr, x.shape[0], x.shape[1], 1e-5, a.buf.ptr, nrm.buf.ptr, None))
    assert np.array_equal(bits(a.to_vec()), bits(so.reshape(-1))) and close(nrm.to_vec(), no, 2e-6)
    zero = X.rmsnorm(F.Tensor.from_vec(np.zeros((2, 64), np.float32), (2, 64)), F.Tensor.from_vec(np.ones(64, np.float32), (64,)), 1e-6)
    assert not zero.to_vec().any()
    with pytest.raises(AssertionError, match="shape mismatch"):
        X.add_rmsnorm(xt, F.Tensor.from_vec(np.zeros(4, np.float32), (1, 4)), wt, 1e-5)


# rows below and beyond which a norm requests its weights with the row (1024 workgroups, of a row or of four), by registers' worth of a row and its remainders
@pytest.mark.parametrize("rows,d", [(1024, 516), (1025, 516), (1025, 5120), (1025, 8192), (4096, 64), (4097, 64), (4099, 500), (1100, 8196), (1030, 517)])
def test_a_norm_s_bits_do_not_depend_on_how_many_rows_there_are(F, rows, d):
    lib, rng = F._lib.load(), np.random.default_rng(d)
    T = lambda a: F.Tensor.from_vec(a, a.shape)
    x, y, w = T(rng.standard_normal((rows, d)).astype(np.float32)), T(rng.standard_normal((rows, d)).astype(np.float32)), T(rng.standard_normal(d).astype(np.float32))

    def norms(first, n):
        at = lambda t, size: t.buf.ptr.value + first * d * size
        o, s, h = F.Tensor.empty((n, d)), F.Tensor.empty((n, d)), F.Tensor.empty((n, d), np.uint16)
        F._lib.check(lib.fhip_rmsnorm(at(x, 4), w.buf.ptr, n, d, 1e-6, o.buf.ptr, None))
        F._lib.check(lib.fhip_add_rmsnorm_bf16(at(x, 4), at(y, 4), w.buf.ptr, n, d, 1e-6, s.buf.ptr, h.buf.ptr, None))
        return [t.to_vec().reshape(n, d).view(np.uint16 if t is h else np.uint32) for t in (o, s, h)]
    whole = norms(0, rows)
    for first, n in ((0, 1), (rows - 9, 9), (rows // 2 & ~3, 64)):
        for a, b in zip(whole, norms(first, n)):
            assert np.array_equal(a[first:first + n], b), (first, n)


def test_rope_variants(F, X, D):
    rng = np.random.default_rng(1)
    for t, heads, hd, base, off in [(1, 40, 128, 1e6, 0), (1, 48, 128, 1e6, 4095), (5, 8, 64, 1e4, 129), (3, 2, 8, 1e4, 7), (2, 3, 256, 5e5, 31999)]:
        x = rng.standard_normal((t, heads * hd)).astype(np.float32)
        xt = F.Tensor.from_vec(x, x.shape)
        pos = [off + i for i in range(t)]
        # |error| <= 2e-6 of the largest magnitude: sin / cos of the same f32 angle to a few ulp, three roundings per output
        assert close(X.rope(xt, heads, hd, base, off).to_vec(), D.rope(x, heads, hd, base, pos), 2e-6), (t, heads, hd)
        assert close(X.rope(xt, heads, hd, base, off, interleaved=True).to_vec(), D.rope(x, heads, hd, base, pos, interleaved=True), 2e-6)
        scattered = [int(p) for p in rng.integers(0, 40000, t)]
        assert close(X.rope(xt, heads, hd, base, positions=scattered).to_vec(), D.rope(x, heads, hd, base, scattered), 2e-6)
        fs = (rng.random(hd // 2) + 0.5).astype(np.float32)
        got = X.rope(xt, heads, hd, base, positions=scattered, freq_scale=F.Tensor.from_vec(fs, fs.shape), interleaved=True).to_vec()
        assert close(got, D.rope(x, heads, hd, base, scattered, interleaved=True, freq_scale=fs), 2e-6)
        n_rot = hd // 2 + (hd // 2) % 2
        part = X.rope(xt, heads, hd, base, off, n_rot=n_rot).to_vec().reshape(t, heads, hd)
        assert close(part, D.rope(x, heads, hd, base, pos, n_rot=n_rot).reshape(t, heads, hd), 2e-6)
        assert np.array_equal(bits(part[:, :, n_rot:]), bits(x.reshape(t, heads, hd)[:, :, n_rot:]))   # the tail is a copy
    assert np.array_equal(bits(X.rope(xt, heads, hd, base, 0, positions=[0] * t).to_vec()), bits(x.reshape(-1)))   # position 0: identity
    with pytest.raises(AssertionError, match="n_rot must be even"):
        X.rope(xt, heads, hd, base, 0, n_rot=3)
    with pytest.raises(AssertionError, match="one position per row"):
        X.rope(xt, heads, hd, base, positions=[1] * (t + 1))
    # a strided window (the q|k span of a fused qkv row) read in place
    lib = F._lib.load()
    t, nh, nkv, hd = 3, 4, 2, 64
    qkv = rng.standard_normal((t, (nh + 2 * nkv) * hd)).astype(np.float32)
    qt = F.Tensor.from_vec(qkv, qkv.shape)
    out = F.Tensor.empty((t, (nh + nkv) * hd))
    F._lib.check(lib.fhip_rope(qt.buf.ptr, (nh + 2 * nkv) * hd, t, nh + nkv, hd, hd, 1e6, None, 11, None, 0, out.buf.ptr, None))
    assert close(out.to_vec(), D.rope(qkv[:, :(nh + nkv) * hd], nh + nkv, hd, 1e6, [11, 12, 13]), 2e-6)


def test_kv_append2_and_decode_attention(F, X, D):
    rng = np.random.default_rng(2)
    # (14, 2, 64, [8192]): head_dim 64 with more than 64 splits of the key range (2 KV heads on 256 CUs), the case in which
    # the combine kernel's thread count and its loop stride have to agree
    for nh, nkv, hd, lens in [(40, 8, 128, [1, 7, 64, 65, 255, 256, 257, 384, 1000, 5120, 5121]), (8, 8, 64, [3, 257]), (16, 2, 128, [130]), (6, 2, 64, [33]), (5, 1, 128, [2049]),
                              (64, 8, 128, [4097]), (14, 2, 64, [8192])]:
        cap = max(lens) + 3
        width = nkv * hd
        k = rng.standard_normal((cap, width)).astype(np.float32)
        v = rng.standard_normal((cap, width)).astype(np.float32)
        k[:, :hd] *= 4.0                                      # one KV head with peaky scores
        cache = X.KvCache(cap, width)
        cache.append2(F.Tensor.from_vec(k[:5], (5, width)), F.Tensor.from_vec(v[:5], (5, width)))
        cache.append2(F.Tensor.from_vec(k[5:], (cap - 5, width)), F.Tensor.from_vec(v[5:], (cap - 5, width)))
        assert cache.len == cap and np.array_equal(bits(cache.k.to_vec()), bits(k.reshape(-1))) and np.array_equal(bits(cache.v.to_vec()), bits(v.reshape(-1)))
        q = rng.standard_normal((1, nh * hd)).astype(np.float32)
        qt = F.Tensor.from_vec(q, q.shape)
        for s in lens:
            want = D.decode_attention(q[0], k[:s], v[:s], nh, nkv)
            got = X.decode_attention(qt, cache, nh, nkv, length=s).to_vec()
            # <= 1e-5 of the largest value: f32 dots of head_dim terms, expf to a few ulp, sums over s keys in f32
            assert close(got, want, 1e-5), (nh, nkv, hd, s)
            # the length read on the device (newest row = s - 1) under a launch sized for the whole cache
            last = X._u32_tensor([s - 1])
            got2 = X.decode_attention(qt, cache, nh, nkv, length=cap, last_pos=last).to_vec()
            assert close(got2, want, 1e-5), (nh, nkv, hd, s, "device length")
    with pytest.raises(AssertionError, match="exceed the capacity"):
        cache.append2(F.Tensor.from_vec(k[:1], (1, width)), F.Tensor.from_vec(v[:1], (1, width)))
    with pytest.raises(AssertionError, match="head_dim must be 64 or 128"):
        X.decode_attention(F.Tensor.from_vec(np.zeros((1, 96), np.float32), (1, 96)), X.KvCache(4, 96), 1, 1, length=1)
    with pytest.raises(AssertionError, match="1..=8 supported"):
        X.decode_attention(F.Tensor.from_vec(np.zeros((1, 9 * 64), np.float32), (1, 9 * 64)), X.KvCache(4, 64), 9, 1, length=1)


def test_empty_inputs_and_argument_errors(F, X):
    """Zero-sized calls return without touching memory; bad shapes and NULL pointers are reported, never launched."""
    lib, chk, E = F._lib.load(), F._lib.check, F._lib.FerricHipError
    t = F.Tensor.from_vec(np.ones(256, np.float32), (2, 128))
    o = F.Tensor.from_vec(np.full(256, 5.0, np.float32), (2, 128))
    w = F.Tensor.from_vec(np.ones(128, np.float32), (128,))
    pos = X._u32_tensor([0, 1])
    chk(lib.fhip_rmsnorm(t.buf.ptr, w.buf.ptr, 0, 128, 1e-6, o.buf.ptr, None))
    chk(lib.fhip_add_rmsnorm(t.buf.ptr, t.buf.ptr, w.buf.ptr, 2, 0, 1e-6, o.buf.ptr, o.buf.ptr, None))
    chk(lib.fhip_add(t.buf.ptr, t.buf.ptr, 0, o.buf.ptr, None))
    chk(lib.fhip_rope(t.buf.ptr, 0, 0, 1, 128, 128, 1e4, None, 0, None, 0, o.buf.ptr, None))
    chk(lib.fhip_kv_append2(t.buf.ptr, t.buf.ptr, 0, 128, None, 0, o.buf.ptr, o.buf.ptr, 2, None))
    chk(lib.fhip_qkv_post(t.buf.ptr, None, None, None, pos.buf.ptr, None, 0, 1, 1, 64, 64, 0, 1e-6, 1e4, o.buf.ptr, o.buf.ptr, o.buf.ptr, 2, None))
    chk(lib.fhip_u32_add(pos.buf.ptr, 0, 1, None))
    assert np.array_equal(o.to_vec(), np.full(256, 5.0, np.float32))                      # nothing was written
    assert lib.fhip_decode_attention_ws_bytes(8, 2, 64, 0) == 0
    for call, msg in [
        (lambda: lib.fhip_rmsnorm(None, w.buf.ptr, 1, 128, 1e-6, o.buf.ptr, None), "NULL pointer"),
        (lambda: lib.fhip_rope(t.buf.ptr, 0, 2, 1, 128, 130, 1e4, None, 0, None, 0, o.buf.ptr, None), "n_rot must be even and <= head_dim"),
        (lambda: lib.fhip_rope(t.buf.ptr, 0, 2, 1, 128, 7, 1e4, None, 0, None, 0, o.buf.ptr, None), "n_rot must be even"),
        (lambda: lib.fhip_decode_attention(t.buf.ptr, t.buf.ptr, t.buf.ptr, 2, 1, 64, 0, None, None, o.buf.ptr, None), "empty cache"),
        (lambda: lib.fhip_decode_attention(t.buf.ptr, t.buf.ptr, t.buf.ptr, 3, 2, 64, 1, None, None, o.buf.ptr, None), "multiple of n_kv_heads"),
        (lambda: lib.fhip_decode_attention(t.buf.ptr, t.buf.ptr, t.buf.ptr, 2, 1, 32, 1, None, None, o.buf.ptr, None), "head_dim must be 64 or 128"),
        (lambda: lib.fhip_qkv_post(t.buf.ptr, None, None, None, None, None, 1, 1, 1, 64, 64, 0, 1e-6, 1e4, o.buf.ptr, o.buf.ptr, o.buf.ptr, 2, None), "NULL pointer"),
        (lambda: lib.fhip_norm_matmul_q(None, t.buf.ptr, None, w.buf.ptr, 1e-6, None, o.buf.ptr, 0, o.buf.ptr, None), "NULL pointer"),
    ]:
        with pytest.raises((E, AssertionError), match=msg):
            chk(call())
    # a long cache without its workspace is refused, not run with a NULL scratch
    with pytest.raises(E, match="needs the workspace"):
        big = X.KvCache(4096, 64)
        chk(lib.fhip_decode_attention(t.buf.ptr, big.k.buf.ptr, big.v.buf.ptr, 2, 1, 64, 4096, None, None, o.buf.ptr, None))


def test_attention_window_and_softcap(F, X, D):
    rng = np.random.default_rng(12)
    for nh, nkv, hd, s in [(40, 8, 128, 1500), (8, 2, 64, 70)]:
        width = nkv * hd
        k = rng.standard_normal((s, width)).astype(np.float32)
        v = rng.standard_normal((s, width)).astype(np.float32)
        q = (rng.standard_normal((1, nh * hd)) * 2).astype(np.float32)
        cache = X.KvCache(s, width)
        cache.append2(F.Tensor.from_vec(k, k.shape), F.Tensor.from_vec(v, v.shape))
        qt = F.Tensor.from_vec(q, q.shape)
        for window, cap in [(0, 0.0), (1, 0.0), (33, 0.0), (s - 1, 0.0), (s, 0.0), (s + 7, 0.0), (0, 50.0), (0, 2.5), (100, 30.0)]:
            got = X.decode_attention(qt, cache, nh, nkv, window=window, softcap=cap).to_vec()
            want = D.decode_attention(q[0], k, v, nh, nkv, window=window, softcap=cap)
            assert close(got, want, 1e-5), (nh, s, window, cap)
        # a window under a length read on the device
        last = X._u32_tensor([s // 2 - 1])
        got = X.decode_attention(qt, cache, nh, nkv, length=s, last_pos=last, window=20).to_vec()
        assert close(got, D.decode_attention(q[0], k[: s // 2], v[: s // 2], nh, nkv, window=20), 1e-5)
    with pytest.raises(F._lib.FerricHipError, match="softcap must be >= 0"):
        X.decode_attention(qt, cache, nh, nkv, softcap=-1.0)


def test_attention_properties_at_a_32k_context(F, X):
    """Sizes the f64 loop oracle does not reach: properties that hold at any length. Attention is linear in V; adding
    one constant to every score (q -> q, K -> K + c e with q.e = 0 is not available, so: duplicate the cache) leaves the
    output unchanged -- keys [K; K], values [V; V] give the same output as K, V; equal keys give the mean of the values."""
    rng = np.random.default_rng(11)
    nh, nkv, hd, s = 40, 8, 128, 16384
    width = nkv * hd
    k = (rng.standard_normal((s, width)) * 0.3).astype(np.float32)
    v1 = rng.standard_normal((s, width)).astype(np.float32)
    v2 = rng.standard_normal((s, width)).astype(np.float32)
    q = rng.standard_normal((1, nh * hd)).astype(np.float32)
    qt = F.Tensor.from_vec(q, q.shape)

    def run(keys, vals):
        c = X.KvCache(keys.shape[0], width)
        c.append2(F.Tensor.from_vec(keys, keys.shape), F.Tensor.from_vec(vals, vals.shape))
        return X.decode_attention(qt, c, nh, nkv).to_vec().astype(np.float64)
    a1, a2 = run(k, v1), run(k, v2)
    mix = run(k, (np.float32(0.5) * v1 - np.float32(2.0) * v2).astype(np.float32))
    assert np.abs(mix - (0.5 * a1 - 2.0 * a2)).max() <= 2e-5 * np.abs(a2).max()
    twice = run(np.concatenate([k, k]), np.concatenate([v1, v1]))          # 32768 keys
    assert np.abs(twice - a1).max() <= 1e-5 * np.abs(a1).max()
    flat = run(np.tile(k[:1], (s, 1)), v1)
    want = np.repeat(v1.astype(np.float64).mean(axis=0).reshape(nkv, 1, hd), nh // nkv, axis=1).reshape(-1)
    assert np.abs(flat - want).max() <= 1e-5 * np.abs(want).max() + 1e-6


@pytest.mark.parametrize("t,nh,nkv,norms", [(513, 10, 2, True), (1100, 5, 1, False), (205, 32, 4, True)])
def test_qkv_post_of_many_rows_has_the_bits_of_single_rows(F, X, D, t, nh, nkv, norms):
    """Eight heads a wave (a last group that is not full; groups that hold query, key and value heads at once) against one head a wave,
    with positions past the cache among the rows: they are dropped by both. One row also against the oracle."""
    rng = np.random.default_rng(t)
    lib, hd, cap = F._lib.load(), 128, 700
    T = lambda a: F.Tensor.from_vec(a, a.shape)
    qkv = rng.standard_normal((t, (nh + 2 * nkv) * hd)).astype(np.float32)
    bias, qn, kn = (rng.standard_normal(n).astype(np.float32) for n in ((nh + 2 * nkv) * hd, hd, hd))
    pos = (rng.permutation(t) + max(0, cap - t + 3)).astype(np.uint32)                # distinct; some at or past the capacity
    bt, qnt, knt = (T(bias), T(qn), T(kn)) if norms else (None, None, None)
    P = lambda x: x.buf.ptr if x is not None else None
    pt, qt = F.Tensor(F.DeviceBuffer(4 * t), (t,), np.uint32), T(qkv)
    F._lib.check(lib.fhip_memcpy_h2d(pt.buf.ptr, pos.ctypes.data, 4 * t, None))
    out = []
    for rows in (t, 1):
        qo, kc, vc = (T(np.full(sh, 7.0, np.float32)) for sh in ((t, nh * hd), (cap, nkv * hd), (cap, nkv * hd)))
        for i in range(0, t, rows):
            F._lib.check(lib.fhip_qkv_post(qt.buf.ptr.value + 4 * i * qkv.shape[1], P(bt), P(qnt), P(knt), pt.buf.ptr.value + 4 * i, None, rows, nh, nkv, hd, hd, 0,
                                           1e-6, 1e6, qo.buf.ptr.value + 4 * i * nh * hd, kc.buf.ptr, vc.buf.ptr, cap, None))
        out.append([x.to_vec() for x in (qo, kc, vc)])
    for a, b in zip(*out):
        assert np.array_equal(bits(a), bits(b))
    i = t // 2
    wq, _, _ = D.qkv_post(qkv[i:i + 1], bias if norms else None, qn if norms else None, kn if norms else None, pos[i:i + 1], nh, nkv, hd, 1e-6, 1e6, interleaved=False)
    assert close(out[0][0].reshape(t, nh * hd)[i], wq.reshape(-1), 1e-5)


def test_qkv_post_fuses_bias_norm_rope_and_append(F, X, D):
    rng = np.random.default_rng(3)
    lib = F._lib.load()
    for nh, nkv, hd, t, use_bias, use_norm, inter in [(40, 8, 128, 1, False, True, False), (4, 2, 64, 3, True, False, False),
                                                      (6, 3, 128, 2, True, True, True), (2, 1, 32, 2, False, False, False)]:
        width = (nh + 2 * nkv) * hd
        qkv = rng.standard_normal((t, width)).astype(np.float32)
        bias = rng.standard_normal(width).astype(np.float32) if use_bias else None
        qn = (rng.random(hd) + 0.5).astype(np.float32) if use_norm else None
        kn = (rng.random(hd) + 0.5).astype(np.float32) if use_norm else None
        pos = [int(p) for p in rng.choice(60, t, replace=False)]
        cap = 64
        kc0, vc0 = rng.standard_normal((cap, nkv * hd)).astype(np.float32), rng.standard_normal((cap, nkv * hd)).astype(np.float32)
        kc, vc = F.Tensor.from_vec(kc0, kc0.shape), F.Tensor.from_vec(vc0, vc0.shape)
        T = lambda a: F.Tensor.from_vec(a, a.shape) if a is not None else None
        qt, bt, qnt, knt, pt = T(qkv), T(bias), T(qn), T(kn), X._u32_tensor(pos)
        qo = F.Tensor.empty((t, nh * hd))
        P = lambda x: x.buf.ptr if x is not None else None
        F._lib.check(lib.fhip_qkv_post(qt.buf.ptr, P(bt), P(qnt), P(knt), pt.buf.ptr, None, t, nh, nkv, hd, hd, int(inter), 1e-6, 1e6,
                                       qo.buf.ptr, kc.buf.ptr, vc.buf.ptr, cap, None))
        wq, wk, wv = D.qkv_post(qkv, bias, qn, kn, pos, nh, nkv, hd, 1e-6, 1e6, interleaved=inter)
        assert close(qo.to_vec(), wq, 3e-6), (nh, nkv, hd)
        kg, vg = kc.to_vec().reshape(cap, -1), vc.to_vec().reshape(cap, -1)
        assert close(kg[pos], wk, 3e-6)
        assert np.array_equal(bits(vg[pos]), bits(wv.astype(np.float32)))                   # values are copied (+ bias: one f32 add)
        rest = [r for r in range(cap) if r not in pos]
        assert np.array_equal(bits(kg[rest]), bits(kc0[rest])) and np.array_equal(bits(vg[rest]), bits(vc0[rest]))   # no other row touched
    # a position past the capacity leaves the caches alone (and still produces the query)
    pt = X._u32_tensor([cap + 5] * t)
    kc, vc = F.Tensor.from_vec(kc0, kc0.shape), F.Tensor.from_vec(vc0, vc0.shape)
    F._lib.check(lib.fhip_qkv_post(qt.buf.ptr, None, None, None, pt.buf.ptr, None, t, nh, nkv, hd, hd, 0, 1e-6, 1e6, qo.buf.ptr, kc.buf.ptr,
                                   vc.buf.ptr, cap, None))
    assert np.array_equal(bits(kc.to_vec()), bits(kc0.reshape(-1))) and np.array_equal(bits(vc.to_vec()), bits(vc0.reshape(-1)))


def test_post_processing_inside_the_attention_launch(F, X, D):
    # fhip_qkv_post_attention against fhip_qkv_post followed by fhip_decode_attention_ex on copies of the same caches: the same
    # attention output, the same appended K and V rows, nothing else touched; one split and many, windows, softcap, a position
    # in the middle of a longer cache (keys past it do not count), group sizes 1..5, both head widths
    rng = np.random.default_rng(31)
    lib = F._lib.load()
    cases = [(40, 8, 128, 700, 699, True, False, False, 0, 0.0), (40, 8, 128, 64, 63, True, False, False, 0, 0.0),
             (4, 2, 64, 300, 120, False, True, False, 0, 0.0), (6, 3, 128, 2100, 2099, True, True, True, 0, 0.0),
             (8, 8, 64, 90, 89, False, False, False, 0, 0.0), (12, 4, 128, 1500, 1499, True, False, False, 256, 0.0),
             (10, 2, 128, 513, 512, True, True, False, 0, 30.0), (2, 1, 128, 1, 0, True, False, False, 0, 0.0),
             # caches of up to 256 rows under grouped query heads: one workgroup per query head, each of a KV head's workgroups
             # appending the same rows; the first key step requested ahead of the post-processing (position past the first 32
             # rows) or behind the append (position among them); the first length past that launch shape
             (40, 8, 128, 256, 255, True, True, False, 0, 0.0), (14, 2, 64, 200, 20, True, False, True, 0, 0.0),
             (14, 2, 64, 200, 199, True, False, True, 64, 0.0), (40, 8, 128, 257, 256, True, False, False, 0, 0.0),
             (14, 2, 64, 300, 20, True, False, True, 0, 0.0), (40, 8, 128, 5120, 5119, True, False, False, 0, 0.0)]
    for nh, nkv, hd, cap, pos, use_norm, use_bias, inter, window, softcap in cases:
        width = (nh + 2 * nkv) * hd
        qkv = rng.standard_normal(width).astype(np.float32)
        bias = rng.standard_normal(width).astype(np.float32) if use_bias else None
        qn = (rng.random(hd) + 0.5).astype(np.float32) if use_norm else None
        kn = (rng.random(hd) + 0.5).astype(np.float32) if use_norm else None
        kc0 = (rng.standard_normal((cap, nkv * hd)) * 0.5).astype(np.float32)
        vc0 = rng.standard_normal((cap, nkv * hd)).astype(np.float32)
        T = lambda a: F.Tensor.from_vec(a, a.shape) if a is not None else None
        P = lambda x: x.buf.ptr if x is not None else None
        qt, bt, qnt, knt, pt = T(qkv.reshape(1, -1)), T(bias), T(qn), T(kn), X._u32_tensor([pos])
        ws = F.DeviceBuffer(max(256, lib.fhip_decode_attention_ws_bytes(nh, nkv, hd, cap)))
        # the two calls
        kc, vc = T(kc0), T(vc0)
        qo, want = F.Tensor.empty((1, nh * hd)), F.Tensor.empty((1, nh * hd))
        F._lib.check(lib.fhip_qkv_post(qt.buf.ptr, P(bt), P(qnt), P(knt), pt.buf.ptr, None, 1, nh, nkv, hd, hd, int(inter), 1e-6, 1e6,
                                       qo.buf.ptr, kc.buf.ptr, vc.buf.ptr, cap, None))
        F._lib.check(lib.fhip_decode_attention_ex(qo.buf.ptr, kc.buf.ptr, vc.buf.ptr, nh, nkv, hd, cap, pt.buf.ptr, window, softcap, ws.ptr,
                                                  want.buf.ptr, None))
        # one call
        kc2, vc2 = T(kc0), T(vc0)
        got = F.Tensor.empty((1, nh * hd))
        F._lib.check(lib.fhip_qkv_post_attention(qt.buf.ptr, P(bt), P(qnt), P(knt), pt.buf.ptr, None, nh, nkv, hd, hd, int(inter), 1e-6, 1e6,
                                                 kc2.buf.ptr, vc2.buf.ptr, cap, cap, window, softcap, ws.ptr, got.buf.ptr, None))
        case = (nh, nkv, hd, cap, pos)
        assert np.array_equal(bits(kc2.to_vec()), bits(kc.to_vec())) and np.array_equal(bits(vc2.to_vec()), bits(vc.to_vec())), case
        assert close(got.to_vec(), want.to_vec(), 2e-6), case
    # a position past the rows attention may look at (len 200 of a cache of 300 rows, position 250): the rows are still appended
    nh, nkv, hd, cap, alen, pos = 8, 2, 128, 300, 200, 250
    width = (nh + 2 * nkv) * hd
    qkv = rng.standard_normal(width).astype(np.float32)
    kc0 = (rng.standard_normal((cap, nkv * hd)) * 0.5).astype(np.float32)
    vc0 = rng.standard_normal((cap, nkv * hd)).astype(np.float32)
    qt, pt = T(qkv.reshape(1, -1)), X._u32_tensor([pos])
    ws = F.DeviceBuffer(max(256, lib.fhip_decode_attention_ws_bytes(nh, nkv, hd, alen)))
    kc, vc, kc2, vc2 = T(kc0), T(vc0), T(kc0), T(vc0)
    qo, want, got = F.Tensor.empty((1, nh * hd)), F.Tensor.empty((1, nh * hd)), F.Tensor.empty((1, nh * hd))
    F._lib.check(lib.fhip_qkv_post(qt.buf.ptr, None, None, None, pt.buf.ptr, None, 1, nh, nkv, hd, hd, 0, 1e-6, 1e6, qo.buf.ptr, kc.buf.ptr,
                                   vc.buf.ptr, cap, None))
    F._lib.check(lib.fhip_decode_attention_ex(qo.buf.ptr, kc.buf.ptr, vc.buf.ptr, nh, nkv, hd, alen, pt.buf.ptr, 0, 0.0, ws.ptr, want.buf.ptr, None))
    F._lib.check(lib.fhip_qkv_post_attention(qt.buf.ptr, None, None, None, pt.buf.ptr, None, nh, nkv, hd, hd, 0, 1e-6, 1e6, kc2.buf.ptr,
                                             vc2.buf.ptr, cap, alen, 0, 0.0, ws.ptr, got.buf.ptr, None))
    assert np.array_equal(bits(kc2.to_vec()), bits(kc.to_vec())) and np.array_equal(bits(vc2.to_vec()), bits(vc.to_vec()))
    assert not np.array_equal(bits(kc2.to_vec().reshape(cap, -1)[pos]), bits(kc0[pos]))
    assert close(got.to_vec(), want.to_vec(), 2e-6)
    with pytest.raises(AssertionError, match="length outside the cache"):
        F._lib.check(lib.fhip_qkv_post_attention(qt.buf.ptr, None, None, None, pt.buf.ptr, None, nh, nkv, hd, hd, 0, 1e-6, 1e6, kc2.buf.ptr,
                                                 vc2.buf.ptr, cap, cap + 1, 0, 0.0, ws.ptr, got.buf.ptr, None))
    with pytest.raises(F._lib.FerricHipError, match="NULL pointer"):
        F._lib.check(lib.fhip_qkv_post_attention(None, None, None, None, pt.buf.ptr, None, nh, nkv, hd, hd, 0, 1e-6, 1e6, kc2.buf.ptr,
                                                 vc2.buf.ptr, cap, cap, 0, 0.0, ws.ptr, got.buf.ptr, None))


# the norm inside the mat-vec (Q4_K), in a launch of its own whose thread takes the word along (Q4_0; rows that are and are not whole 16-byte pieces)
@pytest.mark.parametrize("ty,cols", [(12, 1024), (2, 1024), (2, 8224), (2, 9248)])
@pytest.mark.parametrize("resid", [False, True])
def test_the_position_word_goes_along(F, ty, cols, resid):
    """fhip_norm_matmul_q_count and fhip_add_count: the bits of the calls without the word, and the word."""
    from ferric_amd.synth import synth_weights
    lib, rng = F._lib.load(), np.random.default_rng(cols)
    T = lambda a: F.Tensor.from_vec(a, a.shape)
    x, r, nw = (T(rng.standard_normal(cols).astype(np.float32)) for _ in range(3))
    w = F.QMatrix.from_bytes(synth_weights(ty, 70, cols, 3), ty, 70, cols)
    word = F.Tensor(F.DeviceBuffer(8), (2,), np.uint32)
    start = np.array([0xFFFFFFFE, 7], np.uint32)
    F._lib.check(lib.fhip_memcpy_h2d(word.buf.ptr, start.ctypes.data, 8, None))
    got = []
    for count in (False, True):
        y, xo, hs, total = (F.Tensor.empty((n,)) for n in (70, cols, cols, cols))
        args = (w.handle, x.buf.ptr, r.buf.ptr if resid else None, nw.buf.ptr, 1e-6, xo.buf.ptr if resid else None, hs.buf.ptr, 0, y.buf.ptr)
        F._lib.check(lib.fhip_norm_matmul_q_count(*args, word.buf.ptr, 1, None) if count else lib.fhip_norm_matmul_q(*args, None))
        F._lib.check(lib.fhip_add_count(x.buf.ptr, r.buf.ptr, cols, total.buf.ptr, word.buf.ptr, 40, None) if count else lib.fhip_add(x.buf.ptr, r.buf.ptr, cols, total.buf.ptr, None))
        got.append([t.to_vec().view(np.uint32) for t in ((y, total, xo) if resid else (y, total))])
    for a, b in zip(*got):
        assert np.array_equal(a, b)
    assert word.to_vec().tolist() == [(0xFFFFFFFE + 41) & 0xFFFFFFFF, 7]
    assert lib.fhip_add_count(x.buf.ptr, r.buf.ptr, 4, total.buf.ptr, None, 1, None) != 0


# workgroups that take every CU (the word is a launch of its own); rows dealt in turn to all CUs, or to all but one, which has the word; short of that
@pytest.mark.parametrize("ty", [Q4_K, 13, Q6_K, Q8_0])
@pytest.mark.parametrize("rows", [255, 256, 512, 513, 4096, 66001])
@pytest.mark.parametrize("resid", [False, True])
def test_the_position_word_goes_along_with_full_launches(F, ty, rows, resid):
    """Once, and beside the same bits."""
    from ferric_amd.synth import synth_weights
    lib, cols, rng = F._lib.load(), 768, np.random.default_rng(rows)
    T = lambda a: F.Tensor.from_vec(a, a.shape)
    x, r, nw = (T(rng.standard_normal(cols).astype(np.float32)) for _ in range(3))
    w = F.QMatrix.from_bytes(synth_weights(ty, rows, cols, 3), ty, rows, cols)
    word = T(np.array([5, 9], np.uint32).view(np.float32))
    got = []
    for count in (False, True):
        y, xo, hs = (F.Tensor.empty((n,)) for n in (rows, cols, cols))
        args = (w.handle, x.buf.ptr, r.buf.ptr if resid else None, nw.buf.ptr, 1e-6, xo.buf.ptr if resid else None, hs.buf.ptr, 0, y.buf.ptr)
        F._lib.check(lib.fhip_norm_matmul_q_count(*args, word.buf.ptr, 3, None) if count else lib.fhip_norm_matmul_q(*args, None))
        got.append([bits(t.to_vec()) for t in ((y, xo) if resid else (y,))])
    for a, b in zip(*got):
        assert np.array_equal(a, b)
    assert word.to_vec().view(np.uint32).tolist() == [8, 9]


def test_norm_fused_into_the_matvec(F, X, D, O, precision):
    """fhip_norm_matmul_q against rmsnorm / add_rmsnorm followed by the mat-vec: the residual sum bit-exact, the product
    within the dot-product bound of the unfused pair (the sum of squares is added in another order: ~1e-7 on the scale),
    on shapes the streaming kernel takes (fused) and on ones it does not (the two steps run apart)."""
    from ferric_amd.synth import synth_weights
    rng = np.random.default_rng(6)
    lib = F._lib.load()
    for ty, rows, cols, swiglu in [(Q4_K, 7168, 5120, False), (Q4_K, 2 * 1024, 5120, True), (Q6_K, 512, 5120, False), (Q8_0, 96, 4096, False),
                                   (Q4_K, 64, 768, False), (Q6_K, 40, 17408, False), (Q4_K, 2 * 96, 1024, True)]:
        raw = synth_weights(ty, rows, cols, 3)
        w = F.QMatrix.from_bytes(raw, ty, rows, cols)
        x = rng.standard_normal(cols).astype(np.float32)
        r = rng.standard_normal(cols).astype(np.float32)
        nw = ((rng.random(cols) + 0.5) * 0.05).astype(np.float32)
        xt, rt, nt = F.Tensor.from_vec(x, (1, cols)), F.Tensor.from_vec(r, (1, cols)), F.Tensor.from_vec(nw, (cols,))
        out_rows = rows // 2 if swiglu else rows
        for resid in (rt, None):
            xo, hs, y = F.Tensor.from_vec(np.full(cols, 7.0, np.float32), (1, cols)), F.Tensor.empty((1, cols)), F.Tensor.empty((1, out_rows))
            F._lib.check(lib.fhip_norm_matmul_q(w.handle, xt.buf.ptr, resid.buf.ptr if resid is not None else None, nt.buf.ptr, 1e-6,
                                                xo.buf.ptr, hs.buf.ptr, int(swiglu), y.buf.ptr, None))
            if resid is not None:
                s_ref, h_ref = X.add_rmsnorm(xt, rt, nt, 1e-6)
                assert np.array_equal(bits(xo.to_vec()), bits(s_ref.to_vec())), (ty, rows, cols)
            else:
                h_ref = X.rmsnorm(xt, nt, 1e-6)
                assert np.array_equal(xo.to_vec(), np.full(cols, 7.0, np.float32))        # nothing to store without a residual
            y_ref = (h_ref.matmul_q(w).swiglu(out_rows) if swiglu else h_ref.matmul_q(w)).to_vec()
            h64 = D.rmsnorm((x + r) if resid is not None else x, nw, 1e-6)
            y64, wn = O.matmul_f64(h64.astype(np.float32), raw, ty, rows, cols)
            if swiglu:
                y64 = D.silu_mul(y64, out_rows)
                assert close(y.to_vec(), y64, dot_bar(2)), (ty, rows, cols)
            else:
                assert (np.abs(y.to_vec() - y64[0]) <= 1e-3 * wn * np.linalg.norm(h64)).all()
                assert close(y.to_vec(), y64, dot_bar()), (ty, rows, cols)
            assert close(y.to_vec(), y_ref, 2e-5)
    # outputs that share memory with an input (the in-place residual update included) or with each other are refused
    with pytest.raises(F._lib.FerricHipError, match="x_out must not overlap"):
        F._lib.check(lib.fhip_norm_matmul_q(w.handle, xt.buf.ptr, rt.buf.ptr, nt.buf.ptr, 1e-6, xt.buf.ptr, hs.buf.ptr, 0, y.buf.ptr, None))
    with pytest.raises(F._lib.FerricHipError, match="x_out must not overlap"):
        F._lib.check(lib.fhip_norm_matmul_q(w.handle, xt.buf.ptr, rt.buf.ptr, nt.buf.ptr, 1e-6, rt.buf.ptr, hs.buf.ptr, 0, y.buf.ptr, None))
    with pytest.raises(F._lib.FerricHipError, match="y must not overlap"):
        F._lib.check(lib.fhip_norm_matmul_q(w.handle, xt.buf.ptr, rt.buf.ptr, nt.buf.ptr, 1e-6, xo.buf.ptr, hs.buf.ptr, 0, xo.buf.ptr, None))


def _tiny_model(F, X, O, rng, n_layer, d, nh, nkv, hd, n_ff, qk_norm):
    """Random Q4_K / Q6_K projections (synthetic blocks have rows of norm ~ 2 sqrt(cols)), block norms small enough that the
    projections of a normalised vector are O(1); the f64 twin holds the oracle-dequantized weights."""
    from ferric_amd.synth import synth_weights
    from oracle import decode_oracle as D
    layers, olayers = [], []
    T = lambda a: F.Tensor.from_vec(a, a.shape)
    for il in range(n_layer):
        shapes = {"wqkv": (Q4_K, (nh + 2 * nkv) * hd, d), "wo": (Q4_K, d, nh * hd), "gate_up": (Q4_K, 2 * n_ff, d), "down": (Q6_K, d, n_ff)}
        qm, deq = {}, {}
        for name, (ty, r, c) in shapes.items():
            b = synth_weights(ty, r, c, 100 * il + len(qm))
            qm[name] = F.QMatrix.from_bytes(b, ty, r, c)
            deq[name] = O.deq_raw(b, r * c, ty).reshape(r, c).astype(np.float64)
        norms = {"attn_norm": ((rng.random(d) + 0.5) * 0.02).astype(np.float32), "ffn_norm": ((rng.random(d) + 0.5) * 0.02).astype(np.float32),
                 "q_norm": (rng.random(hd) + 0.5).astype(np.float32), "k_norm": (rng.random(hd) + 0.5).astype(np.float32)}
        layers.append(X.Qwen3Layer(T(norms["attn_norm"]), qm["wqkv"], qm["wo"], T(norms["ffn_norm"]), qm["gate_up"], qm["down"],
                                   T(norms["q_norm"]) if qk_norm else None, T(norms["k_norm"]) if qk_norm else None))
        olayers.append(D.Layer(attn_norm=norms["attn_norm"], ffn_norm=norms["ffn_norm"], q_norm=norms["q_norm"] if qk_norm else None,
                               k_norm=norms["k_norm"] if qk_norm else None, wqkv=deq["wqkv"], wo=deq["wo"], gate_up=deq["gate_up"], down=deq["down"]))
    return layers, olayers


@pytest.mark.parametrize("qk_norm,fuse_norm,fuse_attn", [(True, True, True), (False, True, True), (True, False, False), (True, True, False)])
def test_decoder_steps_match_the_oracle_layer_by_layer_and_replay_as_a_graph(F, X, O, D, qk_norm, fuse_norm, fuse_attn, precision):
    rng = np.random.default_rng(4)
    n_layer, d, nh, nkv, hd, n_ff, steps = 3, 1024, 8, 2, 128, 1536, 6
    cfg = X.Qwen3Cfg(d, nh, nkv, hd, n_ff, eps=1e-6, rope_base=1e6)
    layers, olayers = _tiny_model(F, X, O, rng, n_layer, d, nh, nkv, hd, n_ff, qk_norm)
    xs = (rng.standard_normal((steps, d)) * 0.5).astype(np.float32)
    # oracle: f64 on the dequantized weights, token by token
    kcs, vcs = [[] for _ in olayers], [[] for _ in olayers]
    want = []
    for pos in range(steps):
        x = xs[pos].astype(np.float64)
        for l, kc, vc in zip(olayers, kcs, vcs):
            x = D.apply_layer(x, l, kc, vc, pos, cfg)
        want.append(x)
    stream = F.Stream()
    dec = X.Qwen3Decoder(cfg, layers, max_len=steps + 2, stream=stream, fuse_norm=fuse_norm, fuse_attn=fuse_attn)
    eager = []
    for pos in range(steps):
        dec.set_input(xs[pos])
        dec.step()
        eager.append(dec.hidden())
        # <= 20 times the bar of one dot product, of the largest hidden value: three layers of quantized dots feeding
        # norms, attention and the next projections
        assert close(eager[-1], want[pos], dot_bar(20)), pos
    assert dec.caches[0].len == steps
    # the same steps as one captured graph, replayed with host work and synchronisation between replays
    dec.set_pos(0)
    dec.capture()
    for pos in range(steps):
        dec.set_input(xs[pos])
        dec.step_graph()
        got = dec.hidden()
        assert np.array_equal(bits(got), bits(eager[pos])), pos        # same launches, same order: bit-identical to eager
    pos_word = np.empty(1, np.uint32)
    F._lib.check(F._lib.load().fhip_memcpy_d2h(pos_word.ctypes.data, dec.pos.buf.ptr, 4, stream.handle))
    assert pos_word[0] == steps
    # with the output norm and LM head in the step: logits = rmsnorm(hidden) W_out^T
    from ferric_amd.synth import synth_weights
    head_raw = synth_weights(Q6_K, 300, d, 77)
    onorm = ((rng.random(d) + 0.5) * 0.02).astype(np.float32)
    dec2 = X.Qwen3Decoder(cfg, layers, max_len=4, stream=stream, output_norm=F.Tensor.from_vec(onorm, onorm.shape),
                          lm_head=F.QMatrix.from_bytes(head_raw, Q6_K, 300, d), fuse_norm=fuse_norm)
    dec2.set_input(xs[0])
    dec2.step()
    assert np.array_equal(bits(dec2.hidden()), bits(eager[0]))
    head = O.deq_raw(head_raw, 300 * d, Q6_K).reshape(300, d).astype(np.float64)
    assert close(dec2.logits.to_vec(stream), D.rmsnorm(want[0], onorm, 1e-6) @ head.T, dot_bar(20))


@pytest.mark.parametrize("head,fuse_norm", [(None, True), (Q6_K, True), (2, True), (Q6_K, False)])
def test_the_launches_of_a_step_are_as_many_as_it_says(F, X, O, head, fuse_norm):
    import ctypes as C
    from ferric_amd.synth import synth_weights
    d, n_layer, stream = 1024, 2, F.Stream()
    layers, _ = _tiny_model(F, X, O, np.random.default_rng(3), n_layer, d, 8, 2, 128, 1536, True)
    w = F.QMatrix.from_bytes(synth_weights(head, 300, d, 77), head, 300, d) if head is not None else None
    dec = X.Qwen3Decoder(X.Qwen3Cfg(d, 8, 2, 128, 1536), layers, max_len=4, stream=stream, output_norm=F.Tensor.from_vec(np.ones(d, np.float32), (d,)) if head is not None else None,
                         lm_head=w, fuse_norm=fuse_norm)
    dec.set_input(np.ones(d, np.float32))
    dec.step()
    hip, graph, nodes = C.CDLL("libamdhip64.so.7"), C.c_void_p(), C.c_size_t()
    stream.synchronize()
    assert hip.hipStreamBeginCapture(stream.handle, 2) == 0
    dec.step()
    assert hip.hipStreamEndCapture(stream.handle, C.byref(graph)) == 0
    assert hip.hipGraphGetNodes(graph, None, C.byref(nodes)) == 0
    hip.hipGraphDestroy(graph)
    assert nodes.value == n_layer * dec.launches_per_layer + dec.launches_per_token_extra


# ---------------------------------------------------------------- the other arms of the layer (qwen3.rs:857-863, 917-938, 953-958, 1015-1020)

def test_mul_sigmoid_and_geglu(F, X, D):
    rng = np.random.default_rng(31)
    T = lambda a: F.Tensor.from_vec(a, a.shape)
    # magnitudes from 1e-3 to 40, both signs, the saturated ends, zero; sizes that do not fill a workgroup
    for n in (1, 255, 5120, 12345):
        a = (rng.standard_normal(n) * 3).astype(np.float32)
        g = (rng.standard_normal(n) * rng.choice([1e-3, 1.0, 10.0, 40.0], n)).astype(np.float32)
        g[:1] = 0.0
        got = X.mul_sigmoid(T(a.reshape(1, n)), T(g.reshape(1, n))).to_vec()
        want = a.astype(np.float64) * D.sigmoid(g)
        # expf and the division are each good to an ulp or two: 1e-6 of the value
        assert (np.abs(got.reshape(-1) - want) <= 1e-6 * np.abs(want) + 1e-37).all(), n
    out_in_place = T(np.ones((1, 64), np.float32))
    F._lib.check(F._lib.load().fhip_mul_sigmoid(out_in_place.buf.ptr, T(np.zeros((1, 64), np.float32)).buf.ptr, 64, out_in_place.buf.ptr, None))
    assert np.array_equal(out_in_place.to_vec(), np.full(64, 0.5, np.float32))
    for t, d in ((1, 1), (1, 17408), (3, 1000), (5, 7)):
        gu = (rng.standard_normal((t, 2 * d)) * rng.choice([0.01, 1.0, 4.0, 30.0], (t, 2 * d))).astype(np.float32)
        gu[0, 0] = 0.0
        got = X.geglu(T(gu)).to_vec().reshape(t, d)
        want = D.gelu_mul(gu.astype(np.float64), d)
        # tanhf to a few ulp, and 1 + tanh cancels for very negative gates, where the value itself is below 1e-6 |v u|
        assert (np.abs(got - want) <= 2e-6 * np.abs(gu[:, :d].astype(np.float64) * gu[:, d:]) + 1e-37).all(), (t, d)
    lib = F._lib.load()
    assert lib.fhip_geglu(None, 1, 8, None, None) != 0 and b"NULL" in lib.fhip_last_error()
    assert lib.fhip_mul_sigmoid(None, None, 0, None, None) == 0          # nothing to do


def _arm_model(F, X, O, rng, n_layer, d, nh, nkv, hd, n_ff, arms):
    """_tiny_model with the optional members of each layer: arms is a list (one per layer) of sets out of
    {"gate", "post", "nope", "window", "base"}."""
    from ferric_amd.synth import synth_weights
    from oracle import decode_oracle as D
    layers, olayers = _tiny_model(F, X, O, rng, n_layer, d, nh, nkv, hd, n_ff, True)
    T = lambda a: F.Tensor.from_vec(a, a.shape)
    for il, (l, ol, arm) in enumerate(zip(layers, olayers, arms)):
        if "gate" in arm:
            b = synth_weights(Q4_K, nh * hd, d, 900 + il)
            l.attn_gate = F.QMatrix.from_bytes(b, Q4_K, nh * hd, d)
            ol.attn_gate = O.deq_raw(b, nh * hd * d, Q4_K).reshape(nh * hd, d).astype(np.float64)
        if "post" in arm:
            pa, pf = (rng.random(d) + 0.5).astype(np.float32), (rng.random(d) + 0.5).astype(np.float32)
            l.post_attn_norm, l.post_ffn_norm, ol.post_attn_norm, ol.post_ffn_norm = T(pa), T(pf), pa, pf
        if "nope" in arm:
            l.rope = ol.rope = False
        if "window" in arm:
            l.window = ol.window = 3
        if "base" in arm:
            l.rope_base = ol.rope_base = 1e4
    return layers, olayers


POST = {"post_norm_eps": 1e-8}


@pytest.mark.parametrize("name,arms,cfg_kw,without,fuse", [
    ("gated attention", [{"gate"}, set(), {"gate"}], {}, ([set()] * 3, {}), True),
    ("gated attention, launches apart", [{"gate"}, {"gate"}, set()], {}, ([set()] * 3, {}), False),
    ("post-norms with their own epsilon", [{"post"}] * 3, POST, ([set()] * 3, {}), True),
    ("post-norms, launches apart", [{"post"}] * 3, POST, ([set()] * 3, {}), False),
    ("local and global layers, NoPE on the global ones", [{"window", "base", "post"}, {"nope", "post"}, {"window", "base", "post"}],
     dict(POST, attn_softcap=30.0), ([{"post"}] * 3, POST), True),
    ("the same, launches apart", [{"window", "base", "post"}, {"nope", "post"}, {"window", "base", "post"}],
     dict(POST, attn_softcap=30.0), ([{"post"}] * 3, POST), False),
    ("GEGLU on post-normed layers", [{"post"}] * 3, dict(POST, geglu=True), ([{"post"}] * 3, POST), True),
    ("GEGLU, launches apart", [{"post"}] * 3, dict(POST, geglu=True), ([{"post"}] * 3, POST), False),
    ("everything at once", [{"gate", "post", "window"}, {"gate", "post", "nope"}, {"post", "base"}],
     dict(POST, geglu=True, attn_softcap=50.0), ([{"post"}] * 3, POST), True),
])
def test_decoder_arms_match_the_oracle_and_replay_as_a_graph(F, X, O, D, name, arms, cfg_kw, without, fuse, precision):
    n_layer, d, nh, nkv, hd, n_ff, steps = 3, 1024, 8, 2, 128, 1536, 6
    cfg = X.Qwen3Cfg(d, nh, nkv, hd, n_ff, eps=1e-6, rope_base=1e6, **cfg_kw)
    rng = np.random.default_rng(8)
    layers, olayers = _arm_model(F, X, O, rng, n_layer, d, nh, nkv, hd, n_ff, arms)
    xs = (np.random.default_rng(9).standard_normal((steps, d)) * 0.5).astype(np.float32)

    def oracle_steps(ols, c):
        kcs, vcs = [[] for _ in ols], [[] for _ in ols]
        out = []
        for pos in range(steps):
            x = xs[pos].astype(np.float64)
            for l, kc, vc in zip(ols, kcs, vcs):
                x = D.apply_layer(x, l, kc, vc, pos, c)
            out.append(x)
        return out
    want = oracle_steps(olayers, cfg)
    # as the default arm's test: <= 20 times the bar of one dot product, of the step's largest hidden value
    bar = dot_bar(20)
    # The bar tells the arm from its absence: the oracle without it (same weights and norms) lies five bars away or more at some step.
    _, oplain = _arm_model(F, X, O, np.random.default_rng(8), n_layer, d, nh, nkv, hd, n_ff, without[0])
    plain = oracle_steps(oplain, X.Qwen3Cfg(d, nh, nkv, hd, n_ff, eps=1e-6, rope_base=1e6, **without[1]))
    assert max(np.abs(a - b).max() / np.abs(a).max() for a, b in zip(want, plain)) > 5 * bar, name
    stream = F.Stream()
    dec = X.Qwen3Decoder(cfg, layers, max_len=steps + 2, stream=stream, fuse_norm=fuse, fuse_attn=fuse)
    eager = []
    for pos in range(steps):
        dec.set_input(xs[pos])
        dec.step()
        eager.append(dec.hidden())
        assert close(eager[-1], want[pos], bar), (name, pos)
    dec.set_pos(0)
    dec.capture()
    for pos in range(steps):
        dec.set_input(xs[pos])
        dec.step_graph()
        assert np.array_equal(bits(dec.hidden()), bits(eager[pos])), (name, pos)


@pytest.mark.parametrize("kv_fmt,arms,cfg_kw", [(0, [set()] * 3, {}), (1, [set()] * 3, {}), (2, [set()] * 3, {}),
                                                (0, [{"gate", "post", "window"}, {"gate", "post", "nope"}, {"post", "base"}],
                                                 dict(POST, geglu=True, attn_softcap=50.0))])
def test_decoder_on_a_block_quantized_cache(F, X, O, D, kv_fmt, arms, cfg_kw, precision):
    """The quantized arm of the layer (qwen3.rs:906-912): K and V rows stored as Q8_0 / Q4_0 / Q4_1 blocks, attention over what
    they dequantize to. The oracle quantizes its own f64 rows (rounded to f32) the same way. Same bar as the f32 cache; and the
    quantized cache is live: what the device cache dequantizes to is the oracle's dequantized rows (the hidden state itself
    moves by less than the bar between an f32 and a quantized cache on this model, so it cannot tell)."""
    n_layer, d, nh, nkv, hd, n_ff, steps = 3, 1024, 8, 2, 128, 1536, 6
    cfg = X.Qwen3Cfg(d, nh, nkv, hd, n_ff, eps=1e-6, rope_base=1e6, **cfg_kw)
    ocfg = X.Qwen3Cfg(d, nh, nkv, hd, n_ff, eps=1e-6, rope_base=1e6, **cfg_kw)
    ocfg.kv_fmt = kv_fmt
    layers, olayers = _arm_model(F, X, O, np.random.default_rng(8), n_layer, d, nh, nkv, hd, n_ff, arms)
    xs = (np.random.default_rng(9).standard_normal((steps, d)) * 0.5).astype(np.float32)

    def oracle_steps(c):
        kcs, vcs = [[] for _ in olayers], [[] for _ in olayers]
        out = []
        for pos in range(steps):
            x = xs[pos].astype(np.float64)
            for l, kc, vc in zip(olayers, kcs, vcs):
                x = D.apply_layer(x, l, kc, vc, pos, c)
            out.append(x)
        return out, kcs
    want, kcs = oracle_steps(ocfg)
    bar = dot_bar(20)
    stream = F.Stream()
    dec = X.Qwen3Decoder(cfg, layers, max_len=steps + 2, stream=stream, kv_fmt=kv_fmt)
    eager = []
    for pos in range(steps):
        dec.set_input(xs[pos])
        dec.step()
        eager.append(dec.hidden())
        assert close(eager[-1], want[pos], bar), (kv_fmt, pos)
    # the first layer's key cache against the oracle's dequantized rows: the same blocks up to codes that sat near a rounding
    # boundary (what is quantized differs between the mat-vec kernel and the f64 oracle by up to the dot-product bar, a few
    # per cent of a Q8_0 step): never more than one step off, and few of them off at all
    got = dec.caches[0][0].dequantize(stream).to_vec(stream).reshape(steps, nkv * hd)
    ref = np.stack(kcs[0])
    step = np.abs(ref).reshape(steps, -1, 32).max(axis=2) / (127 if kv_fmt == 0 else 7)
    off = np.abs(got - ref).reshape(steps, -1, 32)
    assert (off <= 1.01 * step[:, :, None] + 1e-6).all() and (off > 1e-4 * step[:, :, None] + 1e-6).mean() < 0.1
    dec.set_pos(0)
    dec.capture()
    for pos in range(steps):
        dec.set_input(xs[pos])
        dec.step_graph()
        assert np.array_equal(bits(dec.hidden()), bits(eager[pos])), (kv_fmt, pos)


@pytest.mark.parametrize("name,arms,cfg_kw,kv_fmt", [
    ("default arm", [set()] * 3, {}, None),
    ("every arm", [{"gate", "post", "window"}, {"gate", "post", "nope"}, {"post", "base"}], dict(POST, geglu=True, attn_softcap=50.0), None),
    ("post-normed, Q8_0 cache", [{"post"}] * 3, POST, 0),
])
def test_prefill_of_a_prompt_block_then_decode(F, X, O, D, name, arms, cfg_kw, kv_fmt, precision):
    """forward_cached for t > 1 (qwen3.rs:917-930 inside :979-1052): a block of prompt rows through the whole stack in one pass
    per layer -- projections for all rows at once, causal attention over the cache -- equals the oracle run token by token (a
    causal stack is the same function either way). Two blocks (7 rows, then 5 against the 7 cached: the chunked case), then
    single-token steps on the cache the prefill left. precise=True (the f32-grade projections) is held to the decode step's
    bar; the bf16 matrix-core projections (operands rounded to 8 bits of mantissa, three layers deep) to a median of 5e-3 of the
    largest hidden value."""
    n_layer, d, nh, nkv, hd, n_ff = 3, 1024, 8, 2, 128, 1536
    blocks, steps = (7, 5), 3
    total = sum(blocks) + steps
    cfg = X.Qwen3Cfg(d, nh, nkv, hd, n_ff, eps=1e-6, rope_base=1e6, **cfg_kw)
    ocfg = X.Qwen3Cfg(d, nh, nkv, hd, n_ff, eps=1e-6, rope_base=1e6, **cfg_kw)
    ocfg.kv_fmt = kv_fmt
    layers, olayers = _arm_model(F, X, O, np.random.default_rng(8), n_layer, d, nh, nkv, hd, n_ff, arms)
    xs = (np.random.default_rng(10).standard_normal((total, d)) * 0.5).astype(np.float32)
    kcs, vcs = [[] for _ in olayers], [[] for _ in olayers]
    want = []
    for pos in range(total):
        x = xs[pos].astype(np.float64)
        for l, kc, vc in zip(olayers, kcs, vcs):
            x = D.apply_layer(x, l, kc, vc, pos, ocfg)
        want.append(x)
    want = np.stack(want)
    stream = F.Stream()
    # the synthetic default-arm stack amplifies perturbations (its hidden values reach 1e5 and a change of 1e-3 in a branch
    # moves them by their own size): it checks the f32-grade route only; the post-normed stacks, whose branches are rescaled
    # to RMS 1 at every add, carry the bf16 route as well
    routes = ((True, dot_bar(20)), (False, 1.5e-2)) if all("post" in a for a in arms) else ((True, dot_bar(20)),)
    rel = lambda got, w: float(np.abs(np.asarray(got, np.float64) - w).max() / np.abs(w).max())
    for precise, bar in routes:
        dec = X.Qwen3Decoder(cfg, layers, max_len=total + 1, stream=stream, kv_fmt=kv_fmt)
        errs, at = [], 0
        for n in blocks:
            got = dec.prefill(xs[at:at + n], precise=precise)
            errs += [rel(got[r], want[at + r]) for r in range(n)]
            at += n
        assert dec._all_caches()[0].len == at
        for pos in range(at, total):                  # decode continues on the cache and the position the prefill left
            dec.set_input(xs[pos])
            dec.step()
            errs.append(rel(dec.hidden(), want[pos]))
        errs = np.array(errs)
        if precise:
            assert (errs <= bar).all(), (name, errs.max())
        else:
            # With operands rounded to bf16 most rows land at 2e-3 .. 3e-3. The synthetic stack's attention is close to a hard
            # maximum over the keys (unnormalised scores in the tens), so on a few rows a perturbation of that size changes which
            # key wins and the row's hidden state with it: the median and three rows in four are held, not every row.
            assert np.median(errs) <= 5e-3 and (errs <= bar).mean() >= 0.75, (name, np.sort(errs)[-4:])
    with pytest.raises(AssertionError, match="exceed the capacity"):
        dec.prefill(xs[:2])


def test_rows_rounded_to_bf16_by_their_producer(F, X):
    """fhip_add_rmsnorm_bf16 and fhip_causal_attention_bf16 store the bits fhip_cvt_f32_bf16 makes of their f32 forms (both row kernels, a
    width that is not a multiple of four, NaN and infinities; both head sizes and workgroup shapes); fhip_ffn_bf16 on converted rows has
    the bits of fhip_ffn_coop."""
    rng = np.random.default_rng(3)
    lib, chk = F._lib.load(), F._lib.check
    T = lambda a: F.Tensor.from_vec(a, a.shape)
    E = F.Tensor.empty
    raw = lambda t: t.to_vec().view(np.uint16 if t.dtype == np.uint16 else np.uint32)
    for rows, d in ((3, 5120), (7, 130), (5, 512), (2, 9001), (1, 3)):
        a, b, w = (rng.standard_normal(n).astype(np.float32) for n in ((rows, d), (rows, d), (d,)))
        a[0, 0], w[-1] = np.inf, np.nan
        at, bt, wt = T(a), T(b), T(w)
        for resid in (None, bt):
            f, s0, s1, h = E((rows, d)), E((rows, d)), E((rows, d)), E((rows, d), np.uint16)
            if resid is None:
                chk(lib.fhip_rmsnorm(at.buf.ptr, wt.buf.ptr, rows, d, 1e-6, f.buf.ptr, None))
                chk(lib.fhip_add_rmsnorm_bf16(at.buf.ptr, None, wt.buf.ptr, rows, d, 1e-6, None, h.buf.ptr, None))
            else:
                chk(lib.fhip_add_rmsnorm(at.buf.ptr, bt.buf.ptr, wt.buf.ptr, rows, d, 1e-6, s0.buf.ptr, f.buf.ptr, None))
                chk(lib.fhip_add_rmsnorm_bf16(at.buf.ptr, bt.buf.ptr, wt.buf.ptr, rows, d, 1e-6, s1.buf.ptr, h.buf.ptr, None))
                assert np.array_equal(raw(s0), raw(s1))
            assert np.array_equal(raw(f.cvt_bf16()), raw(h)), (rows, d)
    for t, s, nh, nkv, hd in ((33, 70, 10, 2, 128), (100, 100, 4, 4, 64), (512, 512, 136, 8, 64), (520, 520, 104, 8, 128)):
        q, k, v = (T(rng.standard_normal(n).astype(np.float32)) for n in ((t, nh * hd), (s, nkv * hd), (s, nkv * hd)))
        f, h = E((t, nh * hd)), E((t, nh * hd), np.uint16)
        chk(lib.fhip_causal_attention(q.buf.ptr, k.buf.ptr, v.buf.ptr, t, s, nh, nkv, hd, 0, 0.0, f.buf.ptr, None))
        chk(lib.fhip_causal_attention_bf16(q.buf.ptr, k.buf.ptr, v.buf.ptr, t, s, nh, nkv, hd, 0, 0.0, h.buf.ptr, None))
        assert np.array_equal(raw(f.cvt_bf16()), raw(h)), (t, hd)
    from ferric_amd.synth import synth_weights
    d, ff = 512, 768
    gu, down = (F.QMatrix.from_bytes(synth_weights(Q4_K, r, c, 1), Q4_K, r, c) for r, c in ((2 * ff, d), (d, ff)))
    for t in (7, 32, 33, 200):
        x = T(rng.standard_normal((t, d)).astype(np.float32))
        ws, y = F.DeviceBuffer(lib.fhip_ffn_coop_ws_bytes(gu.handle, down.handle, t)), E((t, d))
        xb = x.cvt_bf16()
        chk(lib.fhip_ffn_bf16(gu.handle, down.handle, xb.buf.ptr, None, t, y.buf.ptr, ws.ptr, None))
        assert np.array_equal(raw(x.ffn_coop(gu, down)), raw(y)), t
        # gate|up in memory: the bits of the steps one by one
        g, y2 = E((t, 2 * ff)), E((t, d))
        chk(lib.fhip_ffn_bf16(gu.handle, down.handle, xb.buf.ptr, g.buf.ptr, t, y2.buf.ptr, ws.ptr, None))
        h2 = xb.gemm_q_bf16(gu)
        assert np.array_equal(raw(h2), raw(g)), t
        f = E((t, ff))
        chk(lib.fhip_swiglu(h2.buf.ptr, t, ff, f.buf.ptr, None))
        assert np.array_equal(raw(f.cvt_bf16().gemm_q_bf16(down)), raw(y2)), t
    one = E((1, 8), np.uint16)
    assert lib.fhip_add_rmsnorm_bf16(wt.buf.ptr, bt.buf.ptr, wt.buf.ptr, 1, 2, 1e-6, None, one.buf.ptr, None) != 0       # a sum asked for and no place for it
    assert lib.fhip_causal_attention_bf16(q.buf.ptr, k.buf.ptr, v.buf.ptr, 1, 1, 1, 1, 64, 0, 0.0, one.buf.ptr.value + 8, None) != 0
    assert b"16-byte aligned" in lib.fhip_last_error()


@pytest.mark.parametrize("nh,nkv,hd,seed", [(8, 2, 128, 0), (8, 4, 64, 1)])
def test_a_prefill_stack_is_as_near_f64_with_either_attention_kernel(F, X, O, D, monkeypatch, nh, nkv, hd, seed):
    """A block of prompt rows behind another through four layers, the bf16 route, with fhip_causal_attention's kernel and with the f32 one in its
    place. A last bit of the attention moves some bf16 roundings of its rows by one place, so the two runs part, but a value that is moved lies
    half way between its neighbours: either rounding is as far from f64. Held to 3 % of the 2-norm of the error: at 200 .. 700 rows of four
    layers (d 2048 and 5120) the two came within 0.13 % of each other while the hidden rows were 2.5e-3 .. 3e-3 apart. Weights of mean zero, as
    trained ones: a common part in them would carry everything and hide the difference."""
    n_layer, d, n_ff, blocks = 4, 512, 768, (40, 80)
    rng = np.random.default_rng(20 + seed)
    cfg = X.Qwen3Cfg(d, nh, nkv, hd, n_ff, eps=1e-6, rope_base=1e6)
    T = lambda a: F.Tensor.from_vec(a, a.shape)

    def weight(r, c):                                            # Q8_0, normal, rows of norm about 1
        codes = np.clip(np.rint(rng.standard_normal((r * c // 32, 32)) * 40), -127, 127).astype(np.int8)
        scale = np.full((r * c // 32, 1), 1 / (40 * np.sqrt(c)), np.float16)
        raw = np.concatenate([scale.view(np.uint8), codes.view(np.uint8)], axis=1).reshape(-1)
        return F.QMatrix.from_bytes(raw, F.Q8_0, r, c), (scale.astype(np.float64) * codes).reshape(r, c)
    layers, olayers = [], []
    for _ in range(n_layer):
        (wqkv, oqkv), (wo, oo), (gu, ogu), (dn, odn) = (weight(*s) for s in (((nh + 2 * nkv) * hd, d), (d, nh * hd), (2 * n_ff, d), (d, n_ff)))
        an, fn, qn, kn = ((rng.random(n) + 0.5).astype(np.float32) for n in (d, d, hd, hd))
        layers.append(X.Qwen3Layer(T(an), wqkv, wo, T(fn), gu, dn, T(qn), T(kn)))
        olayers.append(D.Layer(attn_norm=an, wqkv=oqkv, wo=oo, ffn_norm=fn, gate_up=ogu, down=odn, q_norm=qn, k_norm=kn))
    xs = np.random.default_rng(30 + seed).standard_normal((sum(blocks), d)).astype(np.float32)
    kcs, vcs = [[] for _ in olayers], [[] for _ in olayers]
    want = []
    for pos, row in enumerate(xs):
        x = row.astype(np.float64)
        for l, kc, vc in zip(olayers, kcs, vcs):
            x = D.apply_layer(x, l, kc, vc, pos, cfg)
        want.append(np.asarray(x).reshape(-1))
    want = np.stack(want)

    def run():
        dec = X.Qwen3Decoder(cfg, layers, max_len=sum(blocks), stream=F.Stream())
        return np.concatenate([dec.prefill(xs[:blocks[0]]), dec.prefill(xs[blocks[0]:])])
    cut = run()
    lib = F._lib.load()
    monkeypatch.setattr(lib, "fhip_causal_attention_bf16", lambda *a: lib.fhip_causal_attention_f32_products(*a[:10], 1, *a[10:]))
    f32 = run()
    err = lambda got: np.linalg.norm(got - want) / np.linalg.norm(want)
    print("error against f64", err(cut), err(f32), "apart", np.linalg.norm(cut - f32) / np.linalg.norm(want))
    assert not np.array_equal(bits(cut), bits(f32))              # (the two kernels did run)
    assert err(f32) <= 1e-2 and err(cut) <= 1.03 * err(f32)
