"""fhip_causal_attention (prefill / chunked prefill / windowed / softcapped causal attention on the matrix instructions)
through the C ABI against the f64 oracle. Floating point: the bar is 1e-5 of the largest expected output, the bar of the
single-query attention tests; a row that sees one key only must return that key's value row exactly."""
import numpy as np
import pytest

from conftest import bits

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def D():
    from oracle import decode_oracle
    return decode_oracle


@pytest.fixture(scope="module")
def X(F):
    from ferric_amd import decode
    return decode


def run(F, X, D, t, s, nh, nkv, hd, window=0, cap=0.0, seed=0, scale=1.0):
    rng = np.random.default_rng(seed)
    q = (rng.standard_normal((t, nh * hd)) * scale).astype(np.float32)
    k = rng.standard_normal((s, nkv * hd)).astype(np.float32)
    v = rng.standard_t(3, (s, nkv * hd)).astype(np.float32)
    T = lambda a: F.Tensor.from_vec(a, a.shape)
    got = X.causal_attention(T(q), T(k), T(v), nh, nkv, window, cap).to_vec().reshape(t, nh * hd)
    want = D.causal_attention(q, k, v, nh, nkv, window, cap)
    err = np.abs(got - want).max() / np.abs(want).max()
    assert err <= 1e-5, (t, s, nh, nkv, hd, window, cap, err)
    return got, q, k, v


def test_shapes_groups_and_ragged_ends(F, X, D):
    # stateless prefill (s == t): one row, less than a tile, exactly one, ragged, several query blocks; both head sizes;
    # group sizes 1, 2, 5, 8; then t rows against a longer cache (chunked prefill / a prefix-cached suffix), off inside a tile
    for i, (t, s, nh, nkv, hd) in enumerate([(1, 1, 4, 2, 64), (7, 7, 4, 4, 128), (32, 32, 8, 4, 64), (33, 33, 10, 2, 128), (100, 100, 8, 1, 64),
                                             (130, 130, 5, 1, 128), (257, 257, 16, 2, 128), (300, 300, 6, 3, 64),
                                             (1, 40, 8, 2, 128), (5, 70, 8, 2, 64), (64, 200, 10, 2, 128), (90, 91, 4, 2, 128), (31, 160, 8, 8, 64)]):
        got, q, k, v = run(F, X, D, t, s, nh, nkv, hd, seed=i)
        if s == t:          # the first row sees its own key only
            g = nh // nkv
            assert np.array_equal(bits(got[0].reshape(nh, hd)), bits(np.repeat(v[0].reshape(nkv, hd), g, axis=0)))


def test_window_and_softcap(F, X, D):
    for i, (t, s, nh, nkv, hd, w, cap) in enumerate([(70, 70, 4, 2, 64, 16, 0.0), (70, 70, 4, 2, 128, 1, 0.0), (150, 150, 8, 2, 128, 33, 0.0),
                                                     (40, 300, 8, 2, 64, 100, 0.0), (150, 150, 8, 2, 128, 0, 30.0), (96, 130, 5, 1, 128, 40, 50.0),
                                                     (50, 50, 4, 2, 64, 1000, 0.0)]):
        got, q, k, v = run(F, X, D, t, s, nh, nkv, hd, w, cap, seed=20 + i, scale=3.0)
        if w == 1:          # a window of one key: every row returns its own value row
            g = nh // nkv
            assert np.array_equal(bits(got.reshape(t, nh, hd)), bits(np.repeat(v[s - t:].reshape(t, nkv, hd), g, axis=1)))


def test_a_prefill_sized_block_on_sampled_rows(F, X, D):
    """2048 tokens of the 40 / 8-head x 128 model in one launch; the oracle on a sample of rows (first, tile edges, last)."""
    t, nh, nkv, hd = 2048, 40, 8, 128
    rng = np.random.default_rng(5)
    q = rng.standard_normal((t, nh * hd)).astype(np.float32)
    k = rng.standard_normal((t, nkv * hd)).astype(np.float32)
    v = rng.standard_normal((t, nkv * hd)).astype(np.float32)
    T = lambda a: F.Tensor.from_vec(a, a.shape)
    qt, kt, vt = T(q), T(k), T(v)
    got = X.causal_attention(qt, kt, vt, nh, nkv).to_vec().reshape(t, nh * hd)
    for r in (0, 1, 31, 32, 127, 128, 1000, 1023, 1024, 2047):
        want = D.decode_attention(q[r], k[:r + 1], v[:r + 1], nh, nkv)[0]
        assert np.abs(got[r] - want).max() <= 1e-5 * np.abs(want).max(), r
    again = X.causal_attention(qt, kt, vt, nh, nkv).to_vec().reshape(t, nh * hd)
    assert np.array_equal(bits(got), bits(again))                 # no atomics, a fixed order: the same bits every run
    # a row of the block equals the single-query op on the same cache prefix to the two kernels' rounding
    r = 777
    cache = type("C", (), {})()
    cache.k, cache.v, cache.cap, cache.width, cache.len = kt, vt, t, nkv * hd, r + 1
    one = X.decode_attention(T(q[r:r + 1]), cache, nh, nkv, length=r + 1).to_vec()
    assert np.abs(one - got[r]).max() <= 2e-6 * np.abs(got[r]).max()


def test_argument_checks(F, X):
    lib = F._lib.load()
    a = F.Tensor.from_vec(np.zeros((4, 256), np.float32), (4, 256))
    assert lib.fhip_causal_attention(a.buf.ptr, a.buf.ptr, a.buf.ptr, 4, 3, 4, 4, 64, 0, 0.0, a.buf.ptr, None) != 0
    assert b"cannot be shorter than the query block" in lib.fhip_last_error()          # nn.rs:73
    assert lib.fhip_causal_attention(a.buf.ptr, a.buf.ptr, a.buf.ptr, 4, 4, 4, 3, 64, 0, 0.0, a.buf.ptr, None) != 0
    assert lib.fhip_causal_attention(a.buf.ptr, a.buf.ptr, a.buf.ptr, 4, 4, 8, 8, 32, 0, 0.0, a.buf.ptr, None) != 0
    assert b"head_dim must be 64 or 128" in lib.fhip_last_error()
    assert lib.fhip_causal_attention(None, a.buf.ptr, a.buf.ptr, 4, 4, 4, 4, 64, 0, 0.0, a.buf.ptr, None) != 0
    assert lib.fhip_causal_attention(None, None, None, 0, 0, 4, 4, 64, 0, 0.0, None, None) == 0       # nothing to do


@pytest.mark.parametrize("t,s,nh,nkv,hd,w,cap,vscale", [(1, 1, 2, 1, 64, 0, 0.0, 1.0), (33, 70, 10, 2, 128, 0, 0.0, 1e30), (130, 130, 4, 4, 64, 17, 0.0, 1e-30),
                                                        (65, 300, 5, 1, 128, 0, 30.0, 1.0), (1100, 1100, 64, 8, 64, 0, 0.0, 1.0)])
def test_f32_products_beside_the_cut_ones(F, X, D, t, s, nh, nkv, hd, w, cap, vscale):
    # both kernels at the bar of this file, f32 and bf16 rows of the f32 one, and the two beside each other: each is within a few f32
    # roundings of sums of s terms (4e-6 of the largest output: sums of up to 1100 terms, 2e-6 each at the most). Values far from 1 keep their 24 bits in three cuts; 1100 rows of 64 heads take
    # the workgroups of eight waves.
    rng = np.random.default_rng(t + s)
    q = rng.standard_normal((t, nh * hd)).astype(np.float32)
    k = rng.standard_normal((s, nkv * hd)).astype(np.float32)
    v = (rng.standard_normal((s, nkv * hd)) * vscale).astype(np.float32)
    T = lambda a: F.Tensor.from_vec(a, a.shape)
    tq, tk, tv = T(q), T(k), T(v)
    cut = X.causal_attention(tq, tk, tv, nh, nkv, w, cap).to_vec().reshape(t, nh * hd)
    lib = F._lib.load()
    out, half = T(np.zeros((t, nh * hd), np.float32)), T(np.zeros((t, nh * hd), np.float32))
    args = (tq.buf.ptr, tk.buf.ptr, tv.buf.ptr, t, s, nh, nkv, hd, w, cap)
    assert lib.fhip_causal_attention_f32_products(*args, 0, out.buf.ptr, None) == 0
    assert lib.fhip_causal_attention_f32_products(*args, 1, half.buf.ptr, None) == 0
    f32 = out.to_vec().reshape(t, nh * hd)
    top = np.abs(f32).max()
    assert np.abs(cut - f32).max() <= 4e-6 * top
    if t <= 130:
        want = D.causal_attention(q, k, v, nh, nkv, w, cap)
        for got in (cut, f32):
            assert np.abs(got - want).max() <= 1e-5 * np.abs(want).max()
    b = f32.view(np.uint32).astype(np.uint64)
    rounded = ((b + 0x7FFF + ((b >> 16) & 1)) >> 16).astype(np.uint16)
    assert np.array_equal(half.to_vec().view(np.uint16).reshape(-1)[:t * nh * hd], rounded.reshape(-1))
    assert lib.fhip_causal_attention_f32_products(*args[:3], s + 1, s, *args[5:], 0, out.buf.ptr, None) != 0


@pytest.mark.parametrize("t,nh,nkv,hd,w,cap", [(1100, 64, 8, 64, 0, 0.0), (800, 64, 8, 128, 0, 30.0), (1100, 64, 16, 64, 77, 0.0), (1100, 64, 4, 128, 300, 0.0)])
def test_f32_products_by_four_waves(F, X, t, nh, nkv, hd, w, cap):
    # all rows at once give a wave its 16 rows, few of them four waves of work: the same products in the same order, so the same bits.
    # Blocks of 1, 15 .. 17, 33 and 70 rows whose keys end at, before and behind the ends of tiles and of steps of two tiles; values of
    # both signs and of a wide range.
    lib, T = F._lib.load(), (lambda a: F.Tensor.from_vec(a, a.shape))
    rng = np.random.default_rng(t + hd + w)
    q = rng.standard_normal((t, nh * hd)).astype(np.float32) * 2
    k = rng.standard_normal((t, nkv * hd)).astype(np.float32)
    v = (rng.standard_normal((t, nkv * hd)) * np.exp(3 * rng.standard_normal((t, 1)))).astype(np.float32)

    def rows(first, end, half):
        tq, tk, tv = T(np.ascontiguousarray(q[first:end])), T(np.ascontiguousarray(k[:end])), T(np.ascontiguousarray(v[:end]))
        out = T(np.zeros((end - first, nh * hd), np.float32))
        assert lib.fhip_causal_attention_f32_products(tq.buf.ptr, tk.buf.ptr, tv.buf.ptr, end - first, end, nh, nkv, hd, w, cap, int(half), out.buf.ptr, None) == 0
        got = out.to_vec()
        return got.view(np.uint16).reshape(-1)[:got.size].reshape(end - first, -1) if half else got.reshape(end - first, -1)

    for half in (False, True):
        all_rows = rows(0, t, half)
        assert np.abs(all_rows.view(np.uint16 if half else np.uint32)).max() > 0
        for first, end in ((0, 1), (0, 15), (0, 16), (1, 18), (31, 64), (30, 63), (33, 65), (64, 97), (200, 270), (400, 401), (479, 512), (703, 720), (t - 17, t)):
            assert np.array_equal(rows(first, end, half), all_rows[first:end]), (half, first, end)


def both_kernels(F, X, q, k, v, nh, nkv, cap=0.0):
    """[t, nh * hd] of fhip_causal_attention and of fhip_causal_attention_f32_products, f32; the bf16 form of the first has to be its rounding."""
    lib, T, t, s, hd = F._lib.load(), (lambda a: F.Tensor.from_vec(a, a.shape)), q.shape[0], k.shape[0], q.shape[1] // nh
    tq, tk, tv, out, half = T(q), T(k), T(v), T(np.zeros(q.shape, np.float32)), T(np.zeros(q.shape, np.float32))
    cut = X.causal_attention(tq, tk, tv, nh, nkv, 0, cap).to_vec().reshape(q.shape)
    args = (tq.buf.ptr, tk.buf.ptr, tv.buf.ptr, t, s, nh, nkv, hd, 0, cap)
    assert lib.fhip_causal_attention_f32_products(*args, 0, out.buf.ptr, None) == 0
    assert lib.fhip_causal_attention_bf16(*args, half.buf.ptr, None) == 0
    b = cut.view(np.uint32).astype(np.uint64)
    rounded = ((b + 0x7FFF + ((b >> 16) & 1)) >> 16).astype(np.uint16)
    got = half.to_vec().view(np.uint16).reshape(-1)[:cut.size].reshape(cut.shape)
    assert np.array_equal(got[~np.isnan(cut)], rounded[~np.isnan(cut)])
    assert ((got[np.isnan(cut)] & 0x7FFF) > 0x7F80).all()
    return cut, out.to_vec().reshape(q.shape)


# four and eight waves a workgroup at both head sizes (eight from 512 workgroups of 128 rows on)
RANGE_SHAPES = [(70, 130, 10, 2, 128), (70, 130, 4, 4, 64), (200, 200, 256, 32, 128), (1100, 1100, 64, 8, 64)]


@pytest.mark.parametrize("shape", RANGE_SHAPES)
@pytest.mark.parametrize("kind", ["key -inf", "key inf, softcap", "key nan", "scores overflow", "value inf", "value largest", "query nan"])
def test_members_that_three_cuts_do_not_carry(F, X, D, shape, kind):
    """Members beyond the range the bf16 cuts hold: a row that sees one is the f32 kernel's, bit for bit (a NaN a NaN); where the result is finite
    it is the oracle's at the bar of this file; rows that are not computed beside such a one keep their bits."""
    t, s, nh, nkv, hd = shape
    rng = np.random.default_rng(hd + s)
    q = rng.standard_normal((t, nh * hd)).astype(np.float32)
    k = rng.standard_normal((s, nkv * hd)).astype(np.float32)
    v = rng.standard_normal((s, nkv * hd)).astype(np.float32)
    cap, j, off = 0.0, s - 20, s - t
    first = j - off                                             # the first row that sees key j
    if kind == "key -inf":
        q[:, ::hd] = -np.abs(q[:, ::hd]) - 0.1                  # an infinite negative score: weight 0
    if kind == "key inf, softcap":
        cap = 30.0                                              # an infinite score is 30 or -30
    clean, _ = both_kernels(F, X, q, k, v, nh, nkv, cap)
    if kind in ("key -inf", "key inf, softcap"):
        k[j, ::hd] = np.inf
    elif kind == "key nan":
        k[j, ::hd] = np.nan
    elif kind == "scores overflow":
        k[j] *= 1e25
        q[first:] *= 1e25
    elif kind == "value inf":
        v[j, 5::hd] = -np.inf
    elif kind == "value largest":
        v[j] = np.where(v[j] > 0, 1, -1) * np.finfo(np.float32).max
    else:
        q[first:, 7::hd] = np.nan
    cut, f32 = both_kernels(F, X, q, k, v, nh, nkv, cap)
    same = (bits(cut) == bits(f32)) | (np.isnan(cut) & np.isnan(f32))
    assert same[first:].all(), np.argwhere(~same[first:])[:4]
    before = first // 16 * 16                                   # the wave that holds row `first` starts there ...
    while before > 0 and (off + before - 1) // 32 >= j // 32:   # ... and the wave before it reads no key of j's tile
        before -= 16
    assert np.array_equal(bits(cut[:before]), bits(clean[:before]))
    if kind in ("key -inf", "key inf, softcap", "value largest"):
        for r in (first, t - 1):
            want = D.decode_attention(q[r], k[:off + r + 1], v[:off + r + 1], nh, nkv, 0, cap)[0]
            assert np.isfinite(want).all() and np.abs(cut[r] - want).max() <= 1e-5 * np.abs(want).max()


@pytest.mark.parametrize("shape", RANGE_SHAPES)
@pytest.mark.parametrize("scale", [1e-33, 1e-36, 3e-38, 1e-41, 1e16])
def test_small_and_large_values_keep_their_bits(F, X, D, shape, scale):
    """V of every magnitude down to f32's subnormals: the cuts hold all of an f32's bits, so the error stays that of f32 sums of up to 1100 terms (4e-6 of
    the largest output, as above) and, for results that are subnormal themselves, half a unit of their last place."""
    t, s, nh, nkv, hd = shape
    rng = np.random.default_rng(hd + s + 1)
    q = rng.standard_normal((t, nh * hd)).astype(np.float32)
    k = rng.standard_normal((s, nkv * hd)).astype(np.float32)
    v = (rng.standard_normal((s, nkv * hd)) * scale).astype(np.float32)
    cut, _ = both_kernels(F, X, q, k, v, nh, nkv)
    for r in (0, t // 2, t - 1):
        want = D.decode_attention(q[r], k[:s - t + r + 1], v[:s - t + r + 1], nh, nkv)[0]
        assert np.abs(cut[r] - want).max() <= 4e-6 * np.abs(want).max() + 2.0 ** -149, (r, np.abs(cut[r] - want).max() / np.abs(want).max())


def split(F, q, k, v, nh, nkv, w=0, cap=0.0):
    """[t, nh * hd] of fhip_causal_attention_split; its bf16 form has to be the rounding of it."""
    lib, T, t, s, hd = F._lib.load(), (lambda a: F.Tensor.from_vec(a, a.shape)), q.shape[0], k.shape[0], q.shape[1] // nh
    need = lib.fhip_causal_attention_ws_bytes(t, s, nh, hd, w)
    assert need, (t, s, nh, hd, w)
    tq, tk, tv, out, half, ws = T(q), T(k), T(v), T(np.zeros(q.shape, np.float32)), T(np.zeros(q.shape, np.float32)), F.DeviceBuffer(need)
    args = (tq.buf.ptr, tk.buf.ptr, tv.buf.ptr, t, s, nh, nkv, hd, w, cap)
    assert lib.fhip_causal_attention_split(*args, 0, out.buf.ptr, ws.ptr, need, None) == 0
    assert lib.fhip_causal_attention_split(*args, 1, half.buf.ptr, ws.ptr, need, None) == 0
    got = out.to_vec().reshape(q.shape)
    b = got.view(np.uint32).astype(np.uint64)
    rounded = ((b + 0x7FFF + ((b >> 16) & 1)) >> 16).astype(np.uint16)
    bf16 = half.to_vec().view(np.uint16).reshape(-1)[:got.size].reshape(got.shape)
    assert np.array_equal(bf16[~np.isnan(got)], rounded[~np.isnan(got)]) and ((bf16[np.isnan(got)] & 0x7FFF) > 0x7F80).all()
    assert lib.fhip_causal_attention_split(*args, 0, out.buf.ptr, ws.ptr, need - 1, None) != 0        # too little scratch
    assert lib.fhip_causal_attention_split(*args, 0, out.buf.ptr, None, 0, None) == 0                 # none: the keys in one piece
    whole = out.to_vec().reshape(q.shape)
    assert lib.fhip_causal_attention(*args, out.buf.ptr, None) == 0
    assert np.array_equal(bits(whole), bits(out.to_vec().reshape(q.shape)))
    return got, whole


# one row, ragged rows and tiles, the last range a single tile, 32 ranges, more workgroups than CUs, ranges that the first waves of a block do not see, a window that leaves
# a block's first keys out, the softcap
@pytest.mark.parametrize("t,s,nh,nkv,hd,w,cap", [(1, 193, 2, 1, 64, 0, 0.0), (95, 722, 8, 8, 128, 0, 0.0), (33, 1057, 4, 4, 64, 0, 30.0), (17, 2100, 1, 1, 128, 0, 0.0),
                                                 (509, 809, 40, 8, 128, 0, 0.0), (129, 500, 10, 2, 64, 0, 0.0), (200, 640, 6, 3, 128, 333, 0.0), (160, 160, 8, 1, 128, 0, 50.0)])
def test_keys_split_between_workgroups(F, X, D, t, s, nh, nkv, hd, w, cap):
    rng = np.random.default_rng(t + s)
    q = rng.standard_normal((t, nh * hd)).astype(np.float32)
    k = rng.standard_normal((s, nkv * hd)).astype(np.float32)
    v = rng.standard_t(3, (s, nkv * hd)).astype(np.float32)
    got, whole = split(F, q, k, v, nh, nkv, w, cap)
    assert np.abs(got - whole).max() <= 4e-6 * np.abs(whole).max()                                    # two f32 sums of up to 2100 terms (2e-6 each at the most)
    off = s - t
    for r in sorted({0, min(15, t - 1), min(16, t - 1), t // 2, t - 1}):
        lo = max(0, off + r + 1 - w) if w else 0
        want = D.decode_attention(q[r], k[lo:off + r + 1], v[lo:off + r + 1], nh, nkv, 0, cap)[0]
        assert np.abs(got[r] - want).max() <= 1e-5 * np.abs(want).max(), r


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("kind", ["key nan", "value inf", "sum past the largest", "key -inf"])
def test_split_keys_that_three_cuts_do_not_carry(F, X, hd, kind):
    """Rows that meet such a member, in a range or only in the sum over ranges, are the f32 kernel's, bit for bit; other rows keep theirs."""
    t, s, nh, nkv = 70, 500, 4, 2
    rng = np.random.default_rng(hd)
    q, k, v = (rng.standard_normal((n, h * hd)).astype(np.float32) for n, h in ((t, nh), (s, nkv), (s, nkv)))
    clean, _ = split(F, q, k, v, nh, nkv)
    j, first = s - 20, t - 20
    if kind == "key nan":
        k[j, ::hd] = np.nan
    elif kind == "value inf":
        v[j, 5::hd] = -np.inf
    elif kind == "key -inf":                                          # a row's only infinite score: weight 0
        q[:, ::hd] = -np.abs(q[:, ::hd]) - 0.1
        k[j, ::hd] = np.inf
    else:
        q[:] = 0                                                      # equal weights: sums of s values of 2^88 * 2^40 pass f32's largest in every range
        v[:] = np.float32(2.0 ** 88)
        first = 0
    got, _ = split(F, q, k, v, nh, nkv)
    lib, T = F._lib.load(), (lambda a: F.Tensor.from_vec(a, a.shape))
    tq, tk, tv, out = T(q), T(k), T(v), T(np.zeros(q.shape, np.float32))
    assert lib.fhip_causal_attention_f32_products(tq.buf.ptr, tk.buf.ptr, tv.buf.ptr, t, s, nh, nkv, hd, 0, 0.0, 0, out.buf.ptr, None) == 0
    f32 = out.to_vec().reshape(q.shape)
    same = (bits(got) == bits(f32)) | (np.isnan(got) & np.isnan(f32))
    assert same[first:].all(), np.argwhere(~same[first:])[:4]
    if kind in ("key nan", "value inf"):
        before = first // 16 * 16
        while before > 0 and (s - t + before - 1) // 32 >= j // 32:
            before -= 16
        assert np.array_equal(bits(got[:before]), bits(clean[:before]))
