"""Prefill dequant-GEMM (bf16 activations, matrix cores) vs the CPU oracle, through the C ABI.

Three bars:
  * against the SAME arithmetic model evaluated in f64 -- activations as given (bf16), weights =
    oracle-dequantized f32 rounded to bf16 (RNE) -- the GPU may differ only by f32 accumulation order:
    max|d| / max|ref| < 2e-5. This is the check that catches a wrong lane/column mapping.
  * the north-star bound |y - y64| <= 1e-3 * ||w_row|| * ||x_t|| against unrounded oracle weights;
  * the reference's own bar for its matrix-unit prefill: max|d| / max|ref| < 6e-2
    (crates/ferric-tensor/examples/coop_q4_k.rs:38).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
Q8_0, Q4_K, Q6_K, Q5_K = 8, 12, 14, 13


def bf16_round(a):
    """f32 -> nearest bf16 (ties to even), returned as (bits uint16, value f32)."""
    u = np.ascontiguousarray(a, np.float32).view(np.uint32).astype(np.uint64)
    r = ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint32)
    return r.astype(np.uint16), (r << 16).astype(np.uint32).view(np.float32)


def run_case(F, O, ty, t, n, k, seed, gen=None):
    from ferric_amd.synth import synth_weights
    w = gen(ty, n, k) if gen else synth_weights(ty, n, k, seed)
    x = np.random.default_rng(seed + 1).standard_normal((t, k)).astype(np.float32)
    xb, xv = bf16_round(x)
    qm = F.QMatrix.from_bytes(w, ty, n, k)
    y = F.Tensor.from_bf16_bits(xb, (t, k)).gemm_q_bf16(qm).to_vec().reshape(t, n)
    wd = O.deq_raw(w, n * k, ty).reshape(n, k)
    _, wb = bf16_round(wd)
    x64 = xv.astype(np.float64)
    model = x64 @ wb.astype(np.float64).T
    scale = max(1e-3, np.abs(model).max())
    assert np.abs(y - model).max() / scale < 2e-5, (ty, t, n, k)
    exact = x64 @ wd.astype(np.float64).T
    bound = 1e-3 * np.linalg.norm(wd.astype(np.float64), axis=1)[None, :] * np.linalg.norm(x64, axis=1)[:, None]
    assert (np.abs(y - exact) <= bound).all(), (ty, t, n, k)
    assert np.abs(y - exact).max() / max(1e-3, np.abs(exact).max()) < 6e-2
    return y


@pytest.mark.parametrize("ty", [Q4_K, Q6_K, Q8_0, Q5_K])
def test_small_and_ragged_shapes(F, O, ty):
    for i, (t, n, k) in enumerate([(1, 32, 256), (8, 256, 256), (33, 100, 512), (64, 96, 768), (100, 300, 1024), (130, 257, 2048)]):
        run_case(F, O, ty, t, n, k, 10 + i)


def test_seeded_random_shapes(F, O):
    # 48 shapes drawn with a fixed seed: any row count on either side of the 32-row kernel switch, output widths that are
    # no multiple of a tile (or of 4: the ordered sum of K-split tiles then stores element by element), 1 to 9 chunks of
    # K -- whatever way the launch is cut, every output meets the oracle
    rng = np.random.default_rng(20240607)
    for i in range(48):
        ty = (Q4_K, Q6_K, Q8_0, Q5_K)[i % 4] if i >= 36 else (Q4_K, Q6_K, Q8_0)[i % 3]
        t = int(rng.integers(1, 300)) if i % 4 else int(rng.integers(1, 33))
        n = int(rng.integers(1, 700))
        k = int(rng.integers(1, 10)) * 256 if ty != Q8_0 else int(rng.integers(1, 73)) * 32
        run_case(F, O, ty, t, n, k, 1000 + i)


@pytest.mark.parametrize("tile", [0, 1, 2, 3, 4, 5, 6])
def test_every_tile_on_ragged_shapes(F, O, tile):
    # The launcher picks one of thirteen workgroup tiles by estimate; here the first seven are pinned in turn (64 / 128 / 256 rows x 256
    # outputs, 256 x 160, 128 / 64 rows x 128, 128 x 160) and run on shapes that fill no tile: rows and outputs that end inside a tile, outputs that are no
    # multiple of 4, launches with whole rounds of tiles and a cut remainder, launches where every tile is cut along K.
    lib = F._lib.load()
    before = lib.fhip_debug_gemm_tile(tile)
    try:
        shapes = [(Q4_K, 33, 100, 512), (Q4_K, 300, 4001, 1024), (Q6_K, 130, 257, 2048), (Q8_0, 70, 1283, 1184), (Q4_K, 520, 7000, 768),
                  (Q6_K, 257, 161, 256), (Q8_0, 1025, 330, 96), (Q5_K, 300, 1283, 1024), (Q5_K, 70, 161, 2048)]
        for i, (ty, t, n, k) in enumerate(shapes):
            run_case(F, O, ty, t, n, k, 300 + 10 * tile + i)
    finally:
        lib.fhip_debug_gemm_tile(before)


@pytest.mark.parametrize("tile", [0, 1, 4, 5, 7, 8, 9, 10, 11, 12])
def test_tiles_whose_waves_unpack_for_themselves(F, O, tile):
    # 64 / 128 rows x 32 ... 256 outputs: one, two and three chunks of K a run (the pipeline is two deep), an odd chunk count, a run that
    # starts in one tile and ends in the next, rows and outputs that end inside a tile, a Q8_0 row that ends inside a chunk, every format,
    # and SwiGLU in the launch; the same bits again on a second run.
    lib = F._lib.load()
    before = lib.fhip_debug_gemm_tile(tile)
    try:
        shapes = [(Q4_K, 33, 65, 256), (Q5_K, 129, 193, 512), (Q6_K, 64, 321, 768), (Q8_0, 127, 100, 1312), (Q6_K, 200, 5000, 1280), (Q4_K, 321, 4100, 1792), (Q5_K, 65, 9000, 2304),
                  (Q8_0, 130, 2049, 2080)]
        for i, (ty, t, n, k) in enumerate(shapes):
            y = run_case(F, O, ty, t, n, k, 500 + 10 * tile + i)
            assert np.array_equal(y.view(np.uint32), run_case(F, O, ty, t, n, k, 500 + 10 * tile + i).view(np.uint32)), (tile, ty)
    finally:
        lib.fhip_debug_gemm_tile(before)


@pytest.mark.parametrize("tile", range(-1, 13))
def test_rows_shorter_than_a_chunk(F, O, tile):
    # Q8_0 rows of one to seven blocks, one short of a chunk of 256 columns: what lies behind a row is staged as zeros, behind the last one too.
    lib = F._lib.load()
    before = lib.fhip_debug_gemm_tile(tile)
    try:
        for i, (t, n, k) in enumerate([(33, 65, 32), (64, 320, 64), (65, 130, 96), (128, 257, 160), (300, 100, 224)]):
            from ferric_amd.synth import synth_weights
            w = synth_weights(Q8_0, n, k, 900 + i)
            xb, xv = bf16_round(np.random.default_rng(i).standard_normal((t, k)).astype(np.float32))
            y = F.Tensor.from_bf16_bits(xb, (t, k)).gemm_q_bf16(F.QMatrix.from_bytes(w, Q8_0, n, k)).to_vec().reshape(t, n)
            want = xv.astype(np.float64) @ bf16_round(O.deq_raw(w, n * k, Q8_0).reshape(n, k))[1].astype(np.float64).T
            assert np.abs(y - want).max() < 2e-5 * np.abs(want).max(), (t, n, k)      # f32 sums of bf16 products
    finally:
        lib.fhip_debug_gemm_tile(before)


@pytest.mark.parametrize("ty", [Q4_K, Q5_K, Q6_K, Q8_0])
def test_run_sums_add_in_the_order_of_one_accumulator(F, ty):
    # fhip_gemm_q_bf16_run_sums: the tiles whose waves unpack for themselves, one wave along K, have the bits of the tiles that share the
    # unpacking, one matrix instruction's sum after the other. One chunk of K, which no tile cuts: 256 x 256 pinned against the tile of 64 or
    # 128 rows that run sums take. Up to 32 rows both entry points are one launch.
    from ferric_amd.synth import synth_weights
    lib, k = F._lib.load(), 256
    for t, n in ((60, 3000), (60, 20000), (120, 3000), (250, 30000), (20, 700)):
        qm = F.QMatrix.from_bytes(synth_weights(ty, n, k, 77), ty, n, k)
        xb, _ = bf16_round(np.random.default_rng(78).standard_normal((t, k)).astype(np.float32))
        x, y = F.Tensor.from_bf16_bits(xb, (t, k)), F.Tensor.empty((t, n))
        F._lib.check(lib.fhip_gemm_q_bf16_run_sums(qm.handle, x.buf.ptr, t, y.buf.ptr, None))
        before = lib.fhip_debug_gemm_tile(2)
        try:
            want = x.gemm_q_bf16(qm).to_vec()
        finally:
            lib.fhip_debug_gemm_tile(before)
        assert np.array_equal(y.to_vec().view(np.uint32), want.view(np.uint32)), (ty, t)


# format, rows, outputs, columns and the CRC-32 of what the launches before waves unpacked for themselves made of these weights and activations: every tile of
# run sums, whole and cut along K, runs of one to seven chunks, a run that ends in the next tile, whole tiles in front of cut ones, Q8_0 rows that end inside a chunk, up to 32 rows
RUN_SUMS = [(Q6_K, 33, 2049, 5120, 0x91abb157), (Q6_K, 65, 9000, 1280, 0x4638172c), (Q5_K, 520, 4100, 2304, 0xc744183b),
            (Q4_K, 129, 4100, 1280, 0x9ad97f0c), (Q8_0, 128, 9000, 736, 0x3eee9c02), (Q8_0, 40, 5120, 512, 0x8a60427a),
            (Q4_K, 300, 7000, 256, 0x728fff2a), (Q5_K, 300, 7000, 1280, 0x20469f5f), (Q4_K, 300, 1283, 512, 0xbb42321c),
            (Q6_K, 300, 2049, 5120, 0xea8fa64e), (Q6_K, 65, 700, 1792, 0x617b63db), (Q8_0, 64, 2049, 2080, 0x51921f06),
            (Q8_0, 257, 9000, 512, 0xebb4198c), (Q5_K, 40, 9000, 512, 0xe2e70568), (Q4_K, 33, 7000, 2304, 0xcf249f68),
            (Q5_K, 257, 7000, 1792, 0x0a1e6c7c), (Q4_K, 100, 7000, 256, 0x1a419dc0), (Q8_0, 33, 1283, 4064, 0x08c261e7),
            (Q8_0, 64, 5120, 1312, 0x6aa96d04), (Q6_K, 64, 7000, 3328, 0xc9da5679), (Q6_K, 300, 5120, 1280, 0xf4d32ad6),
            (Q4_K, 20, 700, 768, 0xeb2b6df8)]
# formats of gate|up and down, rows, width, inner width, CRC-32 of gate|up and of the result
FFN_RUN_SUMS = [(Q4_K, Q6_K, 65, 512, 768, 0x0b67cb61, 0x0b3ad60d),
                (Q6_K, Q8_0, 200, 1280, 1312, 0x3b0411ae, 0x4f7554bb),
                (Q5_K, Q4_K, 520, 768, 2304, 0x7c3c39a0, 0x61ed940b),
                (Q4_K, Q8_0, 20, 512, 416, 0xe0c0b31a, 0x9d893b69)]


@pytest.mark.parametrize("i", range(len(RUN_SUMS)))
def test_run_sums_keep_their_bits(F, O, i):
    import zlib
    from ferric_amd.synth import synth_weights
    ty, t, n, k, crc = RUN_SUMS[i]
    w = synth_weights(ty, n, k, 20 + i)
    xb, xv = bf16_round(np.random.default_rng(40 + i).standard_normal((t, k)))
    qm, x, y = F.QMatrix.from_bytes(w, ty, n, k), F.Tensor.from_bf16_bits(xb, (t, k)), F.Tensor.empty((t, n))
    F._lib.check(F._lib.load().fhip_gemm_q_bf16_run_sums(qm.handle, x.buf.ptr, t, y.buf.ptr, None))
    got = y.to_vec().reshape(t, n)
    want = xv.astype(np.float64) @ bf16_round(O.deq_raw(w, n * k, ty).reshape(n, k))[1].astype(np.float64).T
    assert np.abs(got - want).max() < 2e-5 * np.abs(want).max()       # f32 sums of bf16 products
    assert zlib.crc32(got.tobytes()) == crc


@pytest.mark.parametrize("i", range(len(FFN_RUN_SUMS)))
def test_ffn_run_sums_keep_their_bits(F, i):
    import zlib
    from ferric_amd.synth import synth_weights
    lib, (tg, td, t, d, ff, crc_gate_up, crc) = F._lib.load(), FFN_RUN_SUMS[i]
    gu = F.QMatrix.from_bytes(synth_weights(tg, 2 * ff, d, 60 + i), tg, 2 * ff, d)
    dn = F.QMatrix.from_bytes(synth_weights(td, d, ff, 70 + i), td, d, ff)
    xb, _ = bf16_round(np.random.default_rng(80 + i).standard_normal((t, d)))
    x, g, y = F.Tensor.from_bf16_bits(xb, (t, d)), F.Tensor.empty((t, 2 * ff)), F.Tensor.empty((t, d))
    ws = F.DeviceBuffer(lib.fhip_ffn_coop_ws_bytes(gu.handle, dn.handle, t))
    args = (gu.handle, dn.handle, x.buf.ptr)
    assert lib.fhip_ffn_bf16_run_sums(*args, None, t, y.buf.ptr, ws.ptr, None) != 0                   # gate|up has to be in memory
    F._lib.check(lib.fhip_ffn_bf16_run_sums(*args, g.buf.ptr, t, y.buf.ptr, ws.ptr, None))
    assert (zlib.crc32(g.to_vec().tobytes()), zlib.crc32(y.to_vec().tobytes())) == (crc_gate_up, crc)


def test_reference_coop_example_shapes(F, O):
    # crates/ferric-tensor/examples/coop_q4_k.rs: reference-generator weights, M a multiple of 8 and not
    run_case(F, O, Q4_K, 16, 64, 512, 3, gen=O.gen_kquant_matrix)
    run_case(F, O, Q4_K, 13, 128, 1024, 4, gen=O.gen_kquant_matrix)
    run_case(F, O, Q6_K, 24, 64, 512, 5, gen=O.gen_kquant_matrix)


@pytest.mark.parametrize("t", [128, 512, 2048])
def test_config4_prefill_5120(F, O, t):
    # W 5120x5120 Q4_K, X [t, 5120] bf16 ~ N(0,1), f32 out
    run_case(F, O, Q4_K, t, 5120, 5120, 21)


@pytest.mark.parametrize("ty,t,n,k", [(Q4_K, 2048, 34816, 5120), (Q6_K, 512, 5120, 17408), (Q8_0, 2048, 4096, 4096)])
def test_the_layer_s_large_projections_on_sampled_outputs(F, O, ty, t, n, k):
    # The fused gate|up weight at 2048 rows is four whole rounds of 256 x 256 tiles and a remainder cut in four, the down
    # projection at 512 rows 256 x 160 tiles each cut in four, Q8_0 4096 x 4096 a grid of 208 whole 256 x 160 tiles. Too large for
    # the f64 model in full: 384 weight rows spread over the first, the last and random tiles, every activation row.
    from ferric_amd.synth import synth_weights
    w = synth_weights(ty, n, k, 71)
    x = np.random.default_rng(72).standard_normal((t, k)).astype(np.float32)
    xb, xv = bf16_round(x)
    qm = F.QMatrix.from_bytes(w, ty, n, k)
    y = F.Tensor.from_bf16_bits(xb, (t, k)).gemm_q_bf16(qm).to_vec().reshape(t, n)
    rows = np.unique(np.concatenate([np.arange(64), np.arange(n - 64, n), np.random.default_rng(73).integers(0, n, 256)]))
    rb = len(w) // n
    wd = O.deq_raw(np.ascontiguousarray(w.reshape(n, rb)[rows]).reshape(-1), len(rows) * k, ty).reshape(len(rows), k)
    _, wb = bf16_round(wd)
    model = xv.astype(np.float64) @ wb.astype(np.float64).T
    got = y[:, rows]
    assert np.abs(got - model).max() / np.abs(model).max() < 2e-5
    exact = xv.astype(np.float64) @ wd.astype(np.float64).T
    bound = 1e-3 * np.linalg.norm(wd.astype(np.float64), axis=1)[None, :] * np.linalg.norm(xv.astype(np.float64), axis=1)[:, None]
    assert (np.abs(got - exact) <= bound).all()


def test_prefill_other_formats_at_size(F, O):
    run_case(F, O, Q5_K, 512, 5120, 5120, 24)
    run_case(F, O, Q6_K, 256, 5120, 5120, 22)
    run_case(F, O, Q8_0, 256, 4096, 4096, 23)


def test_rows_are_independent_of_the_batch(F, O):
    # A row of a T-row prefill is bit-identical to the same row computed in a smaller batch, as long as
    # both launches have enough output tiles to run without splitting K (a K split changes where the sum over K is cut,
    # so across batch sizes only the tolerance holds there, not bit equality).
    from ferric_amd.synth import synth_weights
    w = synth_weights(Q4_K, 5120, 512, 5)
    qm = F.QMatrix.from_bytes(w, Q4_K, 5120, 512)
    x = np.random.default_rng(1).standard_normal((1536, 512)).astype(np.float32)
    xb, _ = bf16_round(x)
    # 1536 and 1280 rows: 240 and 200 tiles of 128 x 256, each computed whole by one workgroup
    big = F.Tensor.from_bf16_bits(xb, (1536, 512)).gemm_q_bf16(qm).to_vec().reshape(1536, 5120)
    part = F.Tensor.from_bf16_bits(xb[256:], (1280, 512)).gemm_q_bf16(qm).to_vec().reshape(1280, 5120)
    assert np.array_equal(big[256:].view(np.uint32), part.view(np.uint32))
    again = F.Tensor.from_bf16_bits(xb, (1536, 512)).gemm_q_bf16(qm).to_vec().reshape(1536, 5120)
    assert np.array_equal(big.view(np.uint32), again.view(np.uint32))


@pytest.mark.parametrize("ty,t,n,k", [(Q4_K, 128, 5120, 5120), (Q4_K, 512, 5120, 5120), (Q4_K, 2048, 9216, 5120),
                                      (Q6_K, 300, 1000, 4096), (Q8_0, 200, 1300, 2080), (Q4_K, 70, 3000, 8192),
                                      (Q4_K, 8, 5120, 5120), (Q6_K, 20, 1000, 4096), (Q8_0, 3, 1300, 2080), (Q4_K, 32, 1024, 5120),
                                      (Q5_K, 256, 5120, 5120), (Q5_K, 9, 3000, 2048)])
def test_two_runs_give_identical_bits(F, O, ty, t, n, k):
    # Launches with fewer whole tiles than the chip has workgroups cut tiles along K (every shape here does; 2048 x 9216
    # has a cut remainder behind whole tiles; up to 32 rows it is groups of 128 outputs that are cut). The partial tiles are
    # summed in a fixed order, so the bits may not depend on which workgroup finishes first: five runs, with other work on
    # the device in between, one result.
    from ferric_amd.synth import synth_weights
    lib = F._lib.load()
    w = synth_weights(ty, n, k, 31)
    qm = F.QMatrix.from_bytes(w, ty, n, k)
    assert lib.fhip_workspace_bytes_coop(qm.handle, None, t) > 0, "the case is meant to cut tiles along K"
    xb, _ = bf16_round(np.random.default_rng(32).standard_normal((t, k)).astype(np.float32))
    x = F.Tensor.from_bf16_bits(xb, (t, k))
    first = x.gemm_q_bf16(qm).to_vec().view(np.uint32)
    other = F.QMatrix.from_bytes(synth_weights(Q4_K, 512, 1024, 33), Q4_K, 512, 1024)
    xo = F.Tensor.from_bf16_bits(bf16_round(np.ones((40, 1024), np.float32))[0], (40, 1024))
    for _ in range(4):
        xo.gemm_q_bf16(other)              # another launch that uses the same workspace
        assert np.array_equal(first, x.gemm_q_bf16(qm).to_vec().view(np.uint32))


def test_q8_0_rows_ending_inside_a_chunk(F, O):
    # Q8_0 rows are any multiple of 32 long; the kernel walks 256-column chunks, so 32..224 trailing columns
    # exercise the zero-scale / zero-activation padding of the last chunk (and K < 256 has no full chunk at all)
    for i, (t, n, k) in enumerate([(3, 40, 32), (9, 64, 96), (40, 130, 288), (130, 70, 480), (70, 257, 1184)]):
        run_case(F, O, Q8_0, t, n, k, 40 + i)


def test_coop_entry_takes_f32_activations(F, O):
    # dtype.rs:1818 matmul_q4_k_coop reads f32 x; here x is rounded to bf16 (RNE) on the device first. The
    # rounding is checked bit for bit, the product against the bf16 entry point fed host-rounded activations
    # (equal up to the order in which K slices are added when the launch splits K).
    from ferric_amd.synth import synth_weights
    for ty, name, (t, n, k) in [(Q4_K, "matmul_q4_k_coop", (8, 512, 1024)), (Q6_K, "matmul_q6_k_coop", (4, 256, 512)),
                                (Q8_0, "matmul_q8_0_coop", (21, 264, 416)), (Q4_K, "matmul_q4_k_coop", (150, 384, 768)),
                                (Q5_K, "matmul_q5_k_coop", (12, 256, 1024)), (Q5_K, "matmul_q5_k_coop", (150, 384, 768))]:
        w = synth_weights(ty, n, k, 60)
        qm = F.QMatrix.from_bytes(w, ty, n, k)
        x = (np.random.default_rng(61).standard_normal((t, k)) * 3).astype(np.float32)
        x[0, :4] = [0.0, -0.0, 1.00390625, 1.01171875]   # exact ties, to even both ways
        xb, _ = bf16_round(x)
        xt = F.Tensor.from_vec(x.reshape(-1), (t, k))
        assert np.array_equal(xt.cvt_bf16().to_vec().reshape(t, k), xb)
        want = F.Tensor.from_bf16_bits(xb, (t, k)).gemm_q_bf16(qm).to_vec()
        got = getattr(xt, name)(qm).to_vec()
        assert np.abs(got - want).max() <= 2e-5 * np.abs(want).max(), name
    odd = np.arange(13, dtype=np.float32) * 1.001      # a length that is not a multiple of 8: the scalar tail
    odd[:5] = [3.0e38, -3.3895314e38, 1e-40, -65280.0, np.inf]   # near and past the largest bf16, a denormal
    assert np.array_equal(F.Tensor.from_vec(odd, (1, 13)).cvt_bf16().to_vec(), bf16_round(odd)[0])
    with pytest.raises(AssertionError, match="multiple of 8"):
        qm = F.QMatrix.from_bytes(synth_weights(Q4_K, 12, 256, 1), Q4_K, 12, 256)
        F.Tensor.from_vec(np.zeros(256, np.float32), (1, 256)).matmul_q4_k_coop(qm)


def test_batched_decode_ffn_on_the_matrix_cores(F, O):
    # FFN block at batch 4 and 8 through the coop entry points: gate_up -> swiglu -> down, against f64 on
    # oracle-dequantized weights, to the north-star bound applied to each matmul
    from ferric_amd.synth import synth_weights
    d, n_ff = 1024, 2816
    gu = synth_weights(Q4_K, 2 * n_ff, d, 70)
    dn = synth_weights(Q6_K, d, n_ff, 71)
    qgu, qdn = F.QMatrix.from_bytes(gu, Q4_K, 2 * n_ff, d), F.QMatrix.from_bytes(dn, Q6_K, d, n_ff)
    wgu = O.deq_raw(gu, 2 * n_ff * d, Q4_K).reshape(2 * n_ff, d).astype(np.float64)
    wdn = O.deq_raw(dn, d * n_ff, Q6_K).reshape(d, n_ff).astype(np.float64)
    for b in (4, 8):
        x = np.random.default_rng(72 + b).standard_normal((b, d)).astype(np.float32)
        g = F.Tensor.from_vec(x.reshape(-1), (b, d)).matmul_q4_k_coop(qgu)
        g64 = x.astype(np.float64) @ wgu.T
        bound = 1e-3 * np.linalg.norm(wgu, axis=1)[None, :] * np.linalg.norm(x.astype(np.float64), axis=1)[:, None]
        assert (np.abs(g.to_vec().reshape(b, -1) - g64) <= bound).all()
        hid = g.swiglu(n_ff)
        hv = hid.to_vec().reshape(b, n_ff)
        y = hid.matmul_q6_k_coop(qdn).to_vec().reshape(b, d)
        y64 = hv.astype(np.float64) @ wdn.T
        bound = 1e-3 * np.linalg.norm(wdn, axis=1)[None, :] * np.linalg.norm(hv.astype(np.float64), axis=1)[:, None]
        assert (np.abs(y - y64) <= bound).all()
        # the one-call block does the same steps (the SwiGLU output is rounded to bf16 either way)
        y1 = F.Tensor.from_vec(x.reshape(-1), (b, d)).ffn_coop(qgu, qdn).to_vec().reshape(b, d)
        assert np.abs(y1 - y).max() <= 2e-5 * np.abs(y).max()


@pytest.mark.parametrize("tile", [0, 1, 2, 3, 4, 5, 6, -1])
def test_swiglu_inside_the_tiled_gemm(F, tile):
    # ffn_coop over 32 rows applies SwiGLU in the gate|up launch (or in the launch that sums a cut tile): one f32 expression and one rounding to
    # bf16 on sums that are the same f32 sums as those of its steps where both launches cut the same outputs along K. They do on these
    # shapes, whose tiles are all whole or all cut, and the block equals its steps bit for bit; where a launch has whole tiles and cut ones the
    # fused launch cuts other outputs (test_swiglu_beside_whole_and_cut_tiles). Rows that end inside a tile, widths whose tiles are
    # ragged (n_ff = 96: tiles of mostly nothing; 1312: no multiple of any tile's columns).
    from ferric_amd.synth import synth_weights
    lib = F._lib.load()
    before = lib.fhip_debug_gemm_tile(tile)
    try:
        for i, (tg, td, t, d, n_ff) in enumerate([(Q4_K, Q8_0, 33, 512, 96), (Q4_K, Q8_0, 300, 1024, 1312), (Q6_K, Q4_K, 65, 768, 512), (Q8_0, Q6_K, 257, 288, 768),
                                                  (Q5_K, Q8_0, 130, 1024, 1312), (Q4_K, Q6_K, 520, 256, 9984)]):
            gu = F.QMatrix.from_bytes(synth_weights(tg, 2 * n_ff, d, 900 + i), tg, 2 * n_ff, d)
            dn = F.QMatrix.from_bytes(synth_weights(td, 256, n_ff, 950 + i), td, 256, n_ff)
            x = F.Tensor.from_vec(np.random.default_rng(i).standard_normal(t * d).astype(np.float32), (t, d))
            want = x.matmul_q_coop(gu).swiglu(n_ff).matmul_q_coop(dn).to_vec()
            assert np.array_equal(x.ffn_coop(gu, dn).to_vec().view(np.uint32), want.view(np.uint32)), (tile, tg, t, n_ff)
    finally:
        lib.fhip_debug_gemm_tile(before)


@pytest.mark.parametrize("tile", [0, 1, 4, 5, 7, 8, 9, 10, 11, 12])
def test_swiglu_of_rows_turned_through_lds(F, tile):
    # Q6_K and Q8_0 gate|up on the tiles whose waves unpack for themselves: a wave's gate and up rows lie in two places. Rows of an odd number of blocks, whose
    # addresses alternate modulo 4, widths that end inside a tile, one chunk and an odd number of them, a Q8_0 row that ends inside a chunk; against the
    # 256 x 160 tile, whose waves share what they unpack. The f32 sums differ in their last bits, so a value of h may round to the other bf16 neighbour, 2^-8 of it.
    from ferric_amd.synth import synth_weights
    lib = F._lib.load()
    before = lib.fhip_debug_gemm_tile(tile)
    try:
        for i, (ty, t, d, n_ff) in enumerate([(Q6_K, 33, 256, 32), (Q6_K, 70, 768, 160), (Q8_0, 65, 288, 96), (Q8_0, 129, 1312, 1312)]):
            gu = F.QMatrix.from_bytes(synth_weights(ty, 2 * n_ff, d, 700 + i), ty, 2 * n_ff, d)
            dn = F.QMatrix.from_bytes(synth_weights(Q8_0, 64, n_ff, 720 + i), Q8_0, 64, n_ff)
            x = F.Tensor.from_vec(np.random.default_rng(i).standard_normal(t * d).astype(np.float32), (t, d))
            lib.fhip_debug_gemm_tile(3)
            want = x.ffn_coop(gu, dn).to_vec()
            lib.fhip_debug_gemm_tile(tile)
            got = x.ffn_coop(gu, dn).to_vec()
            assert np.linalg.norm(got - want) <= 2.0 ** -8 * np.linalg.norm(want), (tile, ty, t, d, n_ff)
    finally:
        lib.fhip_debug_gemm_tile(before)


# 272 tiles of 64 x 128, 312 of 64 x 256 and of 128 x 256, and the launcher's choice: 256 workgroups take a whole one each and the rest is cut along K
@pytest.mark.parametrize("tile,t,d,n_ff", [(5, 40, 512, 17408), (0, 130, 512, 13312), (1, 270, 768, 13312), (-1, 520, 512, 17408)])
def test_swiglu_beside_whole_and_cut_tiles(F, O, tile, t, d, n_ff):
    # The fused launch deals columns of gate and up in turn to a tile and so cuts other outputs than a launch over the stacked rows does:
    # their sums are added in another order, and a last bit in front of the rounding of h to bf16 may move. Against f64 the block is as exact as
    # its steps. Bound of both: an operand's rounding to bf16 is at most 2^-9 of it; x and the weights of gate and up enter silu(g) u twice (its two
    # factors), h and the weights of down once, so 6 * 2^-9 of the norm if every rounding were its largest and all of them added up.
    from ferric_amd.synth import synth_weights
    lib = F._lib.load()
    before = lib.fhip_debug_gemm_tile(tile)
    try:
        raw = synth_weights(Q4_K, 2 * n_ff, d, 31), synth_weights(Q6_K, 256, n_ff, 32)
        gu, dn = F.QMatrix.from_bytes(raw[0], Q4_K, 2 * n_ff, d), F.QMatrix.from_bytes(raw[1], Q6_K, 256, n_ff)
        x = np.random.default_rng(33).standard_normal((t, d)).astype(np.float32)
        x /= np.float32(np.linalg.norm(O.deq_raw(raw[0], 2 * n_ff * d, Q4_K).reshape(2 * n_ff, d), axis=1).mean())     # gate and up of order one
        X = F.Tensor.from_vec(x, x.shape)
        fused, again = (X.ffn_coop(gu, dn).to_vec().reshape(t, -1) for _ in range(2))
        steps = X.matmul_q_coop(gu).swiglu(n_ff).matmul_q_coop(dn).to_vec().reshape(t, -1)
    finally:
        lib.fhip_debug_gemm_tile(before)
    g = x.astype(np.float64) @ O.deq_raw(raw[0], 2 * n_ff * d, Q4_K).reshape(2 * n_ff, d).astype(np.float64).T
    h = g[:, :n_ff] / (1 + np.exp(-g[:, :n_ff])) * g[:, n_ff:]
    want = h @ O.deq_raw(raw[1], 256 * n_ff, Q6_K).reshape(256, n_ff).astype(np.float64).T
    err = lambda y: np.linalg.norm(y - want) / np.linalg.norm(want)
    assert np.array_equal(fused.view(np.uint32), again.view(np.uint32))
    assert err(fused) < 6 * 2.0 ** -9 and err(fused) < 1.01 * err(steps), (err(fused), err(steps))
    assert np.linalg.norm(fused - steps) < 2e-4 * np.linalg.norm(want), np.linalg.norm(fused - steps) / np.linalg.norm(want)


def test_gemm_errors(F):
    qm = F.QMatrix.from_bytes(np.zeros(144, np.uint8), Q4_K, 1, 256)
    with pytest.raises(AssertionError, match="inner dim mismatch"):
        F.Tensor.from_bf16_bits(np.zeros(512, np.uint16), (1, 512)).gemm_q_bf16(qm)
    assert F.Tensor.from_bf16_bits(np.zeros(0, np.uint16), (0, 256)).gemm_q_bf16(qm).to_vec().size == 0
