"""Batches of the 32-value formats on the kernel that multiplies through the 16 x 16 x 32 int8 matrix instruction (gemv_wide.hip)
against single rows on the dot-product mat-vec it restates: the same bits for every row, whatever the batch a row sits in
(crates/ferric-tensor/src/cpu_simd.rs:175-200); the entry points' own tests hold both to the oracle."""
import numpy as np
import pytest

from conftest import ROUTES, bits, route

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("precision")]
Q4_0, Q4_1, Q5_0, Q5_1, Q8_0, IQ4_NL, IQ4_XS, MXFP4 = 2, 3, 6, 7, 8, 20, 23, 39
# rows x cols: one block; whole tiles and groups; cut tiles and a last group of 1, 4 and 8 blocks; several passes over K (17408
# columns); several tiles a workgroup
SHAPES = [(1, 32), (16, 512), (37, 1056), (130, 2560), (9, 17408), (4200, 768)]


def singles_of(F, qm, x):
    return np.stack([F.Tensor.from_vec(r, (1, x.shape[1])).matmul_q(qm).to_vec() for r in x])


def same(got, want):
    ok = ~np.isnan(want)
    return np.array_equal(np.isnan(got), ~ok) and np.array_equal(bits(got)[ok], bits(want)[ok])


@pytest.mark.parametrize("ty", [Q4_0, Q4_1, Q5_0, Q5_1, Q8_0, IQ4_NL, IQ4_XS, MXFP4])
@pytest.mark.parametrize("rows,cols", SHAPES)
def test_same_bits_as_single_rows(F, ty, rows, cols):
    from ferric_amd.synth import synth_weights
    cols = max(256, cols // 256 * 256) if ty == IQ4_XS else cols
    qm = F.QMatrix.from_bytes(synth_weights(ty, rows, cols, rows + cols), ty, rows, cols)
    qm.batch_policy(F.BATCH_F32_MATVEC)
    x = np.random.default_rng(cols).standard_normal((18, cols)).astype(np.float32)
    x[1] *= np.float32(300.0)
    x[2, ::7] = 0
    # runs block fixed point cannot hold: tiny, huge, infinite and NaN members, in rows of every accumulator
    x[4, :32] *= np.float32(1e-36)
    x[7, -32:] = np.float32(1e30)
    x[9, cols // 2], x[14, 5] = np.inf, np.nan
    one = singles_of(F, qm, x)
    for m in (5, 8, 9, 16, 18):
        got = F.Tensor.from_vec(x[:m], (m, cols)).matmul_q(qm).to_vec().reshape(m, rows)
        assert same(got, one[:m]), m


@pytest.mark.parametrize("ty,rows,cols", [(Q4_1, 530, 8192), (MXFP4, 2100, 11040), (IQ4_NL, 5200, 8224), (IQ4_XS, 900, 4096)])
def test_rows_dealt_out_to_several_workgroups(F, ty, rows, cols):
    # few tiles or long rows: two to four groups of activation rows, the last one short (13 = 4 + 4 + 4 + 1, 5 = 3 + 2), one tile a workgroup and several
    from ferric_amd.synth import synth_weights
    qm = F.QMatrix.from_bytes(synth_weights(ty, rows, cols, cols), ty, rows, cols)
    qm.batch_policy(F.BATCH_F32_MATVEC)
    x = np.random.default_rng(rows).standard_normal((16, cols)).astype(np.float32)
    x[12, 64:96] = np.float32(1e30)
    one = singles_of(F, qm, x)
    for m in (5, 6, 7, 10, 13, 16):
        assert same(F.Tensor.from_vec(x[:m], (m, cols)).matmul_q(qm).to_vec().reshape(m, rows), one[:m]), m


@pytest.mark.parametrize("ty,rows,cols", [(Q5_1, 993, 4320), (Q4_1, 40, 11040), (Q8_0, 257, 5152), (IQ4_NL, 17, 17408)])
def test_more_waves_than_items(F, ty, rows, cols):
    # one tile a workgroup and 9 to 16 groups of 512 columns, the last one short: waves that quantise and have no item, in one pass and in several
    from ferric_amd.synth import synth_weights
    qm = F.QMatrix.from_bytes(synth_weights(ty, rows, cols, 7), ty, rows, cols)
    qm.batch_policy(F.BATCH_F32_MATVEC)
    x = np.random.default_rng(cols).standard_normal((16, cols)).astype(np.float32)
    x[3, -32:] = np.float32(1e30)
    one = singles_of(F, qm, x)
    xt = F.Tensor.from_vec(x, x.shape)
    # (four rows of this few weights: at 24 bits, Q8_0 apart; else they are the dot-product kernel's, which promises no row's bits beside the run of 1e30)
    four = qm.matvec_precision(0) == 24 and ty != Q8_0
    for m in (4, 5, 8, 9, 14, 16) if four else (5, 8, 9, 14, 16):
        assert route(F, qm, xt, m) == [(ROUTES["WIDE"], m)]
        assert same(F.Tensor.from_vec(x[:m], (m, cols)).matmul_q(qm).to_vec().reshape(m, rows), one[:m]), m


@pytest.mark.parametrize("ty,rows,cols,m", [(Q5_1, 12300, 2080, 3), (IQ4_NL, 12289, 2048, 4), (Q8_0, 1200, 7040, 4)])
def test_three_and_four_rows_of_large_weights(F, ty, rows, cols, m):
    from ferric_amd.synth import synth_weights
    qm = F.QMatrix.from_bytes(synth_weights(ty, rows, cols, 3), ty, rows, cols)
    qm.batch_policy(F.BATCH_F32_MATVEC)
    x = np.random.default_rng(4).standard_normal((m, cols)).astype(np.float32)
    assert same(F.Tensor.from_vec(x, x.shape).matmul_q(qm).to_vec().reshape(m, rows), singles_of(F, qm, x))


@pytest.mark.parametrize("ty,rows,cols,m,last", [(Q8_0, 130, 4096, 19, "DOT"), (Q8_0, 130, 4096, 20, "QUAD"), (Q8_0, 96, 5120, 36, "QUAD"), (Q8_0, 40, 5152, 20, "DOT"), (Q8_0, 1700, 5152, 20, "WIDE"), (Q4_0, 70, 1024, 19, "DOT"),
                                                  (IQ4_NL, 64, 512, 21, "WIDE"), (Q5_0, 33, 96, 18, "DOT")])
def test_the_rows_behind_the_last_sixteen_go_where_a_batch_of_them_would(F, ty, rows, cols, m, last):
    from ferric_amd.synth import synth_weights
    qm = F.QMatrix.from_bytes(synth_weights(ty, rows, cols, 5), ty, rows, cols)
    qm.batch_policy(F.BATCH_F32_MATVEC)
    x = np.random.default_rng(6).standard_normal((m, cols)).astype(np.float32)
    xt = F.Tensor.from_vec(x, x.shape)
    assert route(F, qm, xt, m) == [(ROUTES["WIDE"], 16)] * (m // 16) + [(ROUTES[last], m % 16)]
    assert same(xt.matmul_q(qm).to_vec().reshape(m, rows), singles_of(F, qm, x))


@pytest.mark.parametrize("ty,rows,cols,m,at24,at16", [(Q4_0, 520, 1600, 4, "WIDE", "WIDE"), (MXFP4, 20, 352, 4, "WIDE", "WIDE"), (MXFP4, 300, 7168, 4, "WIDE", "DOT"), (IQ4_NL, 1600, 8192, 3, "WIDE", "DOT"),
                                                       (IQ4_NL, 1500, 8192, 3, "DOT", "DOT"), (Q5_1, 1400, 9216, 3, "DOT", "DOT")])
def test_three_and_four_rows_of_small_weights(F, ty, rows, cols, m, at24, at16):
    from ferric_amd.synth import synth_weights
    qm = F.QMatrix.from_bytes(synth_weights(ty, rows, cols, 3), ty, rows, cols)
    qm.batch_policy(F.BATCH_F32_MATVEC)
    x = np.random.default_rng(4).standard_normal((m, cols)).astype(np.float32)
    kernel = at24 if qm.matvec_precision(0) == 24 else at16
    if kernel == "WIDE":
        x[2, 5] = np.float32(1e38)      # a run that block fixed point cannot hold, in one row
    xt = F.Tensor.from_vec(x, x.shape)
    assert route(F, qm, xt, m) == [(ROUTES[kernel], m)]
    assert same(xt.matmul_q(qm).to_vec().reshape(m, rows), singles_of(F, qm, x))


# four rows: short of a group; whole groups; one pass of the dot-product kernel by rows and columns; two (over 1568 .. 2048, 3104 .. 4096, 5152 .. 6144 columns, from 7200 on); three: Q5_0
@pytest.mark.parametrize("ty,rows,cols,m,at24,at16", [
    (Q4_0, 40, 480, 4, "DOT", "DOT"), (MXFP4, 20, 256, 4, "DOT", "DOT"), (MXFP4, 256, 288, 4, "WIDE", "WIDE"), (MXFP4, 257, 288, 4, "DOT", "DOT"), (Q4_0, 10241, 256, 4, "WIDE", "DOT"),
    (Q4_0, 10240, 256, 4, "DOT", "DOT"), (Q5_0, 20481, 288, 4, "WIDE", "WIDE"), (Q5_0, 20480, 288, 4, "DOT", "DOT"), (Q5_0, 700, 512, 4, "WIDE", "WIDE"), (Q5_0, 600, 3072, 4, "WIDE", "WIDE"),
    (Q4_0, 256, 544, 4, "WIDE", "WIDE"), (Q4_0, 257, 544, 4, "WIDE", "DOT"), (Q5_1, 257, 544, 4, "DOT", "DOT"), (Q5_1, 257, 1056, 4, "WIDE", "DOT"), (IQ4_XS, 300, 768, 4, "WIDE", "WIDE"),
    (IQ4_XS, 513, 768, 4, "DOT", "DOT"), (IQ4_NL, 1024, 1056, 4, "DOT", "DOT"), (IQ4_NL, 1025, 1056, 4, "WIDE", "DOT"), (Q4_1, 4097, 544, 4, "WIDE", "WIDE"), (Q5_0, 4097, 544, 4, "WIDE", "DOT"),
    (Q5_0, 4096, 544, 4, "DOT", "DOT"), (Q4_1, 600, 2080, 4, "WIDE", "WIDE"), (Q5_0, 256, 1504, 4, "WIDE", "WIDE"), (Q5_0, 50, 2080, 4, "DOT", "DOT"), (Q5_0, 1537, 2080, 4, "WIDE", "DOT"),
    (MXFP4, 300, 2048, 4, "WIDE", "WIDE"), (Q5_0, 33, 3616, 4, "WIDE", "WIDE"), (Q5_1, 17, 6144, 4, "WIDE", "WIDE"), (Q5_1, 17, 7648, 4, "WIDE", "DOT"), (IQ4_XS, 30, 4608, 4, "WIDE", "DOT"),
    (Q5_1, 326, 4896, 4, "WIDE", "DOT"), (Q5_0, 326, 4896, 4, "DOT", "DOT"), (Q5_0, 20, 12288, 4, "WIDE", "DOT"), (Q5_0, 20, 12320, 4, "DOT", "DOT"), (Q5_0, 1728, 4864, 4, "WIDE", "WIDE"),
    (Q5_0, 1600, 8192, 3, "DOT", "DOT")])
def test_where_three_and_four_rows_of_small_weights_change_kernels(F, ty, rows, cols, m, at24, at16):
    test_three_and_four_rows_of_small_weights(F, ty, rows, cols, m, at24, at16)


def test_mxfp4_blocks_that_may_overflow(F):
    """Scale bytes from 252 on: inf weights, and finite ones near the top of f32, beside ordinary blocks."""
    rng = np.random.default_rng(21)
    rows, cols = 40, 544
    blk = rng.integers(0, 256, (rows, cols // 32, 17), dtype=np.uint8)
    blk[:, :, 0] = rng.integers(0x70, 0x80, (rows, cols // 32), dtype=np.uint8)
    blk[3, 5, 0], blk[7, 0, 0], blk[7, 9, 0], blk[11, 15, 0], blk[12, 2, 0], blk[33, 16, 0] = 255, 254, 253, 252, 251, 253
    qm = F.QMatrix.from_bytes(blk.reshape(-1), MXFP4, rows, cols)
    x = rng.standard_normal((16, cols)).astype(np.float32)
    x[5, 160:168] = 0.0
    one = singles_of(F, qm, x)
    assert not np.isfinite(one[:, 7]).any()
    for m in (5, 16):
        assert same(F.Tensor.from_vec(x[:m], (m, cols)).matmul_q(qm).to_vec().reshape(m, rows), one[:m]), m
