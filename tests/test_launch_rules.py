"""What the launchers decide on the host, without a device: the sources are compiled for the host alone and asked."""
import ctypes as C
import os
import subprocess

import pytest

from conftest import ROOT

Q8_0, Q4_K, Q5_K, Q6_K = 8, 12, 13, 14


def build(d, harness, flags, link):
    """tests/<harness> as a program or a shared object."""
    obj, out = str(d / (harness + ".o")), str(d / (harness + ".so"))
    subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "--offload-host-only", "--offload-arch=gfx950", "-x", "hip", "-std=c++17", "-O1", "-fPIC", "-fuse-cuid=none",
                    *flags, "-c", os.path.join(ROOT, "tests", harness), "-o", obj], check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    subprocess.run(["g++", *link, "-o", out, obj], check=True)
    return out


@pytest.fixture(scope="module")
def gemm(tmp_path_factory):
    return C.CDLL(build(tmp_path_factory.mktemp("gemm"), "gemm_rules_harness.cpp", ["-DFHIP_GEMM_FORMAT=Q80"], ["-shared", "-Wl,-Bsymbolic"]))


def plan(gemm, ty, outputs, cols, rows, run_sums=False):
    """(tile, its rows, its outputs, whole rounds, chunks a run, workgroups) on 256 CUs"""
    out = (C.c_int64 * 6)()
    gemm.h_plan(C.c_uint32(ty), C.c_size_t(outputs), C.c_size_t(cols), C.c_size_t(rows), int(run_sums), out)
    return tuple(out)


@pytest.fixture(scope="module")
def attention(tmp_path_factory):
    """[(rows, keys, heads, head size, window)] -> [(most key tiles of a range, ranges)]"""
    program = build(tmp_path_factory.mktemp("attn"), "attn_rules_harness.cpp", ["-Xarch_host", "-fsanitize=undefined", "-Xarch_host", "-fsanitize-trap=undefined"], [])

    def ask(shapes):
        r = subprocess.run([program], input="".join("%d %d %d %d %d\n" % x for x in shapes), capture_output=True, text=True)
        assert r.returncode == 0, (r.returncode, shapes[len(r.stdout.splitlines())])
        return [tuple(map(int, line.split())) for line in r.stdout.splitlines()]
    return ask


@pytest.fixture(scope="module")
def decode(tmp_path_factory):
    return C.CDLL(build(tmp_path_factory.mktemp("decode"), "decode_rules_harness.cpp", [], ["-shared", "-Wl,-Bsymbolic"]))


def test_when_a_norm_requests_its_weights_with_the_row(decode):
    """Both sides timed on 256 CUs, us by workgroups: weights behind the sum, with the row."""
    timed = {64: (4.0, 3.6), 256: (4.0, 3.7), 1024: (11.6, 10.7), 1500: (5.5, 6.7), 2048: (21.3, 23.3), 16384: (17.6, 20.6)}
    for grid, (behind, with_row) in timed.items():
        assert bool(decode.h_norm_ahead(C.c_size_t(grid))) == (with_row < behind), grid


@pytest.fixture(scope="module")
def wide(tmp_path_factory):
    c = C.CDLL(build(tmp_path_factory.mktemp("wide"), "wide_rules_harness.cpp", ["-DFHIP_GEMV_PLANES=3"], ["-shared", "-Wl,-Bsymbolic"]))

    def ask(ty, rows, cols, t, each):
        out = (C.c_int64 * 7)()
        c.h_wide_plan(C.c_uint32(ty), *(C.c_size_t(n) for n in (rows, cols, t, each)), out)
        return tuple(out)
    return ask


def test_more_waves_than_items_of_a_batch_where_they_were_the_faster(wide):
    """Q8_0 at more than eight rows keeps a wave an item, eight at least: us with those | with all waves."""
    q5_0 = 6
    for ty, rows, cols, t, few, all_waves in ((Q8_0, 9238, 512, 16, 7.9, 8.7), (Q8_0, 4914, 1120, 11, 11.6, 12.4), (Q8_0, 7482, 1088, 11, 11.7, 12.4), (q5_0, 1458, 17248, 7, 41.8, 37.2),
                                              (q5_0, 1312, 13280, 14, 33.1, 29.4)):
        pairs, tiles, groups, _, waves, _, _ = wide(ty, rows, cols, t, t)
        assert (waves > max(8, tiles * groups)) == (all_waves < few), (ty, rows, cols, t)


def test_four_pairs_a_lane_are_one_workgroup_s_only(wide):
    """The kernel of four pairs does not look for rows of its own: whatever a batch is dealt out to, it never shares one."""
    for t in range(1, 17):
        for shares in range(1, min(t, 4) + 1):
            pairs, *_, n = wide(Q8_0, 5000, 2048, t, -(-t // shares))
            assert n <= shares and n * 4 * pairs >= t and (pairs < 4 or n == 1), (t, shares)


@pytest.mark.parametrize("width", [64, 256])      # columns of a step (unpacked weights shared) and of a chunk (waves that unpack for themselves)
def test_no_activation_is_read_from_behind_the_last(gemm, width):
    """Threads stage 16-byte pieces of whole steps or chunks of columns: rows and columns that do not exist are read from x all the same, those that do from where they are."""
    gemm.h_x_at.restype = C.c_uint32
    for K in [*range(32, 544, 32), 1312, 1344, 4064]:
        for T in (33, 64, 100):
            for t in (0, 32, T - 1, T, T + 255):
                for first in range(0, (K + width - 1) // width * width + 1, width):
                    for col in range(0, width, 8):
                        at = gemm.h_x_at(t, T, K, first, col)
                        assert at % 8 == 0 and at + 8 <= T * K, (K, T, t, first, col)
                        assert at // K == min(t, T - 1) and (first + col >= K or at % K == first + col), (K, T, t, first, col)


def test_key_ranges_of_a_query_block(attention):
    """Causal attention, one piece or split: ragged rows, keys and windows, the smallest and the largest; the program checks every block's ranges."""
    rows, behind, windows = (1, 15, 16, 17, 63, 64, 65, 95, 509, 1000), (0, 1, 31, 32, 64, 300, 8191, 1 << 20), (0, 1, 31, 32, 33, 64, 500)
    shapes = [(t, t + b, heads, hd, w) for t in rows for b in behind for w in windows for heads, hd in ((1, 64), (8, 128), (40, 128))]
    shapes += [(33, 0x3FFFFFFF, 1, 64, 0), (33, 0x3FFFFFFF, 1, 64, 4096), (0x3FFFFF, 0x3FFFFF, 1, 128, 0)]
    got = attention(shapes)
    assert len(got) == len(shapes) and all(most == 0 or 2 <= most and ranges <= 32 for most, ranges in got)


def test_keys_are_split_where_that_is_faster(attention):
    """Both sides timed on 256 CUs: us in one piece, us split."""
    timed = {(390, 451, 64, 128, 0): (42.0, 53.4), (834, 870, 32, 128, 433): (52.9, 59.5), (750, 978, 32, 64, 337): (32.4, 36.3), (655, 655, 40, 128, 0): (53.7, 57.5),
             (628, 735, 40, 128, 0): (60.7, 64.3), (341, 341, 64, 128, 0): (31.9, 32.9), (719, 1125, 40, 64, 0): (59.4, 60.1), (205, 205, 64, 64, 0): (12.6, 13.3),
             (95, 722, 8, 128, 0): (54.4, 14.2), (509, 809, 40, 128, 0): (71.9, 56.8), (751, 751, 32, 128, 0): (60.6, 50.4), (923, 1395, 20, 64, 0): (66.6, 47.0),
             (130, 176, 40, 128, 0): (18.3, 15.6), (767, 767, 16, 64, 261): (20.4, 17.7), (589, 1561, 40, 64, 0): (80.0, 69.1), (406, 406, 40, 128, 0): (34.3, 32.8)}
    for (shape, (whole, split)), (most, _) in zip(timed.items(), attention(list(timed))):
        assert (most > 0) == (split < whole), shape


def test_the_tile_of_a_prompt_product(gemm):
    """Every tile timed, us, on 256 CUs. The estimate is off by 10 % rms, so the tile it prefers may be behind another by twice that, on either side, and no more."""
    timed = {
        (Q6_K, 1376, 12544, 126): (25.9, 28.7, 41.8, 34.4, 24.1, 22.6, 28.7, 30.9, 22.4, 24.8, 23.0, 23.4, 27.5),
        (Q5_K, 1288, 12032, 623): (46.9, 43.0, 58.6, 50.7, 44.9, 48.6, 47.3, 50.1, 53.1, 47.4, 43.6, 54.9, 67.2),
        (Q6_K, 2480, 9984, 215): (38.6, 39.8, 47.6, 34.6, 35.5, 31.7, 40.4, 45.3, 39.0, 38.5, 41.5, 37.5, 57.3),
        (Q6_K, 4368, 1536, 1330): (45.0, 33.4, 47.3, 51.9, 47.6, 44.4, 48.5, 48.5, 49.4, 47.9, 63.4, 44.2, 96.0),
        (Q4_K, 1288, 12800, 118): (20.7, 19.9, 30.2, 24.9, 21.6, 15.9, 20.2, 21.6, 17.7, 19.3, 16.9, 17.1, 22.2),
        (Q4_K, 1760, 1024, 356): (13.8, 15.4, 23.8, 19.7, 14.8, 11.4, 16.6, 14.7, 11.4, 12.5, 7.3, 12.5, 13.4),
        (Q5_K, 2280, 1792, 184): (15.5, 17.4, 24.9, 21.1, 17.2, 15.2, 17.9, 18.1, 15.1, 17.1, 14.0, 17.0, 10.3),
        (Q5_K, 4112, 3840, 1786): (91.3, 65.7, 95.1, 91.6, 75.7, 108.2, 103.6, 99.4, 122.8, 97.7, 117.5, 101.4, 190.6),
        (Q6_K, 19880, 4352, 136): (63.1, 71.9, 76.2, 71.8, 70.2, 65.8, 77.7, 86.7, 81.5, 74.0, 91.5, 85.5, 143.7),
        (Q6_K, 2096, 1792, 46): (12.3, 14.7, 19.6, 17.5, 12.3, 10.2, 15.1, 14.5, 9.8, 11.0, 10.1, 11.8, 12.5),
        (Q8_0, 4192, 1280, 542): (29.9, 34.2, 36.7, 40.1, 20.3, 25.2, 33.0, 20.4, 28.7, 19.8, 28.7, 28.4, 38.3),
        (Q8_0, 2384, 2816, 239): (25.2, 23.6, 32.8, 26.6, 25.0, 21.3, 29.8, 23.8, 20.6, 22.5, 19.0, 21.4, 25.0)}
    for shape, us in timed.items():
        assert us[plan(gemm, *shape)[0]] <= 1.25 * min(us), shape


def test_where_the_runs_of_run_sums_end(gemm):
    """fhip_gemm_q_bf16_run_sums promises the order of its sums from version to version: a tile's rows and outputs, the whole tiles of a workgroup and the chunks of a run are
    that order, on 256 CUs, and stand as they are here whatever the launches without that promise come to prefer."""
    order = {
        (Q6_K, 2049, 5120, 33): (64, 256, 0, 1), (Q6_K, 9000, 1280, 65): (128, 256, 0, 1), (Q5_K, 4100, 2304, 520): (128, 256, 0, 3),
        (Q4_K, 4100, 1280, 129): (256, 256, 0, 1), (Q8_0, 9000, 736, 128): (256, 256, 0, 1), (Q8_0, 5120, 512, 40): (256, 160, 0, 1),
        (Q4_K, 7000, 256, 300): (128, 128, 0, 1), (Q5_K, 7000, 1280, 300): (128, 128, 0, 5), (Q4_K, 1283, 512, 300): (128, 128, 0, 1),
        (Q6_K, 2049, 5120, 300): (128, 128, 0, 4), (Q6_K, 700, 1792, 65): (128, 128, 0, 1), (Q8_0, 2049, 2080, 64): (128, 160, 0, 1),
        (Q8_0, 9000, 512, 257): (128, 160, 0, 2), (Q5_K, 9000, 512, 40): (64, 128, 0, 1), (Q4_K, 7000, 2304, 33): (64, 128, 0, 2),
        (Q5_K, 7000, 1792, 257): (64, 128, 1, 1), (Q4_K, 7000, 256, 100): (64, 128, 0, 1), (Q8_0, 1283, 4064, 33): (64, 128, 0, 1),
        (Q8_0, 5120, 1312, 64): (64, 128, 0, 1), (Q6_K, 7000, 3328, 64): (64, 128, 0, 3), (Q6_K, 5120, 1280, 300): (64, 128, 0, 5),
        (Q4_K, 7168, 5120, 509): (256, 256, 0, 5), (Q4_K, 5120, 5120, 509): (256, 160, 0, 5), (Q4_K, 34816, 5120, 509): (256, 256, 1, 2),
        (Q6_K, 5120, 17408, 509): (256, 160, 0, 17), (Q4_K, 34816, 5120, 2048): (256, 256, 4, 5), (Q6_K, 5120, 17408, 2048): (256, 160, 1, 1),
        (Q4_K, 7168, 5120, 64): (64, 128, 0, 5), (Q5_K, 3072, 2048, 700): (256, 256, 0, 2), (Q8_0, 12288, 4096, 128): (128, 160, 0, 5),
        (Q6_K, 4096, 8960, 882): (256, 256, 0, 9)}
    for shape, runs in order.items():
        assert plan(gemm, *shape, run_sums=True)[1:5] == runs, shape


@pytest.fixture(scope="module")
def f16x2(tmp_path_factory):
    lib = C.CDLL(build(tmp_path_factory.mktemp("f16x2"), "f16x2_rules_harness.cpp", [], ["-shared", "-Wl,-Bsymbolic"]))
    lib.h_held.argtypes = [C.c_uint32, C.c_size_t, C.c_size_t, C.c_size_t]
    lib.h_resident.argtypes = lib.h_held.argtypes + [C.POINTER(C.c_int64)]
    return lib


def test_the_kernel_of_a_small_batch(f16x2):
    """Sums in order, both kernels timed, us: the held one, the one whose operand rows lie in LDS (cold weights, 256 CUs). The rule may be off by a tenth, as near its lines, and no more."""
    timed = {
        (Q4_K, 515, 512, 8): (3.8, 4.2), (Q4_K, 34816, 256, 8): (7.3, 5.1), (Q4_K, 8200, 256, 16): (5.4, 4.4), (Q4_K, 4090, 1280, 8): (5.5, 5.6), (Q4_K, 8200, 1280, 8): (7.6, 6.2),
        (Q4_K, 34816, 1280, 8): (13.0, 10.9), (Q6_K, 16400, 3072, 8): (16.6, 18.3), (Q8_0, 20000, 2784, 8): (20.8, 23.3), (Q4_K, 4090, 1024, 16): (5.4, 7.0), (Q4_K, 34816, 1280, 16): (22.8, 13.4),
        (Q4_K, 12000, 2048, 16): (11.4, 12.7), (Q6_K, 20000, 2048, 16): (16.6, 18.4), (Q4_K, 8200, 3584, 16): (14.8, 13.1), (Q8_0, 4090, 2272, 32): (12.7, 14.0), (Q8_0, 6100, 2272, 32): (17.2, 14.9),
        (Q4_K, 34816, 1024, 32): (25.9, 16.1), (Q5_K, 2050, 3584, 32): (12.1, 10.3), (Q4_K, 5130, 6144, 8): (15.7, 11.1), (Q6_K, 515, 6144, 32): (11.4, 9.4), (Q4_K, 100, 4352, 16): (10.2, 7.4),
        (Q6_K, 151936, 5120, 8): (148.9, 164.4), (Q6_K, 8200, 5120, 8): (18.0, 16.2), (Q8_0, 80000, 5632, 8): (115.3, 137.6), (Q6_K, 151936, 3584, 16): (110.8, 136.7),
        (Q8_0, 151936, 3584, 16): (153.5, 174.0), (Q4_K, 151936, 5120, 16): (192.5, 131.7), (Q6_K, 128256, 2560, 8): (76.0, 68.9), (Q8_0, 100000, 5120, 12): (212.3, 153.5)}
    for shape, (held, resident) in timed.items():
        assert (held, resident)[f16x2.h_held(*shape) == 0] <= 1.1 * min(held, resident), shape


@pytest.mark.parametrize("ty,block", [(Q4_K, 256), (Q5_K, 256), (Q6_K, 256), (Q8_0, 32)])
def test_ranges_of_k_of_a_small_batch(f16x2, ty, block):
    """A range's operand rows fit the LDS, no range is empty, the workgroups are no more than the CUs unless K alone asks for them, and the partial outputs fit the space asked for; from one
    chunk to the longest rows."""
    out, cus = (C.c_int64 * 6)(), 256
    for cols in sorted({block, 256, 288 // block * block, *range(256, 65537, 1280 if block == 256 else 1248), 16640, 16896 if block == 256 else 16672, 65536}):
        for rows in (1, 17, 700, 5120, 151936):
            for t in (3, 8, 9, 16, 17, 24, 32):
                f16x2.h_resident(ty, rows, cols, t, out)
                nt, sets, parts, per_part, most, ws = out
                chunks = (cols + 255) // 256
                assert 8 * nt * sets >= t and 1 <= parts <= chunks and (chunks + parts - 1) // parts <= most, (rows, cols, t)
                assert 1 <= per_part <= (rows + 15) // 16 and (per_part == 1 or parts * sets * per_part <= cus), (rows, cols, t)
                assert ws >= (parts * t * rows * 4 if parts > 1 else 0), (rows, cols, t)


class Weight(C.Structure):
    """struct fhip_weight (ferric_amd/csrc/common.hpp), for a query that reads its type and shape."""
    _fields_ = [("type", C.c_uint32), ("rows", C.c_size_t), ("cols", C.c_size_t), ("row_bytes", C.c_size_t), ("nbytes", C.c_size_t), ("d_raw", C.c_void_p), ("owns", C.c_bool),
                ("planes", C.c_int), ("batch_policy", C.c_int)]


@pytest.mark.parametrize("ty,rows,cols", [(Q4_K, 5120, 5120), (Q6_K, 5120, 17408), (Q8_0, 1283, 4064)])
def test_workspace_of_every_batch_a_launch_accepts(ty, rows, cols):
    """What batches of up to that many rows need at most: never less for more rows, and no more behind the largest batch that a launch accepts."""
    from ferric_amd import _lib
    lib, w = _lib.load(), Weight(ty, rows, cols)
    ask = lambda t: lib.fhip_workspace_bytes_coop(C.addressof(w), None, t)
    sizes = [ask(t) for t in (0, 1, 8, 9, 32, 33, 64, 65, 100, 509, 512, 1000, 2048, 4096)]
    assert sizes[0] == 0 and sizes == sorted(sizes) and sizes[-1] > 0
    accepted = (2 ** 31 - 1) // cols
    assert ask(accepted) == ask(accepted + 1) == ask(2 ** 64 - 64) == ask(2 ** 64 - 1) >= sizes[-1]
