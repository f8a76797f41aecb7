"""What the launchers decide on the host, without a device: the sources are compiled for the host alone and asked."""
import ctypes as C
import os
import subprocess

import pytest

from conftest import ROOT


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


@pytest.fixture(scope="module")
def attention(tmp_path_factory):
    """[(rows, keys, heads, head size, window)] -> [(most key tiles of a range, ranges)]"""
    program = build(tmp_path_factory.mktemp("attn"), "attn_rules_harness.cpp", ["-Xarch_host", "-fsanitize=undefined", "-Xarch_host", "-fsanitize-trap=undefined"], [])

    def ask(shapes):
        r = subprocess.run([program], input="".join("%d %d %d %d %d\n" % x for x in shapes), capture_output=True, text=True)
        assert r.returncode == 0, (r.returncode, shapes[len(r.stdout.splitlines())])
        return [tuple(map(int, line.split())) for line in r.stdout.splitlines()]
    return ask


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
