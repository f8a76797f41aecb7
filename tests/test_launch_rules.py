"""What the launchers decide on the host, without a device: the sources are compiled for the host alone and asked."""
import ctypes as C
import os
import subprocess

import pytest

from conftest import ROOT


def build(d, harness, *flags):
    """tests/<harness> as a shared object."""
    obj, so = str(d / (harness + ".o")), str(d / (harness + ".so"))
    subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "--offload-host-only", "--offload-arch=gfx950", "-x", "hip", "-std=c++17", "-O1", "-fPIC", "-fuse-cuid=none",
                    *flags, "-c", os.path.join(ROOT, "tests", harness), "-o", obj], check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    subprocess.run(["g++", "-shared", "-Wl,-Bsymbolic", "-o", so, obj], check=True)
    return C.CDLL(so)


@pytest.fixture(scope="module")
def gemm(tmp_path_factory):
    return build(tmp_path_factory.mktemp("gemm"), "gemm_rules_harness.cpp", "-DFHIP_GEMM_FORMAT=Q80")


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
