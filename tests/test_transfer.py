"""Uploads (ferric_amd/csrc/transfer.hip) on the CPU, over a runtime whose streams do nothing before somebody waits for them and whose pinned memory can run out."""
import ctypes as C
import shutil

import numpy as np
import pytest

from test_launch_rules import build

KIB, MIB = 1 << 10, 1 << 20


@pytest.fixture(scope="module")
def library(tmp_path_factory):
    return build(tmp_path_factory.mktemp("transfer"), "transfer_harness.cpp", [], ["-shared", "-Wl,-Bsymbolic", "-lpthread"])


@pytest.fixture
def bus(library, tmp_path):
    path = str(tmp_path / "bus.so")               # a copy of its own: the slots are as old as the library
    shutil.copy(library, path)
    c = C.CDLL(path)
    for name in ("h_upload", "h_h2d", "h_d2h"):
        getattr(c, name).argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_void_p]
    c.h_waiting.restype, c.h_waiting.argtypes = C.c_size_t, [C.c_void_p]
    c.h_pinned.restype = C.c_size_t
    c.h_no_more_pinned.argtypes = [C.c_size_t]
    return c


def upload(bus, n, stream=16):
    """(what has arrived when the call returns, what should have)"""
    a = np.random.default_rng(n).integers(0, 256, n, np.uint8)
    d = np.zeros(n, np.uint8)
    assert bus.h_upload(d.ctypes.data, a.ctypes.data, n, stream) == 0
    return d, a


@pytest.mark.parametrize("n", [640 * KIB + 1, MIB, MIB + 1, 1280 * KIB + 1, 2 * MIB, 7 * MIB + 260, 12 * MIB, 12 * MIB + 1])
def test_a_long_upload_has_arrived_when_it_returns(bus, n):
    """Also behind other work of its stream: what follows on another stream may read it."""
    small, there = np.ones(100, np.uint8), np.zeros(100, np.uint8)
    assert bus.h_h2d(there.ctypes.data, small.ctypes.data, 100, 16) == 0 and bus.h_waiting(16) == 1
    d, a = upload(bus, n)
    assert np.array_equal(d, a) and bus.h_waiting(16) == 0


def test_a_short_upload_waits_for_nobody(bus):
    d, a = upload(bus, 640 * KIB)
    assert not d.any() and bus.h_waiting(16) == 1 and bus.h_runtime_copies() == 0


@pytest.mark.parametrize("slots", [0, 3])
def test_an_upload_needs_no_pinned_memory(bus, slots):
    """None left, or none left half way: the runtime's copy does it, as it did before there were slots for these sizes, and nothing of the failure stays behind."""
    upload(bus, 100)
    bus.h_no_more_pinned(slots * MIB)
    d, a = upload(bus, 7 * MIB)
    assert np.array_equal(d, a) and bus.h_runtime_copies() == 1 and bus.h_stale_error() == 0
    if slots:
        d, a = upload(bus, 3 * MIB)               # in the slots there are
        assert np.array_equal(d, a) and bus.h_runtime_copies() == 1


def test_slots_for_uploads_are_as_large_as_what_goes_through_them(bus):
    upload(bus, 100)
    before = bus.h_pinned()
    upload(bus, 12 * MIB)
    assert bus.h_pinned() - before == 12 * MIB


def test_an_upload_without_slots_is_the_runtime_s(bus):
    """Others hold them: too few for seven chunks, enough for two."""
    bus.h_hold_upload_slots(7)
    d, a = upload(bus, 7 * MIB)
    assert np.array_equal(d, a) and bus.h_runtime_copies() == 1
    d, a = upload(bus, 2 * MIB)
    assert np.array_equal(d, a) and bus.h_runtime_copies() == 1


@pytest.mark.parametrize("n,by_runtime", [(640 * KIB, 0), (640 * KIB + 1, 0), (MIB, 0), (MIB + 1, 0), (12 * MIB, 0), (12 * MIB + 1, 1)])
def test_who_takes_an_upload(bus, n, by_runtime):
    upload(bus, n)
    assert bus.h_runtime_copies() == by_runtime
