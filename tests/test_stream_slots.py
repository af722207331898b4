"""Which device words a call finds its longest row in (csrc/stream_slots.hpp), on the CPU: calls that can be under
way at once never share them."""
import ctypes
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    path = str(tmp_path_factory.mktemp("slots") / "slots.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-Wall", "-shared", "-fPIC", "-pthread",
                           os.path.join(HERE, "support", "stream_slots_host.cpp"), "-o", path])
    so = ctypes.CDLL(path)
    so.slots_create.restype = ctypes.c_void_p
    return so


@pytest.fixture()
def slot(lib):
    h = ctypes.c_void_p(lib.slots_create())
    yield lambda stream, capture=0: lib.slots_of(h, ctypes.c_void_p(stream), ctypes.c_ulonglong(capture))
    lib.slots_destroy(h)


def test_captured_calls_share_with_their_own_graph_alone(slot):
    eager = [slot(0), slot(0x1000), slot(0x2000)]
    captured = [slot(0x1000, 1), slot(0x1000, 2), slot(0x2000, 2), slot(0, 3)]
    assert len(set(eager + captured)) == 7 and min(eager + captured) == 0
    assert [slot(0), slot(0x1000), slot(0x2000)] == eager                    # calls on one stream are ordered
    assert [slot(0x1000, 1), slot(0x1000, 2), slot(0x2000, 2), slot(0, 3)] == captured


def test_slots_run_out_for_new_ones_only(lib, slot):
    for count, call in ((lib.slots_streams(), lambda i: slot(16 * i)), (lib.slots_captures(), lambda i: slot(16, 1 + i))):
        first = [call(i) for i in range(count)]
        assert len(set(first)) == count and min(first) >= 0 and max(first) < lib.slots_streams() + lib.slots_captures()
        assert call(count) == -1 and call(count + 1) == -1
        assert [call(i) for i in range(count)] == first
