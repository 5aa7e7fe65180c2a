"""The rules a walk is launched by (spinwalk_amd/csrc/launch_rules.hpp), on the host
build of the same header: sorting begins at fewer spins where steps are long."""
import ctypes
import os
import subprocess
import tempfile

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

CODE = r'''
#include "%s"
extern "C" unsigned unsorted(double step) { return sw::unsorted_spins(step); }
extern "C" int order(unsigned n, unsigned long long bytes, double step) { return sw::order_pays(n, bytes, step); }
'''


@pytest.fixture(scope="module")
def rules():
    src = os.path.abspath(os.path.join(HERE, "..", "spinwalk_amd", "csrc", "launch_rules.hpp"))
    with tempfile.TemporaryDirectory() as d:
        cpp, so = os.path.join(d, "r.cpp"), os.path.join(d, "r.so")
        with open(cpp, "w") as f:
            f.write(CODE % src)
        subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-o", so, cpp], check=True)
        lib = ctypes.CDLL(so)
        d_ = ctypes.c_double
        lib.unsorted.argtypes, lib.unsorted.restype = [d_], ctypes.c_uint
        lib.order.argtypes = [ctypes.c_uint, ctypes.c_ulonglong, d_]
        yield lib


def test_sorting_begins_at_fewer_spins_where_steps_are_long(rules):
    big = 64 << 20
    assert not rules.order(212992, big, 0.31) and rules.order(212993, big, 0.31)
    assert not rules.order(212992, big, 0.0)
    for step, unsorted, sort in ((0.63, 131072, 200000), (1.26, 65536, 131072), (2.5, 65536, 131072), (1e9, 90000, 90001)):
        assert not rules.order(unsorted, big, step) and rules.order(sort, big, step)
    assert not rules.order(10 ** 6, (4 << 20) - 1, 2.5) and rules.order(10 ** 6, 4 << 20, 2.5)
    for step in (float("inf"), float("nan")):
        assert 90000 <= rules.unsorted(step) <= 212992
    assert all(rules.unsorted(s / 100) >= rules.unsorted((s + 1) / 100) for s in range(1000))
