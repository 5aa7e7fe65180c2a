"""The rules a walk is launched by (spinwalk_amd/csrc/launch_rules.hpp), on the host
build of the same header: sorting begins at fewer spins where steps are long, and
the wave cap needs a step, not only large records."""
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
extern "C" int general(unsigned n, int f64, double step, int global) { return sw::general_loop(n, f64 != 0, step, global != 0); }
extern "C" double reach(double bytes, double vox, double n, int sorted, double step, double steps) {
    return sw::cap_reach((unsigned long long)bytes, vox, (unsigned long long)n, sorted != 0, step, steps);
}
extern "C" double window(double bytes, double vox, double n, int sorted, double drift) {
    return sw::cap_window((unsigned long long)bytes, vox, (unsigned long long)n, sorted != 0, drift);
}
extern "C" int cap(int kind, int one_tr, double reach, double window, double n) {
    return sw::cap_pays((sw::CapKind)kind, one_tr != 0, reach, window, (unsigned long long)n);
}
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
        d_, i = ctypes.c_double, ctypes.c_int
        lib.unsorted.argtypes, lib.unsorted.restype = [d_], ctypes.c_uint
        lib.order.argtypes = [ctypes.c_uint, ctypes.c_ulonglong, d_]
        lib.general.argtypes = [ctypes.c_uint, i, d_, i]
        lib.reach.argtypes, lib.reach.restype = [d_, d_, d_, i, d_, d_], d_
        lib.window.argtypes, lib.window.restype = [d_, d_, d_, i, d_], d_
        lib.cap.argtypes = [i, i, d_, d_, d_]
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


def test_general_loop_between_half_waves_and_two_waves(rules):
    for n, on in ((32768, False), (32769, True), (131072, True), (131073, False)):
        assert bool(rules.general(n, 0, 0.5, 0)) == on and bool(rules.general(n, 0, 0.1, 1)) == on
        assert not rules.general(n, 1, 0.5, 1) and not rules.general(n, 0, 0.49, 0)


def _reach(rules, side, bytes_per_voxel, n, step, steps, is_sorted=1):
    return rules.reach(side ** 3 * bytes_per_voxel, float(side) ** 3, n, is_sorted, step, steps)


def test_cap_needs_steps_as_well_as_records(rules):
    single, pairs, batch, fused = range(4)
    f32, q16 = 128 / 24, 128 / 36
    on = lambda kind, one, r, n=10 ** 6: bool(rules.cap(kind, one, r, 100.0, n))  # noqa: E731
    # single walks: 4e5 spins on 256^3
    assert on(single, 1, _reach(rules, 256, f32, 4e5, 0.32, 800))
    assert not on(single, 1, _reach(rules, 256, f32, 4e5, 0.16, 160))
    assert not on(single, 1, _reach(rules, 128, f32, 4e5, 0.32, 160))
    assert not on(single, 0, _reach(rules, 256, q16, 1e6, 0.32, 160))
    assert on(pairs, 1, _reach(rules, 500, f32, 5e5, 0.32, 800)) and not on(pairs, 1, _reach(rules, 500, f32, 2e6, 0.2, 160))
    assert on(batch, 0, _reach(rules, 400, f32, 1e5, 0.81, 5100)) and not on(batch, 0, _reach(rules, 256, q16, 2e5, 0.81, 440))
    assert on(fused, 0, _reach(rules, 1000, f32, 2e6, 0.316, 10100)) and not on(fused, 0, _reach(rules, 200, f32, 4e5, 0.32, 1100))
    # batches of one TR go by the records alone
    for side, capped in ((256, True), (190, True), (96, False)):
        w = rules.window(side ** 3 * f32, float(side) ** 3, 1e5, 1, 0.0)
        assert bool(rules.cap(batch, 1, 0.0, w, 10 ** 6)) == capped
    # below 6 waves a SIMD never
    assert not on(single, 1, 100.0, 393215) and on(single, 1, 100.0, 393216)


def test_reach_is_bounded_by_the_phantom(rules):
    whole = _reach(rules, 64, 5.0, 1e5, 2.0, 1e6)
    assert whole == pytest.approx(64 ** 3 * 5.0 / 2 ** 20 * 0.65 ** 2)
    assert _reach(rules, 64, 5.0, 1e5, 2.0, 0, is_sorted=0) == pytest.approx(whole)
    assert _reach(rules, 64, 5.0, 1e5, 2.0, 0) == pytest.approx(whole / 8)
