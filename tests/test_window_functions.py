"""The kernels' own window tests (csrc/pm_window.h, compiled for the host) on random
windows: what window_inside and z_clear accept has only valid taps, what
window_outside accepts has none, tap by tap, and each agrees with its restatement in
test_window_bound.py and test_window_outside.py."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import __graft_entry__ as entry
import test_window_bound as bound
import test_window_outside as outside

f32 = np.float32
SOURCE = """
#include <cmath>
using std::fabs;
#define __device__
#define __forceinline__ inline
#include "pm_window.h"
extern "C" void windows(int n, const float* c, const float* h, float R, float W, float H,
                        unsigned char* in, unsigned char* out, unsigned char* clear)
{
    const float shrink = 0.99999904632568359375f;   // 1 - 2^-20
    for (int i = 0; i < n; ++i, c += 3, h += 6) {
        in[i] = hp3d::window_inside(c[0], c[1], c[2], h[0], h[1], h[2], h[3], h[4], h[5], R,
                                    (W - 1) * shrink, (H - 1) * shrink);
        out[i] = hp3d::window_outside(c[0], c[1], c[2], h[0], h[1], h[2], h[3], h[4], h[5], R, W, H);
        clear[i] = hp3d::z_clear(c[2], h[4], h[5], R);
    }
}
"""


@pytest.fixture(scope="module")
def compiled(tmp_path_factory):
    d = tmp_path_factory.mktemp("windows")
    (d / "windows.cpp").write_text(SOURCE)
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-fPIC", "-shared",
                           "-I", os.path.join(entry.PKG_DIR, "csrc"), "-o", str(d / "windows.so"),
                           str(d / "windows.cpp")])
    lib = ctypes.CDLL(str(d / "windows.so"))

    def run(c, h, R, W, H):
        c, h = np.ascontiguousarray(c, f32), np.ascontiguousarray(h, f32)
        got = [np.zeros(len(c), np.uint8) for _ in range(3)]
        lib.windows(len(c), c.ctypes.data_as(ctypes.c_void_p), h.ctypes.data_as(ctypes.c_void_p),
                    ctypes.c_float(R), ctypes.c_float(W), ctypes.c_float(H),
                    *[g.ctypes.data_as(ctypes.c_void_p) for g in got])
        return [g.astype(bool) for g in got]
    return run


def agree(a, b):
    # the restatements' FMA rounds twice: a window on a bound may fall to either side
    return (a != b).mean() <= 1e-4


@pytest.mark.parametrize("NT,ST", [(2, 2), (3, 1), (5, 1), (6, 2), (11, 1)])
@pytest.mark.parametrize("size", [(17, 13), (640, 480), (16384, 9000)])
def test_outside(compiled, NT, ST, size):
    W, H = size
    R = (NT - 1) * ST // 2
    rng = np.random.default_rng(NT * 1000 + W)
    for kind in ("near", "far", "grazing", "behind"):
        c, h = (x.astype(f32) for x in outside.windows(rng, 20000, W, H, max(R, 1), kind))
        _, got, clear = compiled(c, h, R, W, H)
        assert agree(got, outside.outside(c, h, R, W, H)), kind
        assert got.any() == (kind != "behind")
        assert not outside.any_valid(c[got], h[got], NT, ST, W, H, np.zeros((got.sum(), 2))).any()
        assert agree(clear, bound.z_clear(c, h, R))


@pytest.mark.parametrize("kind", ["edge", "tight", "inside"])
def test_inside(compiled, kind):
    W, H, NT = 640, 480, 11
    rng = np.random.default_rng(4)
    c, h = (x.astype(f32) for x in bound._windows(rng, 20000, W, H, kind))
    got, _, _ = compiled(c, h, 5, W, H)
    assert agree(got, bound.window_inside(c, h, 5, W, H))
    assert got.any() and bound.taps_valid(c[got], h[got], NT, 1, W, H).all()


def test_non_finite_windows_pass_no_test(compiled):
    c, h = np.ones((27, 3), f32), np.full((27, 3, 2), 0.1, f32)
    for i in range(27):
        bad = (np.nan, np.inf, -np.inf)[i % 3]
        (c if i < 9 else h).reshape(27, -1)[i, (i // 3) % 3 if i < 9 else (i - 9) // 3] = bad
    got_in, got_out, _ = compiled(c, h, 3, 640, 480)
    assert not got_in.any() and not got_out.any()
