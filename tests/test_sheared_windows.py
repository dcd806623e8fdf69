"""The stencil rows across a sheared face are looked up by the window cells of a
wave's particles.  Whatever the positions are, also after a run has diverged, the
rows have to stay inside three periods of the cells (the pieces that the scan
splits a row into), and positions in the box keep the cell that they had."""
import ctypes
import math
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mcf_amd", "csrc")


@pytest.fixture(scope="module")
def window_cell(tmp_path_factory):
    d = tmp_path_factory.mktemp("window")
    (d / "w.cpp").write_text('#include "sdpd_window.h"\n'
                             'extern "C" int w(double x, int c, double cs, double sp) '
                             '{ return sdpd::window_cell(x, c, cs, sp); }\n')
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", CSRC, "-o",
                    str(d / "w.so"), str(d / "w.cpp")], check=True)
    f = ctypes.CDLL(str(d / "w.so")).w
    f.argtypes = [ctypes.c_double, ctypes.c_int, ctypes.c_double, ctypes.c_double]
    return f


LOST = [math.nan, math.inf, -math.inf, 1e300, -1e300, 1e10, -1e10, -3.0, 500.0]


@pytest.mark.parametrize("nm0", [6, 8, 10, 42, 128])
def test_rows_stay_within_three_periods(window_cell, nm0):
    rng = np.random.default_rng(nm0)
    cs = 1.53
    L = nm0 * cs
    for _ in range(3000):
        xmin = int(rng.integers(nm0))
        xmax = int(rng.integers(xmin, nm0))
        sp = float(rng.choice([0.0, np.nextafter(L, 0.0), rng.random() * L]))
        wc = []
        for cx in [xmin, xmax] + list(rng.integers(xmin, xmax + 1, size=6)):
            cx = int(cx)
            if rng.random() < 0.3:
                x = float(rng.choice(LOST))
            else:  # in its cell, or a quarter of one outside
                x = (cx + rng.uniform(-0.25, 1.25)) * cs
                assert window_cell(x, cx, cs, sp) == math.floor((x - sp) / cs)
            wc.append(window_cell(x, cx, cs, sp))
        vlo, aend = min(wc) - 2, max(wc) + 3
        m0 = vlo // nm0
        assert aend <= (m0 + 3) * nm0
        assert vlo >= -2 * nm0 - 3 and aend <= 2 * nm0 + 3
