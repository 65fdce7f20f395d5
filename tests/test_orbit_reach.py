"""How far the transfer functions' arguments reach is decided from the
spacecraft positions (OrbitReach, ucb_common.h): L and f* come with the orbit
and need not fit them.  The header's functions, compiled for the host, against
the positions themselves."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

import glass_amd as gl
from glass_amd import build, synth
from glass_amd import wdm as W

pytestmark = pytest.mark.skipif(shutil.which(build.HIPCC) is None and not os.path.exists(build.HIPCC),
                                reason="hipcc not available")

SRC = r"""
#include "ucb_common.h"
using namespace glass;
extern "C" int c_wide(const double* p, int np, double T, double t0, double L, double fstar, double arg, double time)
{
    UcbConst c;
    ucb_setup(p, np, T, t0, L, fstar, OrbitReach{arg, time}, c);
    return c.wide;
}
extern "C" void c_extent(const double* pos, int n, double* arm, double* far) { positions_extent(pos, n, arm, far); }
extern "C" void c_reach(double L, double fstar, double T, double t0, double arm, double far, double* o)
{
    const OrbitReach r = orbit_reach(L, fstar, T, t0, arm, far);
    o[0] = r.arg;
    o[1] = r.time;
}
extern "C" void c_analytic(double L, double fstar, double R, double T, double t0, double* o)
{
    const OrbitReach r = analytic_reach(L, fstar, R, T, t0);
    o[0] = r.arg;
    o[1] = r.time;
}
"""
D, DP = ctypes.c_double, ctypes.POINTER(ctypes.c_double)


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("reach")
    src, so = d / "r.hip", d / "r.so"
    src.write_text(SRC)
    flags = [f for f in build.FLAGS if f != "-O3"]
    subprocess.run([build.HIPCC] + flags + ["-O1", "--offload-host-only", "-shared", "-I", build.CSRC, str(src),
                                            "-o", str(so)], check=True)
    L = ctypes.CDLL(str(so))
    L.c_wide.argtypes = [DP, ctypes.c_int] + [D] * 6
    L.c_extent.argtypes = [DP, ctypes.c_int, DP, DP]
    L.c_reach.argtypes = [D] * 6 + [DP]
    L.c_analytic.argtypes = [D] * 5 + [DP]
    return L


def dp(a):
    return a.ctypes.data_as(DP)


def two(fn, *a):
    o = np.zeros(2)
    fn(*a, dp(o))
    return o


def extent(lib, x, y, z):
    """x, y, z [3, n]"""
    rec = np.ascontiguousarray(np.concatenate([x, y, z]).T)
    arm, far = D(), D()
    lib.c_extent(dp(rec), len(rec), ctypes.byref(arm), ctypes.byref(far))
    return arm.value, far.value


def arguments(p, T, t0, x, y, z, L, fstar):
    """Largest |transfer-function argument| over the links and samples."""
    n = x.shape[1]
    t = t0 + T * np.arange(n) / n
    st = np.sqrt(1 - p[1] ** 2)
    k = -np.array([st * np.cos(p[2]), st * np.sin(p[2]), p[1]])
    r = np.stack([x, y, z])
    worst = 0.0
    for i in range(3):
        xi = t - k @ r[:, i] / 299792458.0
        f = p[0] / T + p[7] / T ** 2 * xi + (0.5 * p[8] / T ** 3 * xi * xi if len(p) > 8 else 0.0)
        for j in range(3):
            if i != j:
                worst = max(worst, np.max(np.abs(0.5 * f / fstar * (1 + k @ (r[:, j] - r[:, i]) / L))))
    return worst


def test_extent(lib):
    rng = np.random.default_rng(1)
    x, y, z = rng.standard_normal((3, 3, 50)) * 1e11
    arm, far = extent(lib, x, y, z)
    r = np.stack([x, y, z])
    d = max(np.max(np.linalg.norm(r[:, i] - r[:, j], axis=0)) for i, j in ((0, 1), (1, 2), (2, 0)))
    assert abs(arm / d - 1) < 1e-14 and abs(far / np.max(np.linalg.norm(r, axis=0)) - 1) < 1e-14
    x[1, 7] = np.nan
    assert np.isnan(extent(lib, x, y, z)).all()
    p = synth.draw_params(rng, 1, 3e7)[0]
    assert np.isnan(two(lib.c_reach, 2.5e9, 0.019, 3e7, 0.0, np.nan, 1e11)[0])
    assert lib.c_wide(dp(p), 8, 3e7, 0.0, 2.5e9, 0.019, float("nan"), 3e7) == 1


@pytest.mark.parametrize("stretch", [0.3, 1.0, 1.6, 4.0])
def test_analytic_orbit(lib, stretch):
    o = gl.analytic_orbit()
    o.R *= stretch
    _, x, y, z = W.interpolated_analytic_orbit(o, synth.YEAR_T)
    arm, far = extent(lib, x, y, z)
    T = synth.YEAR_T
    got = two(lib.c_analytic, o.L, o.fstar, o.R, T, 5.0)
    tight = two(lib.c_reach, o.L, o.fstar, T, 5.0, arm, far)
    assert np.all(got >= tight) and np.all(got <= 1.01 * tight)
    if stretch == 1.0:
        assert got[0] == 1.25 / o.fstar and got[1] == 5.0 + T + 1000.0


def test_wide_wherever_an_argument_leaves_the_polynomials(lib):
    rng = np.random.default_rng(5)
    seen = {0: 0, 1: 0}
    for it in range(300):
        T, t0 = synth.YEAR_T * rng.uniform(0.02, 4), rng.choice([0.0, 1e8])
        L = 2.5e9 * np.exp(rng.uniform(-1.5, 1.5))
        fstar = 299792458.0 / (2 * np.pi * 2.5e9) * np.exp(rng.uniform(-1.0, 1.0))
        c = rng.standard_normal((3, 1, 40)) * rng.choice([1e10, 1.5e11, 1e13])
        x, y, z = c + rng.standard_normal((3, 3, 40)) * 2e9 * np.exp(rng.uniform(-1, 1, (1, 3, 1)))
        p = synth.draw_params(rng, 1, T)[0]
        f = np.exp(rng.uniform(np.log(1e-3), np.log(0.1)))
        p[0], p[7] = f * T, rng.uniform(-1, 1) * 0.3 * f * T * rng.choice([0.0, 1.0])
        if it % 3 == 0:
            p = np.append(p, rng.uniform(-1, 1) * 0.3 * f * T)
        arm, far = extent(lib, x, y, z)
        reach = two(lib.c_reach, L, fstar, T, t0, arm, far)
        wide = lib.c_wide(dp(p), len(p), T, t0, L, fstar, reach[0], reach[1])
        seen[wide] += 1
        if not wide:
            assert arguments(p, T, t0, x, y, z, L, fstar) <= 1.75 * (1 + 1e-12)
    assert min(seen.values()) > 50
