"""The sine, cosine and transfer-function polynomials of the slow series
(glass_amd/csrc/fastmath.h: sincos_half, sinc_phase, sinc_values), compiled
for the host and compared with 150-bit mpmath values.  Bounds: a few units
of 2^-53 relative to 1 (the polynomials' own errors are below 1e-17)."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

mp = pytest.importorskip("mpmath")
mp.mp.prec = 150
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EPS = 2.0 ** -53


@pytest.fixture(scope="module")
def fm(tmp_path_factory):
    d = tmp_path_factory.mktemp("fs")
    src = d / "fs.cpp"
    src.write_text('#include "fastmath.h"\n'
                   'extern "C" void f_sincos(const double* x, double* s, double* c, int n) {'
                   ' for (int i = 0; i < n; i++) { double a[1] = {x[i]}, u[1], v[1]; unsigned f[1];'
                   ' glass::sincos_half<1>(a, u, v, f);'
                   ' s[i] = glass::flip_sign(u[0], f[0]); c[i] = glass::flip_sign(v[0], f[0]); } }\n'
                   'extern "C" void f_sinc(const double* x, double fmax, double* o, int n) {'
                   ' bool w = glass::sinc_wide(fmax); for (int i = 0; i < n; i++) {'
                   ' double a[1] = {x[i]}, r[1], m[1], s[1], c[1], d[1];'
                   ' glass::sinc_phase<1>(a, w, r, m); glass::sinc_values<true, 1>(a, w, s, c, d);'
                   ' double* q = o + 5 * i; q[0] = r[0]; q[1] = m[0]; q[2] = s[0]; q[3] = c[0]; q[4] = d[0]; } }\n')
    with src.open("a") as f:
        f.write('extern "C" void f_sctab(const double* x, double* s, double* c, int n) {'
                ' glass::dd_t t[256]; for (int i = 0; i < 256; i++) t[i] = glass::sin_tab_entry(i);'
                ' for (int i = 0; i < n; i++) { glass::sc_t v = glass::sincos_tab(x[i], t);'
                ' s[i] = v.s; c[i] = v.c; } }\n')
    so = d / "fs.so"
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-std=c++17", "-shared", "-fPIC", "-I",
                    os.path.join(ROOT, "glass_amd", "csrc"), str(src), "-o", str(so)], check=True)
    L = ctypes.CDLL(str(so))
    dp = ctypes.POINTER(ctypes.c_double)
    L.f_sincos.argtypes = [dp, dp, dp, ctypes.c_int]
    L.f_sctab.argtypes = [dp, dp, dp, ctypes.c_int]
    L.f_sinc.argtypes = [dp, ctypes.c_double, dp, ctypes.c_int]
    return L, dp


@pytest.mark.parametrize("lo,hi", [(-2.0, 2.0), (-60.0, 60.0), (1e6, 3e7), (-5.3e8, -2e8)])
def test_sincos_half(fm, lo, hi):
    L, dp = fm
    x = np.random.default_rng(3).uniform(lo, hi, 2000)
    s, c = np.empty_like(x), np.empty_like(x)
    L.f_sincos(x.ctypes.data_as(dp), s.ctypes.data_as(dp), c.ctypes.data_as(dp), len(x))
    es = max(abs(float(mp.sin(mp.mpf(v)) - mp.mpf(a))) for v, a in zip(x, s))
    ec = max(abs(float(mp.cos(mp.mpf(v)) - mp.mpf(a))) for v, a in zip(x, c))
    assert es <= 2 * EPS and ec <= 2 * EPS, (es / EPS, ec / EPS)


def test_sincos_half_domain(fm):
    L, dp = fm
    x = np.array([0.0, -0.0, np.pi, 5.3e8, 2.0 ** 29, -1e10, np.inf, -np.inf, np.nan])
    s, c = np.empty_like(x), np.empty_like(x)
    L.f_sincos(x.ctypes.data_as(dp), s.ctypes.data_as(dp), c.ctypes.data_as(dp), len(x))
    fin = np.abs(x) < 2.0 ** 29
    assert np.allclose(s[fin], np.sin(x[fin]), rtol=0, atol=3e-16) and np.all(np.isnan(s[~fin]) & np.isnan(c[~fin]))


@pytest.mark.parametrize("fmax", [1e-3, 0.5, 1.4, 1.41, 2.8, 2.81, 6.0])
def test_transfer_function(fm, fmax):
    """Every argument the frequency bound fmax = f/f* admits, 0 among them."""
    L, dp = fm
    x = np.concatenate([[0.0, 1e-300], np.random.default_rng(5).uniform(0.0, 1.25 * fmax, 1500)])
    o = np.empty((len(x), 5))
    L.f_sinc(x.ctypes.data_as(dp), fmax, o.ctypes.data_as(dp), len(x))
    worst = np.zeros(5)
    for v, q in zip(x, o):
        m = mp.mpf(v)
        s = mp.sin(m) / m if v else mp.mpf(1)
        c = mp.cos(m)
        d = (c - s) / m if v > 1e-3 else -m / 3 + m ** 3 / 30
        worst = np.maximum(worst, [abs(float(a - mp.mpf(b))) for a, b in zip((s * c, -m * s * s, s, c, d), q)])
    # s, c, d and fr to 3 units; fi = x s s carries 2 |sin x| times the error
    # of s and two roundings of at most 0.73
    assert np.all(worst <= np.array([3, 4.5, 3, 3, 3]) * EPS), worst / EPS


@pytest.mark.parametrize("lo,hi", [(-0.05, 0.05), (-7.0, 7.0), (1e5, 2e6), (-5.3e8, 5.3e8)])
def test_sincos_tab_correctly_rounded(fm, lo, hi):
    """Errors below 2^-72 against half an ulp of a result that is mostly above
    2^-6: fewer than one in 2^13 arguments may round the other way, and those
    by one unit; 8000 arguments hold at most a handful."""
    L, dp = fm
    x = np.random.default_rng(17).uniform(lo, hi, 8000)
    x[:4] = 0.0, np.pi / 2, np.pi / 128 * 1.5, -np.pi
    s, c = np.empty_like(x), np.empty_like(x)
    L.f_sctab(x.ctypes.data_as(dp), s.ctypes.data_as(dp), c.ctypes.data_as(dp), len(x))
    off = 0
    for f, got in ((mp.sin, s), (mp.cos, c)):
        ref = np.array([float(f(mp.mpf(v))) for v in x])
        bad = got != ref
        off += int(bad.sum())
        assert np.all(np.abs(got - ref) <= np.spacing(np.abs(ref)))
    assert off <= 4, off
    y = np.array([2.0 ** 29, np.inf, -np.inf, np.nan])
    L.f_sctab(y.ctypes.data_as(dp), s.ctypes.data_as(dp), c.ctypes.data_as(dp), len(y))
    assert np.isnan(s[:4]).all() and np.isnan(c[:4]).all()
