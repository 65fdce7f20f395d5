"""The host-array reductions on both sides of the sizes that choose how they are
staged (read from the pinned buffer up to 6 MB, 32 KB for the likelihood of two
channels) and how many blocks sum them (1024 bins each), against sums in
extended precision.  All terms have one sign or dominate, so a sum of n terms
agrees to n 2^-53 relative at most, 1e-13 at these sizes with pairwise partials."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# bytes a bin: fourier_nwip 40, snr 96, likelihood of 1 / 2 / 3 channels 80 (each
# array twice) / 80 / 168
SIZES = [1, 63, 64, 400, 409, 1024, 1025, 37440, 37460, 65530, 65550, 78630, 78660, 157270, 157300]
TOL = 1e-12


def inner(a, b, w):
    a, b, w = (np.asarray(v, dtype=np.clongdouble if np.iscomplexobj(v) else np.longdouble) for v in (a, b, w))
    return (a.real * b.real + a.imag * b.imag) * w


@pytest.mark.parametrize("N", SIZES)
def test_against_extended_precision(gl, N):
    rng = np.random.default_rng(N)
    d = rng.standard_normal((5, N)) + 1j * rng.standard_normal((5, N))
    m = 0.3 * (rng.standard_normal((5, N)) + 1j * rng.standard_normal((5, N)))
    C = np.zeros((3, 3, N + 5))  # snr reads the first N bins of longer planes
    for i in range(3):
        C[i, i] = rng.uniform(1.0, 2.0, N + 5)
    for i, j in ((0, 1), (0, 2), (1, 2)):
        C[i, j] = C[j, i] = rng.uniform(-0.2, 0.2, N + 5)

    def form(u, v):
        return sum(np.sum(inner(u[i], v[j], C[i, j, :N])) for i in range(3) for j in range(3))

    def close(got, ref):
        assert abs(got - ref) <= TOL * abs(ref), (N, got, ref)

    close(gl.fourier_nwip(d[0], d[0], C[0, 0], N), 2 * np.sum(inner(d[0], d[0], C[0, 0, :N])))
    close(gl.snr(d[0], d[1], d[2], C, N), np.sqrt(2 * form(d[:3], d[:3])))
    CN = np.ascontiguousarray(C[..., :N])
    r = d - m
    close(gl.gaussian_log_likelihood(d, m, CN), -form(r[:3], r[:3]))
    close(gl.gaussian_log_likelihood(d, m, CN, 1), -np.sum(inner(r[0], r[0], CN[0, 0])))
    close(gl.gaussian_log_likelihood(d, m, CN, 2),
          -np.sum(inner(r[3], r[3], CN[0, 0])) - np.sum(inner(r[4], r[4], CN[1, 1])))


@pytest.mark.parametrize("nmax,n", [(1, 1), (500, 500), (3000, 1025), (250000, 5000), (260000, 20000)])
def test_wavelet_nwip(gl, nmax, n):
    rng = np.random.default_rng(n)
    a, w = rng.standard_normal(nmax), rng.uniform(0.5, 2.0, nmax)
    lst = rng.permutation(nmax)[:n].astype(np.int32)
    ref = np.sum((np.asarray(a, np.longdouble) ** 2 * w)[lst])
    assert abs(gl.wavelet_nwip(a, a, w, lst) - ref) <= TOL * ref


@pytest.mark.parametrize("BW", [-4096, -1, 0, 8, 24, 8192])
def test_waveform_of_an_unsupported_length_is_refused(gl, BW):
    """... before anything is written to the staging buffer that BW sizes."""
    import ctypes
    o = gl.analytic_orbit()
    p = np.full(8, 0.3)
    out = np.full((5, 16), 7.0)
    dp = ctypes.POINTER(ctypes.c_double)
    rows = [r.ctypes.data_as(dp) for r in out]
    rc = gl.lib().glass_hip_ucb_waveform(ctypes.byref(o), b"sangria", 3e7, 0.0, p.ctypes.data_as(dp), 8, *rows, BW, 3)
    assert rc != 0 and f"BW={BW} unsupported" in gl.last_error() and np.all(out == 7.0)
