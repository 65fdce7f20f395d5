"""F-statistic cells of every filter length, 16 to 2048 bins, in each TDI
format, against the oracle: a length below a wave, of one wave, of several
and of several series, cells whose filters reach past the segment, and cells
no length holds.  The gate is the fixed one of the F-statistic (1e-10
relative; the fitted parameters 1e-7)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

YEAR = 3.15581497632e7


@pytest.mark.parametrize("N,years,f,fmt", [(16, 0.5, 3e-4, "sangria"), (32, 0.5, 3e-3, "phase"),
                                           (64, 2, 3e-3, "frequency"), (128, 2, 8e-3, "phase"),
                                           (256, 2, 20e-3, "sangria"), (512, 4, 20e-3, "frequency"),
                                           (1024, 2, 50e-3, "phase"), (2048, 4, 50e-3, "sangria")])
def test_every_filter_length(gl, orc, N, years, f, fmt):
    import torch
    from glass_amd.fstat import Fstat
    T, NFFT, n = YEAR * years, 4096, 12
    rng = np.random.default_rng(N)
    o = orc.analytic_orbit()
    qmin0 = int(f * T) - NFFT // 2
    C00 = 1e-40 * rng.uniform(0.5, 2.0, NFFT)
    X, A, E = (np.sqrt(C00) * (rng.standard_normal(NFFT) + 1j * rng.standard_normal(NFFT)) for _ in range(3))
    off = rng.uniform(-0.3, 0.3, n) * NFFT / 2
    off[0], off[1] = -NFFT / 2 + 0.3 * N, NFFT / 2 - 0.3 * N  # a fifth of the filter outside
    cells = np.stack([f + off / T, rng.uniform(-1, 1, n) * 1e-17, np.arccos(rng.uniform(-0.9, 0.9, n)),
                      rng.uniform(0, 2 * np.pi, n)], axis=1)
    fd = orc.FstatData(T, qmin0, X, A, E, C00, fmt=fmt, orbit=o)
    F = Fstat(gl.analytic_orbit(), fmt, T, 0.0, qmin0, X, A, E, C00, max_cells=n)
    lx, la, fp = (t.cpu().numpy() for t in F.eval(torch.tensor(cells, device="cuda")))
    lengths = set()
    for c in range(n):
        rx, ra, rp, M = fd.logl(*cells[c])
        lengths.add(M)
        assert abs(lx[c] - rx) < 1e-10 * abs(rx) and abs(la[c] - ra) < 1e-10 * abs(ra), (c, M)
        assert np.max(np.abs(fp[c] - rp)) < 1e-7, (c, M, fp[c], rp)
    assert N in lengths
    F.close()


def test_mixed_lengths_and_none(gl, orc):
    """Cells of all lengths in one call; past 2048 bins the outputs are NaN."""
    import torch
    from glass_amd.fstat import Fstat
    T, NFFT = 4 * YEAR, 20000
    rng = np.random.default_rng(7)
    o = orc.analytic_orbit()
    f = 95e-3
    qmin0 = int(f * T) - NFFT // 2
    C00 = np.full(NFFT, 1e-40)
    X, A, E = (1e-20 * (rng.standard_normal(NFFT) + 1j * rng.standard_normal(NFFT)) for _ in range(3))
    n = 40
    cells = np.stack([f + rng.uniform(-0.2, 0.2, n) * NFFT / T, np.zeros(n), np.arccos(rng.uniform(-1, 1, n)),
                      rng.uniform(0, 2 * np.pi, n)], axis=1)
    cells[::2, 1] = 10.0 ** rng.uniform(-13, -11, n // 2)
    F = Fstat(gl.analytic_orbit(), "sangria", T, 0.0, qmin0, X, A, E, C00, max_cells=n)
    lx, la, fp = (t.cpu().numpy() for t in F.eval(torch.tensor(cells, device="cuda")))
    fd = orc.FstatData(T, qmin0, X, A, E, C00, orbit=o)
    M = np.array([orc.ucb_bandwidth(c[0], c[1], np.cos(c[2]), 1e-22, T, NFFT, orbit=o) for c in cells])
    assert (M > 2048).any()
    for c in range(n):
        if M[c] > 2048:
            assert np.isnan(lx[c]) and np.isnan(la[c]) and np.isnan(fp[c]).all()
        else:
            rx, ra, rp, _ = fd.logl(*cells[c])
            assert abs(lx[c] - rx) < 1e-10 * abs(rx) and abs(la[c] - ra) < 1e-10 * abs(ra)
    F.close()


def test_more_cells_than_a_new_plan_has_buffers_for(gl, orc):
    """A new plan has work buffers for 131,072 cells: more give what their parts
    give, bit for bit, before and after the buffers have grown."""
    import torch
    from glass_amd.fstat import Fstat
    T, NFFT, n, turn = YEAR, 3000, 131072 * 2 + 77, 131072
    rng = np.random.default_rng(9)
    f = 3e-3
    qmin0 = int(f * T) - NFFT // 2
    C00 = np.full(NFFT, 1e-40)
    X, A, E = (1e-20 * (rng.standard_normal(NFFT) + 1j * rng.standard_normal(NFFT)) for _ in range(3))
    cells = np.stack([f + rng.uniform(-0.2, 0.2, n) * NFFT / T, np.zeros(n), np.arccos(rng.uniform(-1, 1, n)),
                      rng.uniform(0, 2 * np.pi, n)], axis=1)
    F = Fstat(gl.analytic_orbit(), "sangria", T, 0.0, qmin0, X, A, E, C00, max_cells=n)
    c = torch.tensor(cells, device="cuda")
    before = F.eval(c[:turn])
    whole = F.eval(c)
    assert all(torch.equal(w[:turn], p) for w, p in zip(whole, before))
    for a, b in ((0, 1000), (turn - 500, turn + 500), (turn, 2 * turn), (2 * turn - 3, n)):
        part = F.eval(c[a:b])
        assert all(torch.equal(w[a:b], p) for w, p in zip(whole, part))
    fd = orc.FstatData(T, qmin0, X, A, E, C00, orbit=orc.analytic_orbit())
    for e in (0, turn - 1, turn, n - 1):
        rx, ra, *_ = fd.logl(*cells[e])
        assert abs(float(whole[0][e]) / rx - 1) < 1e-10 and abs(float(whole[1][e]) / ra - 1) < 1e-10
    F.close()
