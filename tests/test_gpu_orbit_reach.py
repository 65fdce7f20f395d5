"""Orbits whose arms are not L (L and f* are the caller's): arguments of the
transfer functions leave the polynomials' range at frequencies where they would
not with arms of L.  Every Fourier-domain path on such an orbit against the
oracle, or against another path that is."""
import numpy as np
import pytest

from conftest import normwise
from glass_amd import synth

pytestmark = pytest.mark.gpu

T = synth.YEAR_T
F = 25e-3  # |f|/f* = 1.31: arguments to 1.31 with arms of L, to 3.3 with arms of 4 L


def gate(BW):
    # the oracle steps exp(i f/f*) from bin to bin: N 2^-53 after N bins
    return 1e-13 + 2 * BW * 2.0 ** -53 / abs(np.sin(F / synth.FSTAR))


def orbits(gl, orc, stretch):
    o, q = gl.analytic_orbit(), orc.analytic_orbit()
    o.R *= stretch
    q.R *= stretch
    return o, q


def source(seed, BW):
    p = synth.draw_params(np.random.default_rng(seed), 1, T)[0]
    p[0], p[7] = int(F * T) + seed % 7 + 0.37, 1e-17 * T * T
    return p


@pytest.mark.parametrize("stretch", [1.6, 4.0])
@pytest.mark.parametrize("BW", [16, 128, 512, 1024, 4096])
def test_waveform(gl, orc, BW, stretch):
    o, q = orbits(gl, orc, stretch)
    p = source(BW, BW)
    h = gl.ucb_waveform(o, "sangria", T, 0.0, p, 8, BW)
    assert normwise(h, orc.ucb_waveform(p, T, BW, orbit=q)) <= gate(BW)


@pytest.mark.parametrize("BW", [32, 512, 2048])
def test_numeric_orbit(gl, orc, BW):
    """One spacecraft far from the other two, and an L that fits neither."""
    t = np.linspace(-0.02 * T, 1.02 * T, 60)
    pos = np.zeros((9, len(t)))
    a = 2 * np.pi * t / synth.YEAR_T
    for i, off in enumerate((0.0, 2.5e9, 1.3e10)):
        pos[3 * i:3 * i + 3] = 1.496e11 * np.array([np.cos(a), np.sin(a), 0 * a]) + off * np.array(
            [np.sin(a + i), np.cos(a - i), 0.3 * np.sin(a)])
    no = gl.numeric_orbit(t, pos[0::3], pos[1::3], pos[2::3])
    p = source(BW + 1, BW)
    with orc.numeric_orbit(t, pos) as onum:
        no.L = onum.orbit.L = 2.5e9
        no.fstar = onum.orbit.fstar = synth.FSTAR
        ref = orc.ucb_waveform(p, T, BW, orbit=onum.orbit)
    assert normwise(gl.ucb_waveform_numeric(no, "sangria", T, 0.0, p, 8, BW), ref) <= gate(BW)


@pytest.mark.parametrize("BW", [64, 512, 1024, 2048])
def test_derivatives_and_gradient(gl, BW):
    import torch
    from glass_amd.derivs import source_derivs, source_grad
    o = gl.analytic_orbit()
    o.R *= 4.0
    W = BW
    rng = np.random.default_rng(BW)
    p = source(BW, BW)
    h = gl.ucb_waveform(o, "sangria", T, 0.0, p, 8, BW)[:3]
    w = np.zeros((6, W))
    w[:3], w[3:] = 1.0 / np.max(np.abs(h)) ** 2, 0.2 / np.max(np.abs(h)) ** 2
    R = 0.7 * h + 0.1 * np.max(np.abs(h)) * (rng.standard_normal((3, W)) + 1j * rng.standard_normal((3, W)))

    def logl(v):
        g = gl.ucb_waveform(o, "sangria", T, 0.0, v, 8, BW)[:3]
        x = R - 0.5 * g
        C = np.array([[w[0], w[3], w[4]], [w[3], w[1], w[5]], [w[4], w[5], w[2]]])
        return 2 * np.einsum("an,bn,abn->", x.conj(), g, C).real

    dev = dict(device="cuda")
    args = (o, T, torch.tensor(p[None], **dev), BW, torch.zeros(1, dtype=torch.int32, **dev),
            torch.tensor(w[None], **dev), torch.tensor(R[None], **dev))
    L, g, _ = source_derivs(*args)
    L, g = float(L[0]), g[0].cpu().numpy()
    # one template, another order of ~BW terms
    assert abs(L / logl(p) - 1) <= 1e-11
    # central differences, step s: truncation s^2, rounding 1e-10/s
    for k, s in ((0, 3e-5), (1, 1e-5), (2, 1e-5), (4, 1e-4), (5, 1e-4)):
        up, dn = p.copy(), p.copy()
        up[k] += s
        dn[k] -= s
        assert abs((logl(up) - logl(dn)) / (2 * s) - g[k]) <= 2e-5 * np.max(np.abs(g)), k
    if BW <= 1024:
        La, ga = source_grad(*args)
        assert abs(float(La[0]) / L - 1) <= 1e-11
        assert np.max(np.abs(ga[0].cpu().numpy() - g)) <= 1e-10 * np.max(np.abs(g))


def test_batched_evaluation(gl):
    """delta-logL of proposals against their waveforms' likelihoods."""
    from glass_amd.batch import FdBatch
    o = gl.analytic_orbit()
    o.R *= 4.0
    W, C = 600, 4
    rng = np.random.default_rng(3)
    qmin = int(F * T) - W // 2
    P = np.stack([source(10 + i, 0) for i in range(3 * C)])
    P[:, 0] = qmin + W // 2 + rng.uniform(-40, 40, 3 * C)
    h0 = gl.ucb_waveform(o, "sangria", T, 0.0, P[0], 8, 512)[:3]
    s = np.max(np.abs(h0))
    data = s * (rng.standard_normal((3, W)) + 1j * rng.standard_normal((3, W)))
    invC = np.zeros((3, 3, W))
    invC[[0, 1, 2], [0, 1, 2]] = 1.0 / s ** 2
    sp = np.zeros((C, 8, 8))
    sp[:, 0] = P[:C]
    plan = FdBatch(o, "sangria", T, 0.0, [qmin], [data], [invC], np.zeros(C, np.int32), np.ones(C, np.int32), sp, 2 * C)
    pc = np.repeat(np.arange(C), 2).astype(np.int32)
    plan.set_proposals(pc, np.zeros(2 * C, np.int32), P[C:])
    l, _ = plan.eval(2 * C)
    from glass_amd.batch import ucb_alignment
    for e in range(2 * C):
        p = P[C + e]
        BW, _, imin = ucb_alignment(o, T, W, qmin, p)
        h = gl.ucb_waveform(o, "sangria", T, 0.0, p, 8, BW)[:3]
        m = np.zeros((3, W), complex)
        synth.scatter(m, h, imin)
        ref = -np.sum(np.abs(data - m) ** 2) / s ** 2
        assert abs(float(l[e]) / ref - 1) <= 1e-10
    plan.close()


def test_fstatistic(gl, orc):
    from glass_amd.fstat import Fstat
    import torch
    o, q = orbits(gl, orc, 4.0)
    NF = 600
    q0 = int(F * T) - NF // 2
    rng = np.random.default_rng(8)
    X, A, E = (rng.standard_normal(NF) + 1j * rng.standard_normal(NF) for _ in range(3))
    C00 = np.full(NF, 2.0)
    cells = np.stack([(q0 + NF / 2 + rng.uniform(-50, 50, 9)) / T, np.where(np.arange(9) % 3, 0.0, 3e-14),
                      np.arccos(rng.uniform(-1, 1, 9)), rng.uniform(0, 6, 9)], 1)
    f = Fstat(o, "sangria", T, 0.0, q0, X, A, E, C00, max_cells=9)
    lx, la, _ = (v.cpu().numpy() for v in f.eval(torch.tensor(cells, device="cuda")))
    fd = orc.FstatData(T, q0, X, A, E, C00, orbit=q)
    for e in range(9):
        rx, ra, *_ = fd.logl(*cells[e])
        # the filters' phases are products of ~1e6 rad, rounded alike to ~1e-10
        assert abs(lx[e] / rx - 1) <= 1e-9 and abs(la[e] / ra - 1) <= 1e-9, e
    f.close()
