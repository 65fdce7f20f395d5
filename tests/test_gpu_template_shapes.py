"""The Fourier-domain template kernels where their branches change: every
template length from one wave to eight passes of 512 points, frequencies
whose transfer-function arguments leave the polynomials' range (above ~27
mHz), and observation times short enough that the TDI phase is evaluated per
bin.  Waveforms against the oracle; the adjoint gradient against the
forward-mode kernel and against central differences of L."""
import numpy as np
import pytest

from conftest import normwise
from glass_amd import synth

pytestmark = pytest.mark.gpu


def params(seed, f, T, fdot=3e-17):
    p = synth.draw_params(np.random.default_rng(seed), 1, T)[0]
    p[0], p[7] = f * T, fdot * T * T
    return p


@pytest.mark.parametrize("fmt", ["sangria", "phase", "frequency"])
@pytest.mark.parametrize("BW", [16, 32, 64, 128, 256, 512, 1024, 2048, 4096])
@pytest.mark.parametrize("f,years", [(3.1e-3, 2.0), (40e-3, 1.0), (95e-3, 0.5), (5e-3, 0.02)])
def test_waveform(gl, orc, BW, fmt, f, years):
    T = synth.YEAR_T * years
    p = params(BW, f, T)
    h = gl.ucb_waveform(gl.analytic_orbit(), fmt, T, 0.0, p, 8, BW)
    ref = orc.ucb_waveform(p, T, BW, fmt=fmt)
    # the oracle steps exp(i f/f*) from bin to bin, as the reference does: up
    # to N 2^-53 after N bins, relative to the channel's sin(f/f*) (twice
    # that for the difference of two rotations in phase and frequency)
    assert normwise(h, ref) <= 1e-13 + 2 * BW * 2.0 ** -53 / abs(np.sin(f / synth.FSTAR))


@pytest.mark.parametrize("fddot", [0.0, 1e-25])
def test_nine_parameters(gl, orc, fddot):
    """f-double-dot: the sample's ninth-parameter terms."""
    T = synth.T_4YR
    p = np.append(params(7, 12e-3, T, fdot=2e-15), fddot * T ** 3)
    o = gl.analytic_orbit()
    h9 = gl.ucb_waveform(o, "sangria", T, 0.0, p, 9, 512)
    h8 = gl.ucb_waveform(o, "sangria", T, 0.0, p[:8], 8, 512)
    if fddot == 0.0:
        assert np.array_equal(h9, h8)
    else:
        assert normwise(h9, h8) > 1e-6


@pytest.mark.parametrize("narrow", [False, True])
@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("BW", [32, 64, 128, 256, 512, 1024])
def test_adjoint_and_forward_mode(gl, BW, mode, narrow):
    import torch
    from glass_amd.derivs import source_derivs, source_grad
    # narrow: a window of fewer bins than the template, which mode 1's weights
    # by template bin leave too
    T, n, W = synth.T_2YR, 5, BW // 2 + 3 if narrow else BW + BW // 2 + 1
    rng = np.random.default_rng(BW)
    P = np.stack([params(100 + i, f, T) for i, f in enumerate((2e-3, 9e-3, 21e-3, 45e-3, 80e-3))])
    # the last template leaves the window at both of its ends in turn
    imin = [-BW // 4, 2 - BW // 2, 0, 1, -3] if narrow else [W // 4, 3, 0, -BW // 4, W - BW // 2]
    imin = torch.tensor(imin, dtype=torch.int32, device="cuda")
    A = rng.standard_normal((n, W, 3, 3))
    C = np.einsum("nwij,nwkj->nwik", A, A) + 3 * np.eye(3)
    ic = np.linalg.inv(C)
    invC = torch.tensor(np.stack([ic[..., a, b] for a, b in ((0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2))], 1),
                        device="cuda")
    amp = 1e-21
    R = torch.tensor((rng.standard_normal((n, 3, W)) + 1j * rng.standard_normal((n, 3, W))) * amp, device="cuda")
    p = torch.tensor(P, device="cuda")
    o = gl.analytic_orbit()
    L, g, F = source_derivs(o, T, p, BW, imin, invC, R, mode=mode)
    La, ga = source_grad(o, T, p, BW, imin, invC, R, mode=mode)
    L0, none = source_grad(o, T, p, BW, imin, invC, R, mode=mode, want_grad=False)
    assert none is None and torch.equal(F, F.transpose(1, 2))
    scale = g.abs().amax(1, keepdim=True)
    # one likelihood, three kernels, the same bins and weights in both modes:
    # sums in other orders of ~BW terms
    assert torch.allclose(La, L, rtol=1e-11, atol=0) and torch.allclose(L0, L, rtol=1e-11, atol=0)
    assert float(((ga - g).abs() / scale).max()) <= 1e-10
    # central differences of L, step h: truncation h^2, rounding 1e-10/h
    for k, h in ((3, 1e-4), (5, 1e-4), (6, 1e-4), (0, 3e-5), (2, 1e-5)):
        up, dn = p.clone(), p.clone()
        up[:, k] += h
        dn[:, k] -= h
        d = (source_derivs(o, T, up, BW, imin, invC, R, mode=mode)[0] -
             source_derivs(o, T, dn, BW, imin, invC, R, mode=mode)[0]) / (2 * h)
        assert float(((d - g[:, k]).abs() / scale[:, 0]).max()) <= 2e-5, k


def test_retired_tiles_run_as_the_default(gl, orc):
    from test_gpu_batch import make_cfg, new_plan
    cfg = make_cfg(orc, seed=5, ngroup=4, ntemp=2, nprop=3)
    E = len(cfg["p_chain"])
    plan = new_plan(gl, cfg, E)
    plan.set_proposals(cfg["p_chain"], cfg["p_src"], cfg["p_params"])
    base = plan.tiles()
    l0, s0 = (x.clone() for x in plan.eval(E))
    old = list(base)
    for k, nthr, waves in ((2, 128, 6), (3, 256, 6), (3, 256, 8), (4, 512, 8)):  # copies of the default
        old[k] = (nthr, 1, waves)
        plan.set_tiles(old)
        assert plan.tiles()[k] == (base[k][0], 1, base[k][2])
    old = list(base)
    old[3], old[4], old[5], old[6] = (128, 2, 4), (256, 0, 1), (1024, 1, 1), (512, 4, 1)
    plan.set_tiles(old)
    now = plan.tiles()
    assert [t[1] for t in now[3:7]] == [2, 0, 1, 4] and [(t[0], t[2]) for t in now] == [(t[0], t[2]) for t in base]
    l1, s1 = plan.eval(E)
    assert float(((l1 - l0) / l0).abs().max()) <= 1e-12 and float(((s1 - s0) / s0).abs().max()) <= 1e-12
    plan.close()
