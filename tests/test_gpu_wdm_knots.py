"""Wavelet templates over orbits of different knot counts (the splines' chunks,
the flips' words and the staging of the splines change with it) and both short
time axes, against the oracle with correctly rounded sine and cosine: lists
identical, values 1e-12 normwise, inner products 1e-10 relative.

A template may exceed 1e-12 where the two sides round one sine of one delayed
term differently (either's correct rounding fails for ~1e-5 of arguments, and a
knot's sums cancel): the reference's own output moves by up to 4e-11 for that,
so one template of 24 may differ by 1e-10."""
import numpy as np
import pytest

from glass_amd import synth
from test_gpu_wdm import grids, normwise

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("years,NT", [(0.05, 256), (0.32, 512), (0.64, 256), (1.0, 256), (1.61, 512), (2.5, 512),
                                      (2.5, 256)])
def test_knot_counts(orc, gl, years, NT):
    import torch
    from glass_amd import wdm as W
    T, NF = years * 3.15581497632e7, (1 << 20) // NT
    ow, gw = grids(orc, W, NF, NT, T / NT)
    oorb, gorb = orc.iorbit(T), W.interpolated_analytic_orbit(gl.analytic_orbit(), T)
    n = 24
    P = synth.draw_params(np.random.default_rng(int(100 * years) + NT), n, T, f_lo=1.5e-3, f_hi=6e-3)
    df = gw.df
    for i in range(6):  # one and three layers as well as two
        P[i, 0] = int(P[i, 0] / T / df) * df * T
        P[i, 7] = 0.0
    for i in range(6, 10):
        P[i, 0] = (int(P[i, 0] / T / df) + 0.5) * df * T
        P[i, 7] = 0.0
    d, ic9 = synth.wdm_random_noise(ow.NF, ow.NT, ow.kmin, ow.kmax, 3)
    B = W.WdmBatch(gw, gorb, T, d, ic9[[0, 4, 8, 1, 2, 5]], max_templates=n)
    dl, sn = (v.cpu().numpy() for v in B.eval(torch.tensor(P, device="cuda")))
    with orc.cr_trig():
        rdl, rsn, rnw, _ = orc.wdm_eval_batch(ow, oorb, T, P, d, ic9)
    nw, lst, val = B.templates(n)
    assert np.array_equal(nw, rnw)
    worst, layers = [], set()
    for e in range(n):
        with orc.cr_trig():
            olst, ov = orc.ucb_waveform_wavelet(ow, oorb, T, P[e])
        layers.add(len(olst) // NT)
        assert np.array_equal(lst[e, :nw[e]], olst)
        worst.append(normwise(val[e, :, :nw[e]], ov))
    print(len(oorb[0]), "knots", NT, "layers", sorted(layers), "worst", sorted(worst)[-2:])
    assert sorted(worst)[-2] < 1e-12 and max(worst) < 1e-10
    assert np.max(np.abs(dl - rdl) / np.maximum(np.abs(rdl), 1.0)) < 1e-10
    assert np.max(np.abs(sn - rsn) / rsn) < 1e-10
    B.close()
