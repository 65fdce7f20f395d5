"""The work that users of this framework have it do, as cases that can be timed.

A case is a dict of plain values; `kind` names the path:

* step      one sampler step of a few chains: eval of one proposal per chain,
            then accept of all of them and the new state (the reference's 12
            chains of one window; latency and launches count)
* sweep     the batched likelihood sweep of a parallel-tempering sampler
            (FdBatch.eval), eager or as a graph, for windows of powers of two
            and of odd lengths
* derivs    the Fisher update of a sampler: exact L, gradient and Fisher
            matrix of four sources a chain of a plan, mixed template lengths
* fisher    source_derivs of many sources of one template length
* grad      ucb_source_logl forward and backward (autograd)
* wavelet   WdmBatch.eval: wavelet-domain templates with their inner products
* transform wdm_transform of a time series on the device
* logl      LoglBatch.eval: full-window likelihoods, resident in HBM
* fstat     F-statistic grid cells of a frequency segment
* plain     the per-call drop-ins on host arrays, one waveform and one
            likelihood, as the reference's callers use them

`exact` restates each path in plain torch in 64 bits: template phases are
formed from their small differences instead of the products of ~1e6 rad that
the reference subtracts, splines are solved with a dense matrix, FFTs are
torch's.
"""
import math

import numpy as np
import torch

import glass_amd as gl
from glass_amd import synth
from glass_amd import wdm as wdmmod
from glass_amd.batch import FdBatch, LoglBatch, ucb_alignment
from glass_amd.derivs import source_derivs, ucb_source_logl
from glass_amd.fstat import Fstat

YEAR = synth.YEAR_T
F64, C128 = torch.float64, torch.complex128
# data windows: the sampler's usual powers of two, odd lengths, short ones
WINDOWS = {"pow2": (512, 1024, 2048, 4096), "odd": (389, 700, 1201, 2050, 3333, 5001), "short": (96, 128, 200, 256)}


# ------------------------------------------------------------- the cases ---

def listed():
    return [
        # the reference's per-call path: ucb_waveform + gaussian_log_likelihood
        dict(name="plain_128", kind="plain", fmt="sangria", years=1, BW=128, W=256),
        # one step of the reference's default sampler: 12 chains, one window
        dict(name="step_12", kind="step", fmt="sangria", years=2, ngroup=1, ntemp=12, windows="pow2", f_lo=3e-3,
             f_hi=8e-3, nprop=1, graph=False),
        # the batched sweep: 256 windows x 16 temperatures x 80 proposals
        dict(name="sweep_327680", kind="sweep", fmt="sangria", years=2, ngroup=256, ntemp=16, windows="pow2",
             f_lo=0.5e-3, f_hi=20e-3, nprop=80, graph=True),
        # odd windows, 4 yr, other TDI format: long templates, eager launches
        dict(name="sweep_odd_4yr", kind="sweep", fmt="phase", years=4, ngroup=37, ntemp=12, windows="odd", f_lo=2e-3,
             f_hi=20e-3, nprop=23, graph=False),
        # Fisher update of a batched sampler's sources
        dict(name="derivs_update", kind="derivs", fmt="sangria", years=2, ngroup=256, ntemp=16, windows="pow2",
             f_lo=0.5e-3, f_hi=20e-3),
        # exact Fisher matrices of a catalogue of sources, Tobs 4 yr
        dict(name="fisher_8192", kind="fisher", fmt="sangria", years=4, n=8192, BW=256),
        # gradient-based sampling through autograd
        dict(name="grad_1501", kind="grad", fmt="sangria", years=2, n=1501, BW=512),
        # wavelet templates: short and long time axes (the reference's
        # default grid has NT 4096)
        dict(name="wavelet_4096", kind="wavelet", n=4096, NT=512),
        dict(name="wavelet_nt4096", kind="wavelet", n=300, NT=4096),
        # full WDM transform of a year at 15 s
        dict(name="transform_2m", kind="transform", NF=4096, NT=512),
        # full-window likelihoods of 4096 chains
        dict(name="logl_4096", kind="logl", n=4096, windows="pow2"),
        # F-statistic proposal grid: 256 frequencies x 20 x 20 sky cells
        dict(name="fstat_102400", kind="fstat", years=2, nf=256, nsky=20, fq=3e-3, NFFT=1024),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["plain", "step", "sweep", "sweep", "sweep", "derivs", "fisher", "grad", "wavelet", "wavelet",
                       "transform", "logl", "fstat"])
    fmt = rng.choice(["sangria", "sangria", "phase", "frequency"])
    years = rng.choice([1, 2, 4])
    if kind == "plain":
        BW = 2 ** rng.randint(5, 11)
        return dict(kind=kind, fmt=fmt, years=years, BW=BW, W=rng.randint(BW, 2 * BW + 77))
    if kind in ("step", "sweep", "derivs"):
        windows = rng.choice(["pow2", "odd", "short"])
        f_hi = 6e-3 if windows == "short" else rng.uniform(8e-3, 20e-3)
        c = dict(kind=kind, fmt=fmt, years=1 if windows == "short" else years, windows=windows,
                 f_lo=rng.uniform(0.5e-3, 4e-3), f_hi=f_hi, ntemp=rng.randint(3, 16))
        if kind == "step":
            return dict(c, ngroup=_log_int(rng, 1, 16), nprop=1, graph=False)
        c["ngroup"] = _log_int(rng, 2, 128)
        if kind == "sweep":
            c.update(nprop=_log_int(rng, 1, 60), graph=rng.random() < 0.5)
        return c
    if kind == "fisher":
        BW = 2 ** rng.randint(5, 12)
        return dict(kind=kind, fmt=fmt, years=years, BW=BW, n=_log_int(rng, 1, max(32, (1 << 20) // BW)))
    if kind == "grad":
        BW = 2 ** rng.randint(5, 10)
        return dict(kind=kind, fmt=fmt, years=years, BW=BW, n=_log_int(rng, 1, (1 << 20) // BW))
    if kind == "wavelet":
        NT = rng.choice([256, 512, 1024, 2048, 4096])
        return dict(kind=kind, NT=NT, n=_log_int(rng, 1, (1 << 20) // NT))
    if kind == "transform":
        return dict(kind=kind, NF=2 ** rng.randint(6, 12), NT=2 ** rng.randint(5, 9))
    if kind == "logl":
        return dict(kind=kind, n=_log_int(rng, 1, 3000), windows=rng.choice(sorted(WINDOWS)))
    return dict(kind="fstat", years=years, nf=_log_int(rng, 1, 200), nsky=rng.randint(4, 20),
                fq=rng.uniform(1e-3, 1e-2), NFFT=rng.choice([512, 1024, 1531, 2048]))


# ---------------------------------------------------------------- inputs ---

def _chains(case, seed):
    """Windows, chains, sources and proposals of a step, sweep or derivs case
    (host arrays)."""
    o = gl.analytic_orbit()
    cfg = synth.config1(seed=seed, ngroup=case["ngroup"], ntemp=case["ntemp"], nprop_per_chain=case.get("nprop", 1),
                        T=YEAR * case["years"], f_lo=case["f_lo"], f_hi=case["f_hi"],
                        windows=WINDOWS[case["windows"]],
                        waveform=lambda p, T, BW: gl.ucb_waveform(o, case["fmt"], T, 0.0, p, 8, BW),
                        alignment=lambda p, T, W, q: ucb_alignment(o, T, W, q, p))
    cfg["invC"] = [gl.invert_noise_covariance_matrix(C)[0] for C in cfg["C"]]
    if case["kind"] == "derivs":  # the sky derivatives have no value at the poles
        cfg["src_params"][..., 1] = np.clip(cfg["src_params"][..., 1], -0.9999, 0.9999)
    return cfg


def _plan(case, cfg):
    plan = FdBatch(gl.analytic_orbit(), case["fmt"], cfg["T"], 0.0, cfg["group_qmin"], cfg["data"], cfg["invC"],
                   cfg["chain_group"], cfg["chain_nsrc"], cfg["src_params"], max_prop=len(cfg["p_chain"]))
    plan.set_proposals(cfg["p_chain"], cfg["p_src"], cfg["p_params"])
    return plan


def _live_sources(cfg):
    live = np.arange(8)[None, :] < cfg["chain_nsrc"][:, None]
    c, s = np.nonzero(live)
    return c.astype(np.int32), s.astype(np.int32)


def _fisher_items(cfg):
    """Four (chain, source) items a chain, cycling over its sources."""
    c = np.repeat(np.arange(len(cfg["chain_nsrc"])), 4)
    s = np.tile(np.arange(4), len(cfg["chain_nsrc"])) % cfg["chain_nsrc"][c]
    return c.astype(np.int32), s.astype(np.int32)


def _sources(case, seed):
    """Sources of one template length, each with its own window of 2 BW bins
    of noise (host arrays): params, imin, invC [n, 6, W], resid [n, 3, W]."""
    T, n, BW = YEAR * case["years"], case["n"], case["BW"]
    W = 2 * BW
    rng = np.random.default_rng(seed)
    P = synth.draw_params(rng, n, T)
    q = P[:, 0].astype(np.int64)
    qmin = q - W // 2
    imin = ((q - BW // 2) - qmin).astype(np.int32)
    f = qmin[:, None] / T + np.arange(W)[None, :] / T
    Spm, Sop = synth.noise_levels_sangria(f)
    x = f / synth.FSTAR
    tr = np.sin(x) ** 2
    d = 16.0 * tr * (2.0 * (1.0 + np.cos(x) ** 2) * Spm + Sop) / 4.0
    b = -8.0 * tr * np.cos(x) * (4.0 * Spm + Sop) / 4.0
    den = (d - b) * (d + 2 * b)
    idg, iof = (d + b) / den, -b / den
    invC = np.stack([idg, idg, idg, iof, iof, iof], axis=1)
    R = (rng.standard_normal((n, 3, W)) + 1j * rng.standard_normal((n, 3, W))) * np.sqrt((d - b) / 2)[:, None, :]
    return dict(T=T, W=W, params=P, imin=imin, invC=invC, resid=R)


def _wavelet_inputs(case, seed):
    NT = case["NT"]
    return synth.config2(seed=seed, n=case["n"], NF=(1 << 20) // NT, NT=NT, T=YEAR)


def _segment(case, seed):
    """A frequency segment with three binaries in noise, and grid cells."""
    o = gl.analytic_orbit()
    T, NFFT = YEAR * case["years"], case["NFFT"]
    rng = np.random.default_rng(seed)
    qmin0 = int(case["fq"] * T)
    C00 = synth.xyz_noise_cov(T, qmin0 / T, NFFT)[0, 0].copy()
    ch = [np.sqrt(C00 / 2) * (rng.standard_normal(NFFT) + 1j * rng.standard_normal(NFFT)) for _ in range(3)]
    for _ in range(3):
        p = synth.draw_params(rng, 1, T, log10A=(-22.0, -21.5))[0]
        p[0] = qmin0 + rng.uniform(80, NFFT - 80)
        h = gl.ucb_waveform(o, "sangria", T, 0.0, p, 8, 64, NI=2)
        at = int(p[0]) - 32 - qmin0
        for c, k in enumerate((0, 3, 4)):
            ch[c][at:at + 64] += h[k]
    nf, ns = case["nf"], case["nsky"]
    fi = np.sort(rng.uniform(qmin0 + 40, qmin0 + NFFT - 40, nf)) / T
    ct = -1.0 + (np.arange(ns) + 0.5) * 2.0 / ns
    ph = (np.arange(ns) + 0.5) * 2 * np.pi / ns
    cells = np.zeros((nf, ns, ns, 4))
    cells[..., 0] = fi[:, None, None]
    cells[..., 1] = rng.uniform(-1e-17, 1e-16, nf)[:, None, None] * (rng.random(nf) < 0.3)[:, None, None]
    cells[..., 2] = np.arccos(ct)[None, :, None]
    cells[..., 3] = ph[None, None, :]
    return dict(T=T, qmin0=qmin0, X=ch[0], A=ch[1], E=ch[2], C00=C00, cells=cells.reshape(-1, 4))


def _one_source(case, seed):
    T, BW, W = YEAR * case["years"], case["BW"], case["W"]
    rng = np.random.default_rng(seed)
    p = synth.draw_params(rng, 1, T)[0]
    qmin = int(p[0]) - W // 2
    C = synth.xyz_noise_cov(T, qmin / T, W)
    data = np.zeros((5, W), dtype=np.complex128)
    data[:3] = synth.noise_draw(rng, C)
    d, b = C[0, 0], C[0, 1]
    den = (d - b) * (d + 2 * b)
    invC = np.empty_like(C)
    for i in range(3):
        for j in range(3):
            invC[i, j] = (d + b) / den if i == j else -b / den
    return dict(T=T, params=p, data=data, invC=invC, imin=int(p[0]) - BW // 2 - qmin)


def prepare(case, seed):
    kind, dev = case["kind"], torch.device("cuda")
    if kind == "plain":
        return dict(case, orbit=gl.analytic_orbit(), **_one_source(case, seed))
    if kind in ("step", "sweep"):
        cfg = _chains(case, seed)
        plan = _plan(case, cfg)
        return dict(case, plan=plan, n=len(cfg["p_chain"]), all=np.arange(len(cfg["p_chain"])))
    if kind == "derivs":
        cfg = _chains(case, seed)
        c, s = _fisher_items(cfg)
        return dict(case, plan=_plan(case, cfg), chain=torch.tensor(c, device=dev), src=torch.tensor(s, device=dev))
    if kind in ("fisher", "grad"):
        r = _sources(case, seed)
        t = {k: torch.tensor(r[k], device=dev) for k in ("params", "imin", "invC", "resid")}
        return dict(case, orbit=gl.analytic_orbit(), T=r["T"], **t)
    if kind == "wavelet":
        r = _wavelet_inputs(case, seed)
        w = wdmmod.Wdm.grid(r["NF"], r["NT"], r["dt"])
        orb = wdmmod.interpolated_analytic_orbit(gl.analytic_orbit(), r["T"])
        B = wdmmod.WdmBatch(w, orb, r["T"], r["data"], r["invC6"], max_templates=case["n"])
        return dict(case, batch=B, params=torch.tensor(r["params"], device=dev))
    if kind == "transform":
        ND = case["NF"] * case["NT"]
        g = torch.Generator(device=dev)
        g.manual_seed(int(seed))
        return dict(case, w=wdmmod.Wdm.grid(case["NF"], case["NT"], YEAR / case["NT"]),
                    x=torch.randn(ND, dtype=F64, device=dev, generator=g), out=torch.empty(ND, dtype=F64, device=dev))
    if kind == "logl":
        r = synth.logl_batch_inputs(case["n"], seed=seed, windows=WINDOWS[case["windows"]], device="cuda")
        return dict(case, batch=LoglBatch(r["W"], r["off"], r["off"], r["off"]), data=r["data"], model=r["model"],
                    invC=r["invC"], out=torch.empty(case["n"], dtype=F64, device=dev))
    r = _segment(case, seed)
    n = len(r["cells"])
    F = Fstat(gl.analytic_orbit(), "sangria", r["T"], 0.0, r["qmin0"], r["X"], r["A"], r["E"], r["C00"], max_cells=n)
    return dict(case, fstat=F, cells=torch.tensor(r["cells"], device=dev))


# ------------------------------------------------------------------- run ---

def run(s):
    kind = s["kind"]
    if kind == "plain":
        h = gl.ucb_waveform(s["orbit"], s["fmt"], s["T"], 0.0, s["params"], 8, s["BW"])
        model = np.zeros((5, s["W"]), dtype=np.complex128)
        synth.scatter(model[:3], h[:3], s["imin"])
        return h, gl.gaussian_log_likelihood(s["data"], model, s["invC"])
    if kind == "step":
        out = s["plan"].eval(s["n"])
        s["plan"].accept(s["all"])
        return out + s["plan"].state()
    if kind == "sweep":
        return s["plan"].eval(s["n"], graph=s["graph"])
    if kind == "derivs":
        return s["plan"].derivs(s["chain"], s["src"])
    if kind == "fisher":
        return source_derivs(s["orbit"], s["T"], s["params"], s["BW"], s["imin"], s["invC"], s["resid"],
                             fmt=s["fmt"])
    if kind == "grad":
        p = s["params"].detach().requires_grad_()
        L = ucb_source_logl(p, s["orbit"], s["T"], s["BW"], s["imin"], s["invC"], s["resid"])
        L.sum().backward()
        return L.detach(), p.grad
    if kind == "wavelet":
        return s["batch"].eval(s["params"])
    if kind == "transform":
        return wdmmod.wdm_transform(s["w"], s["x"], s["out"])
    if kind == "logl":
        return s["batch"].eval(s["data"], s["model"], s["invC"], s["out"])
    return s["fstat"].eval(s["cells"])


# --------------------------------------------------------- work, tolerance ---

def _template_flops(N):
    """Slow series, six FFTs and TDI of one template of N bins (a sine and
    cosine counted as 40 operations)."""
    return 940.0 * N + 30.0 * N * math.log2(N)


def _typical_bins(case, n=2000):
    """Template lengths that a chains case's sources have (one fixed draw)."""
    rng = np.random.default_rng(12345)
    T = YEAR * case["years"]
    P = synth.draw_params(rng, n, T, f_lo=case["f_lo"], f_hi=case["f_hi"])
    return 2 * _half_bandwidth(P[:, 0] / T, P[:, 7] / T / T, P[:, 1], np.exp(P[:, 3]), T,
                               rng.choice(np.asarray(WINDOWS[case["windows"]]), n))


def work(case):
    kind = case["kind"]
    if kind == "plain":
        N, W = case["BW"], case["W"]
        return dict(bytes=64.0 + 80.0 * N + 48.0 * W + 72.0 * W + 48.0 * W, flops=_template_flops(N) + 36.0 * W)
    if kind in ("step", "sweep", "derivs"):
        N = _typical_bins(case).astype(float)
        W = float(np.mean(WINDOWS[case["windows"]]))
        nchain = case["ngroup"] * case["ntemp"]
        nsrc = 4.5 * nchain
        f = np.mean([_template_flops(v) for v in N])
        state = 48.0 * W * (nchain + case["ngroup"]) + 48.0 * nsrc * N.mean()
        if kind == "derivs":
            return dict(bytes=state + 4 * nchain * 648.0, flops=4 * nchain * (6 * f + 1620.0 * N.mean()))
        n = nchain * case["nprop"]
        if kind == "step":  # the accept also writes residuals and templates
            return dict(bytes=2 * state + 160.0 * n, flops=n * (2 * f + 36.0 * N.mean()))
        return dict(bytes=state + 88.0 * n, flops=n * (f + 36.0 * N.mean()))
    if kind in ("fisher", "grad"):
        n, N = case["n"], case["BW"]
        f = _template_flops(N)
        if kind == "fisher":
            return dict(bytes=n * (96.0 * N + 64 + 584), flops=n * (6 * f + 1620.0 * N))
        return dict(bytes=n * (96.0 * N + 64 + 72), flops=n * (2 * f + 60.0 * N))
    if kind == "wavelet":
        n, NT, L = case["n"], case["NT"], 2.3
        s = NT * (L + 1)
        fft = 3 * 2.5 * s * math.log2(s) + L * 3 * 5 * NT * math.log2(NT)
        return dict(bytes=n * (64.0 + 16 + 3 * NT * L * 12 + 72 * NT * L),
                    flops=n * (s * 180.0 + fft + 199 * 24 * 140.0 + 36 * NT * L))
    if kind == "transform":
        ND = float(case["NF"] * case["NT"])
        return dict(bytes=16.0 * ND, flops=2.5 * ND * math.log2(ND) + (case["NF"] + 1) * 5.0 * case["NT"] *
                    math.log2(case["NT"]))
    if kind == "logl":
        bins = case["n"] * float(np.mean(WINDOWS[case["windows"]]))
        return dict(bytes=144.0 * bins, flops=36.0 * bins)
    T = YEAR * case["years"]
    n = case["nf"] * case["nsky"] ** 2
    M = float(_half_bandwidth(np.array([case["fq"]]), np.zeros(1), np.zeros(1), np.full(1, 1e-22), T,
                              np.array([case["NFFT"]]))[0])
    return dict(bytes=n * 80.0 + 56.0 * case["NFFT"], flops=n * (4 * _template_flops(M) + 170.0 * M))


def tolerance(case):
    """Largest relative errors between correct FP64 implementations: the
    template phase is a difference of ~1e6-1e7 rad products in the
    reference's formulas, so its rounding (1e-10 to 1e-9 rad) dominates;
    sums and transforms alone agree to ~1e-14."""
    kind = case["kind"]
    if kind in ("transform", "logl"):
        return {"rel": 4e-13, "max": 1e-11}
    if kind == "fstat":
        # acos / atan2 of near-degenerate fits
        return {"rel": 2e-9, "max": 1e-5}
    if kind in ("derivs", "fisher", "grad"):
        return {"rel": 1e-9, "max": 1e-7}
    return {"rel": 4e-9, "max": 4e-7}


# ----------------------------------------------- exact: plain torch, FP64 ---

CLIGHT, AU, SQ3, YSEC, ARM = 299792458.0, 1.49597870700e11, 1.73205080757, 3.15581497632e7, 2.5e9
FSTAR = CLIGHT / (2 * math.pi * ARM)
DEV = "cuda" if torch.cuda.is_available() else "cpu"


def _t(a, dtype=F64):
    return torch.as_tensor(a, dtype=dtype, device=DEV)


def _half_bandwidth(f, fdot, costh, A, T, W):
    """Template half length: a power of two above the Doppler, chirp and SNR
    spreads, 16 to the largest power of two in W/2 (numpy)."""
    Nmax = 2 ** np.floor(np.log2(W // 2)).astype(int)
    fs = f / FSTAR
    red = 1 + 16 * ((2e-5 / f) ** 10 + (1e-4 / f) ** 2)
    sps, sacc, sloc = 8.321e-23, 9e-30, 2.89e-24
    sn = (16.0 / 3) * np.sin(fs) ** 2 * ((2 + np.cos(fs)) * (sps + sloc) + 2 * (3 + 2 * np.cos(fs) + np.cos(2 * fs)) *
                                         (sloc / 2 + sacc / (2 * np.pi * f) ** 4 * red)) / (2 * ARM) ** 2
    dop = 2 * T * ((4 + 2 * np.pi * f * (AU / CLIGHT) * np.sin(np.arccos(costh))) / YSEC + np.abs(fdot) * T)
    snr = A * np.sqrt(T) * np.sin(fs) / np.sqrt(sn)

    def pow2(x):
        return np.clip(np.where(x >= 8, 2.0 ** (np.floor(np.log2(np.maximum(x, 8))) + 1), 16), 16, Nmax).astype(int)

    return np.maximum(pow2(dop - 1), pow2(snr - 1))


def _align(P, T, W, qmin):
    """(template bins, first bin in the window) per source (numpy)."""
    f = P[:, 0] / T
    BW = 2 * _half_bandwidth(f, P[:, 7] / T / T, P[:, 1], np.exp(P[:, 3]), T, W)
    return BW, (f * T).astype(np.int64) - BW // 2 - qmin


def _orbit(t):
    """Analytic spacecraft positions [..., spacecraft, xyz] in metres."""
    a = 2 * math.pi * t[..., None] / YSEC
    sa, ca = torch.sin(a), torch.cos(a)
    beta = 2 * math.pi / 3 * torch.arange(3, device=t.device, dtype=F64)
    sb, cb = torch.sin(beta), torch.cos(beta)
    R = ARM / (2 * SQ3)
    return torch.stack([AU * ca + R * (sa * ca * sb - (1 + sa * sa) * cb),
                        AU * sa + R * (sa * ca * cb - (1 + ca * ca) * sb), -SQ3 * R * (ca * cb + sa * sb)], dim=-1)


def _sky(ct, ph):
    """Propagation vector and polarisation tensors for (cos theta, phi)."""
    st, cp, sp, z = torch.sqrt(1 - ct * ct), torch.cos(ph), torch.sin(ph), torch.zeros_like(ph)
    u = torch.stack([ct * cp, ct * sp, -st], -1)
    v = torch.stack([sp, -cp, z], -1)
    k = torch.stack([-st * cp, -st * sp, -ct], -1)
    uu, vv, uv = u[..., :, None] * u[..., None, :], v[..., :, None] * v[..., None, :], u[..., :, None] * v[..., None, :]
    return k, vv - uu, uv + uv.transpose(-1, -2)


# links (from, to) and, per channel, the links whose differences enter TDI
_LINKS = [(0, 1), (1, 0), (2, 0), (0, 2), (1, 2), (2, 1)]  # 12 21 31 13 23 32
_TDI = [(0, 3, 1, 2), (4, 1, 5, 0), (2, 5, 3, 4)]


def _waveform(p, q, T, N, fmt="sangria", t0=0.0):
    """X, Y, Z [n, 3, N] of n sources p [n, 8] with carrier bins q [n]."""
    f0 = p[:, 0] / T
    fdot = p[:, 7] / (T * T)
    amp, ci, psi = torch.exp(p[:, 3]), p[:, 4], p[:, 5]
    Ap, Ac = amp * (1 + ci * ci) / 2, -amp * ci
    c2, s2 = torch.cos(2 * psi), torch.sin(2 * psi)
    DP, DC = torch.complex(Ap * c2, -Ac * s2), torch.complex(-Ap * s2, -Ac * c2)
    k, ep, ec = _sky(p[:, 1], p[:, 2])
    n = torch.arange(N, device=p.device, dtype=F64)
    t = t0 + T * n / N
    x = _orbit(t)  # [N, 3, 3]
    links = []
    for i, j in _LINKS:
        r = (x[:, j] - x[:, i]) / ARM
        kr = k @ r.T
        dp = torch.einsum("na,eab,nb->en", r, ep, r)
        dc = torch.einsum("na,eab,nb->en", r, ec, r)
        delay = (k @ x[:, i].T) / CLIGHT
        xi = t - delay
        arg = 0.5 * (f0[:, None] + fdot[:, None] * xi) / FSTAR * (1 + kr)
        phase = (2 * math.pi * ((p[:, 0] - q)[:, None] * (t / T) - f0[:, None] * delay) - p[:, 6:7] +
                 math.pi * fdot[:, None] * xi * xi)
        a = 0.25 * torch.sinc(arg / math.pi) * (1 + (2.0 / 3) * (fdot / f0)[:, None] * xi)
        u = phase - arg
        links.append((a * (dp * DP[:, None] + dc * DC[:, None])) * torch.complex(torch.cos(u), torch.sin(u)))
    d = torch.fft.fftshift(torch.fft.fft(torch.stack(links, 1), dim=-1), dim=-1) / (2 * N)
    f = (q[:, None] + n[None, :] - N // 2) / T
    x1 = f / FSTAR
    e1 = torch.complex(torch.cos(x1), -torch.sin(x1))
    out = []
    for a0, a1, b0, b1 in _TDI:
        a, b = d[:, a0] - d[:, a1], d[:, b0] - d[:, b1]
        if fmt == "sangria":
            out.append(4 * math.sqrt(T) * x1 * torch.sin(x1) * (a * e1 * e1 + b * e1))
        else:
            pf = math.sqrt(T) * (1.0 if fmt == "phase" else 2 * x1)
            out.append(pf * (a * e1 ** 3 + b * e1 ** 2 - a * e1 - b))
    return torch.stack(out, 1)


def _ae(h, fmt):
    A, E = (h[:, 2] - h[:, 0]) / math.sqrt(2.0), (h[:, 0] - 2 * h[:, 1] + h[:, 2]) / math.sqrt(6.0)
    return (A.conj().resolve_conj(), E.conj().resolve_conj()) if fmt == "phase" else (A, E)


def _ip(u, v, w):
    """2 sum_ab Re(u_a conj v_b) w_ab per item: u, v [n, 3, N], w [n, 6, N]."""
    def re(a, b):
        return (a * b.conj()).real

    d = w[:, 0] * re(u[:, 0], v[:, 0]) + w[:, 1] * re(u[:, 1], v[:, 1]) + w[:, 2] * re(u[:, 2], v[:, 2])
    o = (w[:, 3] * (re(u[:, 0], v[:, 1]) + re(u[:, 1], v[:, 0])) + w[:, 4] *
         (re(u[:, 0], v[:, 2]) + re(u[:, 2], v[:, 0])) + w[:, 5] * (re(u[:, 1], v[:, 2]) + re(u[:, 2], v[:, 1])))
    return 2 * (d + o).sum(-1)


def _window(flat, nrow, off, W, j):
    """Rows of windows at bins j (0 outside): flat holds nrow x W per window
    from nrow * off; off, W [n], j [n, N] -> [n, nrow, N]."""
    ok = (j >= 0) & (j < W[:, None])
    at = nrow * off[:, None, None] + torch.arange(nrow, device=j.device)[None, :, None] * W[:, None, None] + \
        torch.where(ok, j, torch.zeros_like(j))[:, None, :]
    return flat[at] * ok[:, None, :]


def _chunks(idx, N, most=1 << 20):
    step = max(1, most // N)
    for a in range(0, len(idx), step):
        yield idx[a:a + step]


class _Exact:
    """The chains of a case: windows, residuals, source templates."""

    def __init__(self, case, cfg):
        T = self.T = cfg["T"]
        self.fmt = case["fmt"]
        W = cfg["group_W"].astype(np.int64)
        goff = np.concatenate([[0], np.cumsum(W)[:-1]])
        six = [(0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2)]
        self.data = _t(np.concatenate([d.reshape(-1) for d in cfg["data"]]), C128)
        self.invC = _t(np.concatenate([np.stack([C[a, b] for a, b in six]).reshape(-1) for C in cfg["invC"]]))
        cg = cfg["chain_group"]
        self.W, self.qmin = W[cg], cfg["group_qmin"].astype(np.int64)[cg]
        self.goff = goff[cg]
        self.roff = np.concatenate([[0], np.cumsum(self.W)[:-1]])
        sc, ss = _live_sources(cfg)
        self.slot = -np.ones((len(cg), 8), dtype=np.int64)
        self.slot[sc, ss] = np.arange(len(sc))
        self.sc, self.P = sc, cfg["src_params"][sc, ss]
        self.bw, self.imin = _align(self.P, T, self.W[sc], self.qmin[sc])
        self.toff = np.concatenate([[0], np.cumsum(self.bw)[:-1]])
        self.tmpl = torch.empty(3 * int(self.bw.sum()), dtype=C128, device=DEV)
        # residuals: data minus every source
        pieces = [self.data[3 * goff[g]:3 * (goff[g] + W[g])] for g in cg]
        self.resid = torch.cat(pieces)
        for idx, N, h, j in self.each(self.P, self.bw, self.imin):
            at = 3 * _t(self.toff[idx], torch.int64)[:, None] + torch.arange(3 * N, device=DEV)[None, :]
            self.tmpl[at] = h.reshape(len(idx), -1)
            c = sc[idx]
            Wc = _t(self.W[c], torch.int64)
            ok = ((j >= 0) & (j < Wc[:, None]))[:, None, :].expand(-1, 3, -1)
            at = 3 * _t(self.roff[c], torch.int64)[:, None, None] + torch.arange(3, device=DEV)[None, :, None] * \
                Wc[:, None, None] + j[:, None, :]
            r = torch.view_as_real(self.resid)
            for part in range(2):
                r[:, part].index_add_(0, at[ok], -torch.view_as_real(h)[..., part][ok])
        chi2 = []
        for c in range(len(cg)):
            w = int(self.W[c])
            r = self.resid[3 * self.roff[c]:3 * (self.roff[c] + w)].reshape(1, 3, w)
            ic = self.invC[6 * self.goff[c]:6 * (self.goff[c] + w)].reshape(1, 6, w)
            chi2.append(_ip(r, r, ic))
        self.logl = -0.5 * torch.cat(chi2)

    def each(self, P, bw, imin):
        """(item indices, N, templates, window bins) in pieces of one length."""
        for N in np.unique(bw):
            for idx in _chunks(np.nonzero(bw == N)[0], int(N)):
                p = _t(P[idx])
                h = _waveform(p, torch.floor(p[:, 0]), self.T, int(N), self.fmt)
                yield idx, int(N), h, _t(imin[idx], torch.int64)[:, None] + torch.arange(int(N), device=DEV)[None, :]

    def windows(self, c, j):
        """(residual, invC) of chains c at bins j."""
        W = _t(self.W[c], torch.int64)
        return (_window(self.resid, 3, _t(self.roff[c], torch.int64), W, j),
                _window(self.invC, 6, _t(self.goff[c], torch.int64), W, j))

    def old(self, s, j):
        """Stored templates of sources s at window bins j."""
        return _window(self.tmpl, 3, _t(self.toff[s], torch.int64), _t(self.bw[s], torch.int64),
                       j - _t(self.imin[s], torch.int64)[:, None])

    def proposals(self, pc, ps, P):
        s = self.slot[pc, ps]
        rho, hoho = torch.empty(len(self.P), dtype=F64, device=DEV), torch.empty(len(self.P), dtype=F64, device=DEV)
        for N in np.unique(self.bw):
            for idx in _chunks(np.nonzero(self.bw == N)[0], int(N)):
                j = _t(self.imin[idx], torch.int64)[:, None] + torch.arange(int(N), device=DEV)[None, :]
                r, w = self.windows(self.sc[idx], j)
                h = self.old(idx, j)
                rho[_t(idx, torch.int64)], hoho[_t(idx, torch.int64)] = _ip(r, h, w), _ip(h, h, w)
        logl, snr = torch.empty(len(pc), dtype=F64, device=DEV), torch.empty(len(pc), dtype=F64, device=DEV)
        bw, imin = _align(P, self.T, self.W[pc], self.qmin[pc])
        for idx, N, h, j in self.each(P, bw, imin):
            c, so, at = pc[idx], _t(s[idx], torch.int64), _t(idx, torch.int64)
            r, w = self.windows(c, j)
            ho = self.old(s[idx], j)
            dl = _ip(r, h, w) - rho[so] - 0.5 * (_ip(h, h, w) - 2 * _ip(h, ho, w) + hoho[so])
            logl[at] = self.logl[_t(c, torch.int64)] + dl
            m = torch.arange(N, device=DEV)[None, :].expand(len(idx), -1)
            snr[at] = torch.sqrt(_ip(h, h, self.windows(c, m)[1]))
        return logl, snr


def _derivs(p, q, T, N, fmt, R, w, want_fisher):
    """L, gradient and Fisher matrix of n sources with residuals R [n, 3, N]
    and weights w [n, 6, N] at their template bins, by forward mode."""
    def f(v):
        return torch.view_as_real(_waveform(v, q, T, N, fmt))

    h, dh = None, []
    for k in range(8):
        tang = torch.zeros_like(p)
        tang[:, k] = 1.0
        h, d = torch.func.jvp(f, (p,), (tang,))
        dh.append(torch.view_as_complex(d.contiguous()))
    h = torch.view_as_complex(h.contiguous())
    L = _ip(R, h, w) - 0.5 * _ip(h, h, w)
    g = torch.stack([_ip(R - h, d, w) for d in dh], -1)
    if not want_fisher:
        return L, g
    F = torch.empty(len(p), 8, 8, dtype=F64, device=p.device)
    for a in range(8):
        for b in range(a, 8):
            F[:, a, b] = F[:, b, a] = _ip(dh[a], dh[b], w)
    return L, g, F


def _exact_chain_derivs(case, cfg):
    x = _Exact(case, cfg)
    ic, js = _fisher_items(cfg)
    src = x.slot[ic, js]
    n = len(src)
    L, g, F = (torch.empty(s, dtype=F64, device=DEV) for s in ((n,), (n, 8), (n, 8, 8)))
    for N in np.unique(x.bw[src]):
        for idx in _chunks(np.nonzero(x.bw[src] == N)[0], int(N), 1 << 19):
            so = src[idx]
            p = _t(x.P[so])
            j = _t(x.imin[so], torch.int64)[:, None] + torch.arange(int(N), device=DEV)[None, :]
            r, w = x.windows(x.sc[so], j)
            h = x.old(so, j)
            at = _t(idx, torch.int64)
            L[at], g[at], F[at] = _derivs(p, torch.floor(p[:, 0]), x.T, int(N), x.fmt, r + h, w, True)
    return L, g, F


def _exact_sources(case, seed):
    r = _sources(case, seed)
    n, N = case["n"], case["BW"]
    fmt = case["fmt"] if case["kind"] == "fisher" else "sangria"
    out = []
    for idx in _chunks(np.arange(n), N, 1 << 19):
        p = _t(r["params"][idx])
        sl = slice(int(r["imin"][0]), int(r["imin"][0]) + N)  # the same place in every window
        out.append(_derivs(p, torch.floor(p[:, 0]), r["T"], N, fmt, _t(r["resid"][idx][..., sl], C128),
                           _t(r["invC"][idx][..., sl]), case["kind"] == "fisher"))
    return tuple(torch.cat(v) for v in zip(*out))


def _meyer(Nf, Nt):
    """Half of the WDM window over Nt/2 + 1 bins, forward normalisation."""
    x = np.arange(Nt // 2 + 1) * 2.0 / Nt
    # regularised incomplete beta I_x(6, 6)
    y = sum(math.comb(11, i) * x ** i * (1 - x) ** (11 - i) for i in range(6, 12))
    dom = math.pi / Nf
    phi = np.where(x < 1, np.cos(y * math.pi / 2), 0.0) / math.sqrt(dom)
    norm = (phi[0] ** 2 + 2 * np.sum(phi[1:] ** 2)) * (2 * dom / Nt) / math.pi
    return phi / (math.sqrt(norm) * Nf / 2.0)


def _layers(spec, win, m, centre, edge):
    """Pixels [..., NT] of layer m from one-sided spectra [..., K] around bin
    `centre`."""
    NT = 2 * (len(win) - 1)
    j = torch.arange(-NT // 2 + 1, NT // 2, device=spec.device)
    idx = centre + j
    ok = (idx >= 0) & (idx < spec.shape[-1])
    if edge == 1:
        ok &= idx <= centre
    wt = win[j.abs()] * ok
    if edge is not None:
        wt = torch.where(j == 0, wt / 2, wt)
    DX = torch.zeros(spec.shape[:-1] + (NT,), dtype=C128, device=spec.device)
    DX[..., 1:] = wt * spec[..., idx.clamp(0, spec.shape[-1] - 1)]
    y = torch.fft.ifft(DX, dim=-1)
    if edge is not None:
        return y.real * math.sqrt(2.0)
    n = torch.arange(NT, device=spec.device)
    return torch.where((n + m) % 2 == 0, y.real, (1 if m % 2 == 0 else -1) * y.imag)


def _exact_transform(case, seed):
    s = prepare(case, seed)
    NF, NT = case["NF"], case["NT"]
    spec = torch.fft.rfft(s["x"])
    win = _t(_meyer(NF, NT))
    out = torch.empty(NF + 1, NT, dtype=F64, device=DEV)
    for m in range(NF):
        out[m] = _layers(spec, win, m, m * NT // 2, 0 if m == 0 else None)
    last = _layers(spec, win, NF, NF * NT // 2, 1)
    out[0, 1::2] = last[0::2]
    return out[:NF].reshape(-1)


def _spline(x, y):
    """Natural cubic spline through y [..., K] at x [K]: [..., 4, K]."""
    K = len(x)
    dx = x[1:] - x[:-1]
    A = torch.zeros(K, K, dtype=F64, device=x.device)
    i = torch.arange(1, K - 1, device=x.device)
    A[0, 0] = A[-1, -1] = 1.0
    A[i, i - 1], A[i, i], A[i, i + 1] = dx[:-1], 2 * (dx[1:] + dx[:-1]), dx[1:]
    s = (y[..., 1:] - y[..., :-1]) / dx
    rhs = torch.zeros_like(y)
    rhs[..., 1:-1] = 3 * (s[..., 1:] - s[..., :-1])
    c2 = torch.linalg.solve(A, rhs.reshape(-1, K).T).T.reshape(y.shape)
    c1, c3 = torch.zeros_like(y), torch.zeros_like(y)
    c1[..., :-1] = s - dx * (c2[..., 1:] + 2 * c2[..., :-1]) / 3
    c3[..., :-1] = (c2[..., 1:] - c2[..., :-1]) / (3 * dx)
    return torch.stack([y, c1, c2, c3], -2)


def _at(x, c, t):
    """Splines c [..., 4, K] at times t [..., M] (leading dims alike)."""
    n = (torch.searchsorted(x, t.contiguous(), right=True) - 1).clamp(0, len(x) - 2)
    d = t - x[n]
    g = [torch.gather(c[..., k, :].expand(n.shape[:-1] + (len(x),)), -1, n) for k in range(4)]
    return g[0] + d * (g[1] + d * (g[2] + d * g[3]))


# delayed one-arm terms of a Michelson channel with vertices a, b, c: vertex,
# arm delays (on a, b, c), and two (sign, plus arm?, arm) antenna terms
_DELAYS = [(0, (0, 2, 2), (1, 0, 1), (-1, 1, 2)), (1, (0, 2, 1), (-1, 0, 2), (1, 1, 2)),
           (2, (0, 1, 2), (1, 1, 1), (-1, 0, 1)), (0, (0, 2, 0), (-1, 0, 1), (1, 0, 2)),
           (0, (0, 0, 2), (1, 1, 2), (-1, 1, 1)), (2, (0, 1, 0), (-1, 1, 1), (1, 0, 1)),
           (1, (0, 0, 1), (1, 0, 2), (-1, 1, 2)), (0, (0, 0, 0), (-1, 0, 2), (1, 1, 1))]


def _amp_phase(M, Mf, ref):
    """Signed amplitude and phase of a response [n, K] against `ref`: the
    amplitude changes sign where it touches zero between samples."""
    K = M.shape[-1]
    A = torch.sqrt(M * M + Mf * Mf)
    flip, jump = torch.ones_like(A), torch.zeros_like(A)
    skip = torch.zeros(A.shape[:-1], dtype=torch.bool, device=A.device)
    i0, i1, i2 = A[:, :-2], A[:, 1:-1], A[:, 2:]
    low = (i1 < i0) & (i1 < i2)
    d1, up, dn = i2 + i0 - 2 * i1, (-i2 + i0 - 2 * i1), (-i2 + i0 + 2 * i1)
    up, dn = low & ((up / d1).abs() < 0.1), low & ((dn / d1).abs() < 0.1)
    for i in range(1, K - 1):
        go = ~skip
        u, d = up[:, i - 1] & go, dn[:, i - 1] & go
        flip[:, i] = torch.where(skip, flip[:, i], flip[:, i - 1])
        jump[:, i] = torch.where(skip, jump[:, i], jump[:, i - 1])
        here = d & ~u
        flip[:, i], jump[:, i] = torch.where(here, -flip[:, i], flip[:, i]), jump[:, i] + math.pi * here
        flip[:, i + 1] = torch.where(u, -flip[:, i], flip[:, i + 1])
        jump[:, i + 1] = torch.where(u, jump[:, i] + math.pi, jump[:, i + 1])
        skip = u
    flip[:, -1], jump[:, -1] = flip[:, -2], jump[:, -2]
    ph = -torch.atan2(Mf, M) + jump - (ref - 2 * math.pi * torch.round(ref / (2 * math.pi)))
    for i in range(1, K):
        d = ph[:, i] - ph[:, i - 1]
        ph[:, i] -= 2 * math.pi * torch.round(d.abs() / (2 * math.pi)) * torch.sign(d)
    return flip * A, ph


def _exact_wavelets(case, seed):
    cfg = _wavelet_inputs(case, seed)
    T, NT, NF, dt = cfg["T"], cfg["NT"], cfg["NF"], cfg["dt"]
    df, kmin, npix = 1 / (2 * dt), cfg["kmin"], cfg["kmax"] - cfg["kmin"]
    K = max(20, int(200 * T / YSEC))
    buf = T / (K - 1)
    knots = -buf + torch.arange(K, dtype=F64, device=DEV) * ((T + 2 * buf) / (K - 1))
    orb = _spline(knots, _orbit(knots).permute(1, 2, 0) / CLIGHT)  # [3, 3, 4, K]
    ts = torch.arange(K, dtype=F64, device=DEV) * (T / (K - 1))
    data, invC = _t(cfg["data"]), _t(cfg["invC6"])
    x = _at(knots, orb, ts.expand(3, 3, K)).permute(2, 0, 1)  # [K, craft, xyz]
    arm = torch.stack([x[:, 1] - x[:, 2], x[:, 2] - x[:, 0], x[:, 0] - x[:, 1]], 1)
    Lk = arm.norm(dim=-1)
    arm = arm / Lk[..., None]
    P = cfg["params"]
    f0, f1 = P[:, 0] / T, P[:, 0] / T + P[:, 7] / T / T
    lo, hi = np.minimum(f0, f1) * (1 - 0.00010103671), np.maximum(f0, f1) * (1 + 0.00010103671)
    j0 = np.rint(lo / df)
    jmin = (j0 - (lo - j0 * df < 0)).astype(int)
    nl = (j0 + (hi - j0 * df > 0)).astype(int) - jmin + 1
    dlogl, snr = torch.empty(len(P), dtype=F64, device=DEV), torch.empty(len(P), dtype=F64, device=DEV)
    for nlay in np.unique(nl):
        win = _t(_meyer(int(nlay) + 1, NT))
        nds = NT * (int(nlay) + 1)
        tds = torch.arange(nds, dtype=F64, device=DEV) * (dt / (int(nlay) + 1))
        x0 = _at(knots, orb[0], tds.expand(3, nds))
        for idx in _chunks(np.nonzero(nl == nlay)[0], nds, 1 << 19):
            p, n = _t(P[idx]), len(idx)
            k, ep, ec = _sky(p[:, 1], p[:, 2])
            F0, FD = p[:, 0:1] / T, p[:, 7:8] / T / T
            # barycentre phase and amplitude on the knots, then their splines
            phs = _spline(knots, 2 * math.pi * (F0 * knots + 0.5 * FD * knots * knots) - p[:, 6:7])
            ams = _spline(knots, torch.exp(p[:, 3:4]) * (1 + 2.0 / 3 * FD / F0 * knots))
            ref = _at(knots, phs, ts - (k @ x[:, 0].T))
            kr = torch.einsum("ea,nia->eni", k, x)
            kn = torch.einsum("ea,nia->eni", k, arm)
            dp = torch.einsum("nia,eab,nib->eni", arm, ep, arm)
            dc = torch.einsum("nia,eab,nib->eni", arm, ec, arm)
            F = {(1, 0): dp / (1 + kn), (0, 0): dp / (1 - kn), (1, 1): dc / (1 + kn), (0, 1): dc / (1 - kn)}
            c2, s2 = torch.cos(2 * p[:, 5:6]), torch.sin(2 * p[:, 5:6])
            Ap, Ac = 0.5 * (1 + p[:, 4:5] ** 2), -p[:, 4:5]
            series = []
            for ch in range(3):
                vt = [ch, (ch + 1) % 3, (ch + 2) % 3]
                M, Mf = torch.zeros(n, K, dtype=F64, device=DEV), torch.zeros(n, K, dtype=F64, device=DEV)
                for v, delay, *terms in _DELAYS:
                    te = ts - kr[:, :, vt[v]] - sum(m * Lk[:, vt[i]] for i, m in enumerate(delay))
                    a, ph = _at(knots, ams, te), _at(knots, phs, te)
                    cp, sp = torch.cos(ph), torch.sin(ph)
                    hp, hc = a * (Ap * c2 * cp + Ac * s2 * sp), a * (Ac * c2 * sp - Ap * s2 * cp)
                    hpf, hcf = a * (-Ap * c2 * sp + Ac * s2 * cp), a * (Ac * c2 * cp + Ap * s2 * sp)
                    for sign, plus, i in terms:
                        M += sign * (hp * F[plus, 0][:, :, vt[i]] + hc * F[plus, 1][:, :, vt[i]])
                        Mf += sign * (hpf * F[plus, 0][:, :, vt[i]] + hcf * F[plus, 1][:, :, vt[i]])
                A, ph = _amp_phase(M, Mf, ref)
                tt = tds.expand(n, nds)
                het = _at(knots, phs, tds - k @ x0) - 2 * math.pi * ((_t(jmin[idx]) - 1) * df)[:, None] * tds
                series.append(_at(ts, _spline(ts, A), tt) * torch.cos(_at(ts, _spline(ts, ph), tt) + het))
            spec = torch.fft.rfft(torch.stack(series, 1), dim=-1)
            hh, dh, dd = (torch.zeros(n, dtype=F64, device=DEV) for _ in range(3))
            norm = math.sqrt(NF) / (nlay + 1.0)
            i = torch.arange(NT, device=DEV)
            edge = (i < 100) | (i > NT - 100)
            jm = _t(jmin[idx], torch.int64)
            for off in range(int(nlay)):
                # the pixel parity follows the layer's own number
                even = _layers(spec, win, 0, (off + 1) * NT // 2, None)
                odd = _layers(spec, win, 1, (off + 1) * NT // 2, None)
                par = ((jm + off) % 2 == 0)[:, None, None]
                h = torch.where(par, even, odd) * norm
                at = i[None, :] + (jm + off)[:, None] * NT - kmin
                ok = (at >= 0) & (at < npix)
                w = invC[:, at.clamp(0, npix - 1)].permute(1, 0, 2) * ok[:, None, :]
                d = data[:, at.clamp(0, npix - 1)].permute(1, 0, 2)
                e = edge[None, None, :]
                # _ip counts twice: pixels are real
                hh += 0.5 * _ip(h.to(C128), h.to(C128), w)
                dh += 0.5 * (_ip(d.to(C128), h.to(C128), w * ~e) - 0.5 * _ip(h.to(C128), h.to(C128), w * ~e))
                dd += 0.25 * _ip(d.to(C128), d.to(C128), w * e)
            dlogl[_t(idx, torch.int64)] = dh + dd
            snr[_t(idx, torch.int64)] = torch.sqrt(hh)
    return dlogl, snr


def _exact_fstat(case, seed):
    r = _segment(case, seed)
    T, NFFT, cells = r["T"], len(r["C00"]), r["cells"]
    M = _half_bandwidth(cells[:, 0], cells[:, 1], np.cos(cells[:, 2]), np.full(len(cells), 1e-22), T,
                        np.full(len(cells), NFFT))
    lx, la, fp = (torch.empty(s, dtype=F64, device=DEV) for s in ((len(cells),), (len(cells),), (len(cells), 4)))
    chans = [_t(r[k], C128) for k in "XAE"]
    C00 = _t(r["C00"])
    for N in np.unique(M):
        for idx in _chunks(np.nonzero(M == N)[0], int(N), 1 << 19):
            c = _t(cells[idx])
            n, at = len(idx), _t(idx, torch.int64)
            q = torch.floor(c[:, 0] * T)
            k = (q.long() - r["qmin0"] - int(N) // 2)[:, None] + torch.arange(int(N), device=DEV)[None, :]
            ok = (k > 0) & (k < NFFT)
            k = k.clamp(0, NFFT - 1)
            w = ok / C00[k]
            H = []
            for psi, ph in ((0.0, 0.0), (math.pi / 4, math.pi), (0.0, 1.5 * math.pi), (math.pi / 4, 0.5 * math.pi)):
                one = torch.ones(n, dtype=F64, device=DEV)
                p = torch.stack([c[:, 0] * T, torch.cos(c[:, 2]), c[:, 3], math.log(2.0) * one, 0 * one, psi * one,
                                 ph * one, c[:, 1] * T * T], -1)
                h = _waveform(p, q, T, int(N))
                H.append((h[:, 0],) + _ae(h, "sangria"))
            d = [v[k] for v in chans]

            def ip(a, b):
                return 4 * ((a * b.conj()).real * w).sum(-1)

            for which in ((0,), (1, 2)):
                Nv = torch.stack([sum(ip(d[s], H[a][s]) for s in which) for a in range(4)], -1)
                G = torch.stack([torch.stack([sum(ip(H[a][s], H[b][s]) for s in which) for b in range(4)], -1)
                                 for a in range(4)], -2)
                a = torch.linalg.solve(G, Nv[..., None])[..., 0]
                F = 0.5 * (a * Nv).sum(-1)
                if which == (0,):
                    lx[at] = F
                    continue
                la[at] = F
                s1 = torch.hypot(a[:, 0] + a[:, 3], a[:, 1] - a[:, 2])
                s2 = torch.hypot(a[:, 0] - a[:, 3], a[:, 1] + a[:, 2])
                Ap, Ac = s1 + s2, s1 - s2
                u = Ap * a[:, 3] - Ac * a[:, 0]
                psi = 0.5 * torch.atan2(u, -(Ac * a[:, 1] + Ap * a[:, 2]))
                sg = torch.sign(torch.sin(2 * psi))
                root = torch.sqrt(Ap * Ap - Ac * Ac)
                fp[at] = torch.stack([0.5 * (Ap + root), torch.acos(-Ac / (Ap + root)), psi,
                                      torch.atan2(sg * u, -sg * (Ac * a[:, 2] + Ap * a[:, 1]))], -1)
    return lx, la, fp


def _exact_plain(case, seed):
    r = _one_source(case, seed)
    p = _t(r["params"][None])
    h = _waveform(p, torch.floor(p[:, 0]), r["T"], case["BW"], case["fmt"])
    out = torch.cat([h[0], torch.cat(_ae(h, case["fmt"]))])
    res = r["data"][:3].copy()
    synth.scatter(res, -h[0].cpu().numpy(), r["imin"])
    six = np.stack([r["invC"][a, b] for a, b in ((0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2))])
    d = _t(res[None], C128)
    return out.cpu().numpy(), float(-0.5 * _ip(d, d, _t(six[None]))[0])


def exact(case, seed):
    kind = case["kind"]
    if kind == "plain":
        return _exact_plain(case, seed)
    if kind in ("step", "sweep"):
        cfg = _chains(case, seed)
        logl, snr = _Exact(case, cfg).proposals(cfg["p_chain"], cfg["p_src"], cfg["p_params"])
        if kind == "sweep":
            return logl, snr
        params = cfg["src_params"].copy()
        params[cfg["p_chain"], cfg["p_src"]] = cfg["p_params"]
        return logl, snr, logl.cpu().numpy(), params
    if kind == "derivs":
        return _exact_chain_derivs(case, _chains(case, seed))
    if kind in ("fisher", "grad"):
        return _exact_sources(case, seed)
    if kind == "wavelet":
        return _exact_wavelets(case, seed)
    if kind == "transform":
        return _exact_transform(case, seed)
    if kind == "logl":
        s = prepare(case, seed)
        r = synth.logl_batch_inputs(case["n"], seed=seed, windows=WINDOWS[case["windows"]], device=DEV)
        out, res = [], s["data"] - s["model"]
        for W, off in zip(r["W"].astype(int), r["off"].astype(int)):
            d = res[3 * off:3 * (off + W)].reshape(1, 3, W)
            out.append(-0.5 * _ip(d, d, s["invC"][6 * off:6 * (off + W)].reshape(1, 6, W)))
        return torch.cat(out)
    return _exact_fstat(case, seed)
