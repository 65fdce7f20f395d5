// ucb_common.h -- shared device code for the UCB frequency-domain path on
// gfx950 (CDNA4).  FP64 throughout.
//
// The slow-series sample restates ucb/src/glass_ucb_waveform.c:840-937 with
// the LISA response helpers of utils/src/glass_lisa.c:1521-1596.  The phase
// chain t -> k.x -> xi -> arg2 is evaluated with contraction disabled and in
// the reference's operation order, because arg2 is a difference of ~1e6-1e7
// rad products whose rounding (~1e-10 rad) would otherwise move the result
// by far more than the 1e-12 parity budget.  Amplitude-only quantities
// (detector tensors, transfer-function sinc) are free to contract.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "fastmath.h"

namespace glass {

// utils/src/glass_constants.h:31-89, utils/src/glass_lisa.h:31-49
constexpr double kPI2 = 6.283185307179586;
constexpr double kPI = 3.14159265358979323846;
constexpr double kCLIGHT = 299792458.;
constexpr double kInvCLIGHT = 1.0 / kCLIGHT;  // correctly rounded (compile time)
constexpr double kYEAR = 3.15581497632e7;
constexpr double kAU = 1.49597870700e11;
constexpr double kSQ3 = 1.73205080757;
constexpr double kLARM = 2.5e9;
constexpr double kSQRT1_2 = 0.70710678118654752440;
constexpr double kINVSQ6 = 0.408248290463863;  // glass_lisa.c:436

// What the spacecraft positions that a template reads reach.  L and f* come
// from the caller, independent of the positions, so the bounds of the
// transfer functions' arguments are taken from the positions themselves.
struct OrbitReach
{
    double arg;   // largest argument over |f|: (1 + longest arm / L) / (2 f*), at least 1.25 / f*
    double time;  // largest |time| at which a frequency is taken: |t0| + T and the light travel time
                  // of the farthest spacecraft, at least 1000 s
};

// From the longest arm and the largest distance from the barycentre (metres);
// a NaN stays one, and sinc_wide then takes the general path.
inline OrbitReach orbit_reach(double L, double fstar, double T, double t0, double arm, double far)
{
    const double a = 0.5 * (1.0 + arm / fabs(L)), t = far * kInvCLIGHT;
    return {(a <= 1.25 ? 1.25 : a) / fabs(fstar), fabs(t0) + T + (t <= 1000.0 ? 1000.0 : t)};
}

// The analytic orbit: spacecraft 2 |R| from a centre at 1 AU, arms of 2
// sqrt(3) |R| (constant in its first order in the eccentricity).
inline OrbitReach analytic_reach(double L, double fstar, double R, double T, double t0)
{
    return orbit_reach(L, fstar, T, t0, 1.001 * 2.0 * kSQ3 * fabs(R), kAU + 2.002 * fabs(R));
}

// Longest arm and largest distance in a table of n records x1 x2 x3 y1 y2 y3 z1
// z2 z3 (NaN if one is).
inline void positions_extent(const double* pos, int n, double* arm, double* far)
{
    double a = 0.0, r = 0.0;
    for (const double* p = pos; p < pos + 9 * (size_t)n; p += 9)
        for (int i = 0; i < 3; i++)
        {
            const int j = (i + 1) % 3;
            const double dx = p[i] - p[j], dy = p[3 + i] - p[3 + j], dz = p[6 + i] - p[6 + j];
            const double d = sqrt(dx * dx + dy * dy + dz * dz);
            const double s = sqrt(p[i] * p[i] + p[3 + i] * p[3 + i] + p[6 + i] * p[6 + i]);
            if (d > a || d != d) a = d;
            if (s > r || s != s) r = s;
        }
    *arm = a;
    *far = r;
}

// Per-template constants (glass_ucb_waveform.c:804-837).
struct UcbConst
{
    double T, t0;
    double f0, phi0, dfdt, d2fdt2;
    double df;      // PI2*(q/T)
    double pi2f0;   // PI2*f0, first factor of arg2
    double pidfdt;  // M_PI*dfdt
    double pid2;    // (M_PI/3)*d2fdt2
    double aevc;    // 0.666...*dfdt/f0
    double halfd2;  // 0.5*d2fdt2
    double DPr, DPi, DCr, DCi;
    double k[3];
    double ua[3], va[2], ka[3];  // u, v (v_z = 0) and k over the arm length L
    double f0h, dfh, d2h;        // f0, dfdt, d2fdt2/2 over 2 f*
    double aevq;                 // aevc/4
    double invfstar, fstar, invL;
    double sqT, invT;  // sqrt(T), 1/T (TDI prefactor and bin frequency)
    double qd;               // q
    double tdx, ttc, tts;    // f/f* per bin, cos and sin of f/f* at bin q (fd_tdi)
    long q;
    int np;
    int wide;  // transfer-function arguments above 1.75 (sinc_wide)
};

// glass_ucb_waveform.c:804-837 + LISA_polarization_tensor (glass_lisa.c:1566-1596)
__host__ __device__ inline void ucb_setup(const double* p, int np, double T, double t0,
                                          double L, double fstar, OrbitReach reach, UcbConst& c)
{
    // k feeds the phase through k.x: no contraction anywhere in the setup
#pragma clang fp contract(off)
    c.T = T;
    c.t0 = t0;
    c.np = np;
    c.f0 = p[0] / T;
    double costh = p[1], phi = p[2], amp = exp(p[3]), cosi = p[4], psi = p[5];
    c.phi0 = p[6];
    c.dfdt = 0.0;
    c.d2fdt2 = 0.0;
    if (np > 7) c.dfdt = p[7] / (T * T);
    if (np > 8) c.d2fdt2 = p[8] / (T * T * T);
    c.q = (long)(c.f0 * T);
    double cosps = cos(2. * psi), sinps = sin(2. * psi);
    double Aplus = amp * (1. + cosi * cosi) * 0.5;
    double Across = -amp * (cosi);
    c.df = kPI2 * (((double)c.q) / T);
    c.pi2f0 = kPI2 * c.f0;
    c.pidfdt = kPI * c.dfdt;
    c.pid2 = (kPI / 3.0) * c.d2fdt2;
    c.aevc = 0.66666666666666666666 * c.dfdt / c.f0;
    c.halfd2 = 0.5 * c.d2fdt2;
    c.DPr = Aplus * cosps;
    c.DPi = -Across * sinps;
    c.DCr = -Aplus * sinps;
    c.DCi = -Across * cosps;
    double sinth = sqrt(1.0 - costh * costh);
    double cosph = cos(phi), sinph = sin(phi);
    double u0 = costh * cosph, u1 = costh * sinph, u2 = -sinth;
    double v0 = sinph, v1 = -cosph;
    c.k[0] = -sinth * cosph;
    c.k[1] = -sinth * sinph;
    c.k[2] = -costh;
    c.fstar = fstar;
    c.invfstar = 1. / fstar;
    c.invL = 1. / L;
    c.sqT = sqrt(T);
    c.invT = 1. / T;
    c.ua[0] = u0 * c.invL;  c.ua[1] = u1 * c.invL;  c.ua[2] = u2 * c.invL;
    c.va[0] = v0 * c.invL;  c.va[1] = v1 * c.invL;
    for (int i = 0; i < 3; i++) c.ka[i] = c.k[i] * c.invL;
    c.wide = sinc_wide(fabs(c.f0) + (fabs(c.dfdt) + fabs(c.halfd2) * reach.time) * reach.time, reach.arg);
    c.f0h = 0.5 * c.f0 * c.invfstar;
    c.dfh = 0.5 * c.dfdt * c.invfstar;
    c.d2h = 0.5 * c.halfd2 * c.invfstar;
    c.aevq = 0.25 * c.aevc;
    c.qd = (double)c.q;
    c.tdx = c.invT * c.invfstar;
    sincos_red(c.qd * c.invT * c.invfstar, &c.tts, &c.ttc);
}

// One slow-series sample at time t: out(l, value) receives the links 12, 21,
// 31, 13, 32 (l = 0..4, a compile-time constant once inlined) less link 23.
// pos: spacecraft positions x1,x2,x3,y1,y2,y3,z1,z2,z3 at t (metres), KS
// doubles apart (1 in a sample record, N in a structure-of-arrays table).
// glass_ucb_waveform.c:843-936, LISA_detector_tensor glass_lisa.c:1521-1564.
//
// The vector issue rate bounds this code, so the sample is arranged for few
// instructions (about 400; 850 before, which with fd_tdi_phase took 130,042
// fused 512-bin evaluations from 3.12 to 2.65 ms, 74,247 of 256 bins from
// 0.93 to 0.77 ms and 23,671 of 2048 bins from 3.87 to 2.96 ms):
//  * r.E.r of the rank-two polarisation tensors from the projections on u
//    and v: d+ = (r.v)^2 - (r.u)^2, dx = 2 (r.u)(r.v); the arm's d+ DP + dx DC
//    is shared by its two links;
//  * a link is T1 exp(i arg2) [sinc(arg1) exp(-i arg1)]: one full-range sine
//    and cosine per spacecraft instead of one per link, and the bracket, of
//    small argument, from two polynomials without range reduction;
//  * the spacecraft unrolled, no selects, each polynomial coefficient set
//    once for all arguments that use it.
template <int KS = 1, typename Out>
__device__ __forceinline__ void ucb_slow_sample_to(const UcbConst& c, double t, const double* __restrict__ pos,
                                                   Out&& out)
{
    double x[3], y[3], z[3];
#pragma unroll
    for (int i = 0; i < 3; i++)
    {
        x[i] = pos[i * KS];
        y[i] = pos[(3 + i) * KS];
        z[i] = pos[(6 + i) * KS];
    }
    double a2[3], hf[3], ae[3];
    double dft;
    {
#pragma clang fp contract(off)
        dft = c.df * t;
    }
#pragma unroll
    for (int i = 0; i < 3; i++)
    {
        double xi;
        {
#pragma clang fp contract(off)
            // the quotient by c, as IEEE division gives it (div_by_recip)
            const double kdotx = div_by_recip(x[i] * c.k[0] + y[i] * c.k[1] + z[i] * c.k[2], kCLIGHT, kInvCLIGHT);
            xi = t - kdotx;
            a2[i] = c.pi2f0 * xi - c.phi0 - dft;
            a2[i] += c.pidfdt * xi * xi;
            if (c.np > 8) a2[i] += c.pid2 * xi * xi * xi;
        }
        // half the frequency over f*, and a quarter of the amplitude
        hf[i] = fma(c.dfh, xi, c.f0h);
        if (c.np > 8) hf[i] = fma(c.d2h * xi, xi, hf[i]);
        ae[i] = fma(c.aevq, xi, 0.25);
    }
    // arms 12, 13, 23: k.r and T1 = d+ DP + dx DC
    double kr[3], t1r[3], t1i[3];
    const double dcr = 2.0 * c.DCr, dci = 2.0 * c.DCi;
#pragma unroll
    for (int m = 0; m < 3; m++)
    {
        const int i0 = m < 2 ? 0 : 1, i1 = m == 0 ? 1 : 2;
        const double r0 = x[i1] - x[i0], r1 = y[i1] - y[i0], r2 = z[i1] - z[i0];
        const double ru = r0 * c.ua[0] + r1 * c.ua[1] + r2 * c.ua[2];
        const double rv = r0 * c.va[0] + r1 * c.va[1];
        kr[m] = r0 * c.ka[0] + r1 * c.ka[1] + r2 * c.ka[2];
        const double dp = rv * rv - ru * ru, dc = ru * rv;
        t1r[m] = dp * c.DPr + dc * dcr;
        t1i[m] = dp * c.DPi + dc * dci;
    }
    __builtin_amdgcn_sched_barrier(0);
    // exp(i arg2) times the amplitude
    double wr[3], wi[3];
    {
        double sn[3], cs[3];
        unsigned fl[3];
        sincos_half<3>(a2, sn, cs, fl);
#pragma unroll
        for (int i = 0; i < 3; i++)
        {
            const double a = flip_sign(ae[i], fl[i]);
            wr[i] = a * cs[i];
            wi[i] = a * sn[i];
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    double2 d23;
#pragma unroll
    for (int q = 0; q < 3; q++)
    {
        const int i = q == 0 ? 1 : (q == 1 ? 0 : 2);  // spacecraft 2 first: link 23
        // links (i, j) of spacecraft i: k.r_ij antisymmetric, T1 symmetric
        const double ka = i == 0 ? kr[0] : (i == 1 ? -kr[0] : -kr[1]), kb = i == 0 ? kr[1] : (i == 1 ? kr[2] : -kr[2]);
        const double arg[2] = {fma(hf[i], ka, hf[i]), fma(hf[i], kb, hf[i])};
        double fr[2], fi[2];
        sinc_phase<2>(arg, c.wide, fr, fi);
        double2 d[2];
#pragma unroll
        for (int h = 0; h < 2; h++)
        {
            const int m = i == 0 ? h : (i == 1 ? 2 * h : 1 + h);
            const double pr = t1r[m] * wr[i] - t1i[m] * wi[i], pi = t1r[m] * wi[i] + t1i[m] * wr[i];
            d[h] = make_double2(pr * fr[h] - pi * fi[h], pr * fi[h] + pi * fr[h]);
        }
        if (i == 1) d23 = d[1];
        out(i, make_double2(d[0].x - d23.x, d[0].y - d23.y));
        if (i != 1) out(i == 0 ? 3 : 4, make_double2(d[1].x - d23.x, d[1].y - d23.y));
        __builtin_amdgcn_sched_barrier(0);
    }
}

// Time of slow sample n (0-based) of a BW-sample series:
// t = t0 + T*(double)(n)/(double)BW  (glass_ucb_waveform.c:843)
__host__ __device__ inline double ucb_sample_time(double T, double t0, int n, int BW)
{
#pragma clang fp contract(off)
    return t0 + T * (double)(n) / (double)BW;
}

// TDI format codes (glass_ucb_waveform.c:965-975)
enum TdiFormat : int { TDI_PHASE = 0, TDI_FREQUENCY = 1, TDI_SANGRIA = 2 };

// utils/src/glass_lisa.h:43-49
constexpr double kSPS = 8.321000e-23;
constexpr double kSACC = 9.000000e-30;
constexpr double kSLOC = 2.89e-24;

__host__ __device__ inline double ipow_(double x, int n)
{
    double xn = 1.0;
    for (int i = 0; i < n; i++) xn *= x;
    return xn;
}

// AEnoise with rednoise (utils/src/glass_lisa.c:1183-1198)
__host__ __device__ inline double ae_noise(double L, double fstar, double f)
{
    double fon = f / fstar;
    double trans = ipow_(sin(fon), 2);
    double red = 1. + 16.0 * (pow((2.0e-5 / f), 10.0) + ipow_(1.0e-4 / f, 2));
    return (16.0 / 3.0) * trans *
           ((2.0 + cos(fon)) * (kSPS + kSLOC) +
            2.0 * (3.0 + 2.0 * cos(fon) + cos(2.0 * fon)) * (kSLOC / 2.0 + kSACC / ipow_(kPI2 * f, 4) * red)) /
           ipow_(2.0 * L, 2);
}

// 2^((int)log2(x) + 1) clamped to [nmin, nmax], as ucb_bandwidth forms its
// Doppler and SNR spreads (ucb/src/glass_ucb_waveform.c:709-722).  Values
// below 8 (including negative or NaN x) land on the floor nmin = 16.
__host__ __device__ inline int pow2_spread(double x, int nmin, int nmax)
{
    if (!(x >= 8.0)) return nmin;
    int e = (int)log2(x) + 1;
    int v = e >= 30 ? (1 << 30) : (1 << e);
    if (v > nmax) v = nmax;
    if (v < nmin) v = nmin;
    return v;
}

// ucb_bandwidth (ucb/src/glass_ucb_waveform.c:698-725)
__host__ __device__ inline int ucb_bandwidth(double L, double fstar, double f, double fdot, double costheta,
                                             double A, double T, int N)
{
#pragma clang fp contract(off)
    const int Nmin = 16;
    int half = N / 2, lg = 0;
    while ((2 << lg) <= half) lg++;  // (int)log2(N/2)
    const int Nmax = 1 << lg;
    double sqT = sqrt(T);
    double sf = sin(f / fstar);
    double sn = ae_noise(L, fstar, f);
    double sintheta = sin(acos(costheta));
    double bw = 2 * T * ((4. + kPI2 * f * (kAU / kCLIGHT) * sintheta) / kYEAR + fabs(fdot) * T);
    int DS = pow2_spread(bw - 1, Nmin, Nmax);
    double SNRm = A * sqT * sf / sqrt(sn);  // analytic_snr, glass_ucb_waveform.c:22-25
    int SS = pow2_spread(SNRm - 1, Nmin, Nmax);
    return (DS > SS) ? DS : SS;
}

}  // namespace glass
