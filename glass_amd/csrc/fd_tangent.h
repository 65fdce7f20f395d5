// fd_tangent.h -- exact parameter derivatives of the frequency-domain UCB
// template (forward mode), built on the same slow-series construction as
// the waveform (ucb/src/glass_ucb_waveform.c:804-962).
//
// One link sample is V = aevol T S E with
//   S  = sin(arg1)/(4 arg1),  arg1 = f_i/(2 f*) (1 + k.r_ij)
//   T  = d+ DP + dx DC,  DP = DPr + i DPi, DC = DCr + i DCi
//   E  = exp(-i Phi),  Phi = arg1 - arg2
// and FFT + TDI are complex-linear with parameter-independent coefficients
// (q and BW held fixed), so d h / d theta = TDI(FFT(d V / d theta)).
// Because V is complex-linear in (DP, DC):
//   h = DP Hp + DC Hc  with Hp = TDI FFT (S aevol d+ E), Hc likewise with dx,
//   d h/d lnA  = h,   d h/d phi0 = -i h,
//   d h/d cos(iota), d h/d psi = DP' Hp + DC' Hc  (DP', DC' closed form),
// leaving genuine tangent series only for f0 T, cos(theta), phi and
// fdot T^2.  The six "series sets" built per sample are
//   0: S aevol d+ E    1: S aevol dx E
//   2: dV/d(f0 T)      3: dV/d cos(theta)   4: dV/d phi   5: dV/d(fdot T^2)
// each as the five series of fd_waveform.h (links less link 23).
//
// With B = S E and B1 = d(S exp(-i arg1))/d arg1 exp(i arg2),
//   dV = T B (daevol + i aevol darg2) + T B1 aevol darg1 + dT B aevol,
// real factors per spacecraft but for T and dT, which belong to the arm: the
// sample's own values (ucb_slow_sample_to) and one more polynomial give all
// sets; the sky derivatives of an arm r follow from its components along
// (cos phi, sin phi), along v and along z.
#pragma once
#include "fd_waveform.h"

namespace glass {

// Sky and polarisation pieces needed by the derivatives.
struct UcbDiff
{
    double ct, st, cph, sph;  // cos, sin of theta and phi
    double cot;               // -d sin(theta)/d cos(theta)
    double DPr4, DPi4, DCr4, DCi4;  // d(DP, DC)/d cos(iota)
    double DPr5, DPi5, DCr5, DCi5;  // d(DP, DC)/d psi
    double invT, invT2, f0;
};

__host__ __device__ inline void ucb_diff_setup(const double* p, double T, UcbDiff& d)
{
    const double costh = p[1], phi = p[2], amp = exp(p[3]), cosi = p[4], psi = p[5];
    d.ct = costh;
    d.st = sqrt(1.0 - costh * costh);
    d.cph = cos(phi);
    d.sph = sin(phi);
    // d sin(theta)/d cos(theta) = -cot diverges at the poles (|cos theta| =
    // 1, where clipped proposals land); there the tangent is taken as at
    // |cos theta| = 1 - 1e-6, the reference's Fisher step
    // (ucb/src/glass_ucb_waveform.c:369-415), so the Fisher matrix stays
    // finite (sin theta >= sqrt(2e-6) in the cotangent only)
    d.cot = costh / fmax(d.st, 1.4142135623730951e-3);
    const double cosps = cos(2. * psi), sinps = sin(2. * psi);
    const double Aplus = amp * (1. + cosi * cosi) * 0.5, Across = -amp * cosi;
    // dAplus/dcos(iota) = amp cos(iota), dAcross/dcos(iota) = -amp
    d.DPr4 = amp * cosi * cosps;  d.DPi4 = amp * sinps;
    d.DCr4 = -amp * cosi * sinps; d.DCi4 = amp * cosps;
    // d cos(2 psi)/d psi = -2 sin(2 psi), d sin(2 psi)/d psi = 2 cos(2 psi)
    d.DPr5 = -2.0 * Aplus * sinps;  d.DPi5 = -2.0 * Across * cosps;
    d.DCr5 = -2.0 * Aplus * cosps;  d.DCi5 = 2.0 * Across * sinps;
    d.invT = 1.0 / T;
    d.invT2 = 1.0 / (T * T);
    d.f0 = p[0] / T;
}

__device__ inline double2 cmulc(double2 a, double2 b) { return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); }

// An arm r (over L): its d+ and dx, T = d+ DP + dx DC, and if TAN their
// derivatives by cos(theta) (1) and phi (2) and those of k.r.
template <bool TAN>
struct UcbArm
{
    double dp, dc, kr;
    double2 T;
    double2 T1, T2;
    double k1, k2;
    __device__ __forceinline__ UcbArm(const UcbConst& c, const UcbDiff& dd, double r0, double r1, double r2)
    {
        r0 *= c.invL;
        r1 *= c.invL;
        r2 *= c.invL;
        const double p = r0 * dd.cph + r1 * dd.sph, v = r0 * dd.sph - r1 * dd.cph, z = r2;
        const double u = dd.ct * p - dd.st * z;
        kr = -(dd.st * p + dd.ct * z);
        dp = v * v - u * u;
        dc = 2.0 * u * v;
        T = make_double2(dp * c.DPr + dc * c.DCr, dp * c.DPi + dc * c.DCi);
        if constexpr (TAN)
        {
            const double u1 = p + dd.cot * z, v2 = 2.0 * v;
            const double dp1 = -2.0 * u * u1, dc1 = v2 * u1;
            const double dp2 = v2 * (p + dd.ct * u), dc2 = 2.0 * u * p - v2 * dd.ct * v;
            T1 = make_double2(dp1 * c.DPr + dc1 * c.DCr, dp1 * c.DPi + dc1 * c.DCi);
            T2 = make_double2(dp2 * c.DPr + dc2 * c.DCr, dp2 * c.DPi + dc2 * c.DCi);
            k1 = dd.cot * p - z;
            k2 = dd.st * v;
        }
    }
};

// What the links of one spacecraft share at a sample.
struct UcbCraft
{
    double ae;             // aevol
    double wr, wi;         // exp(i arg2)/4
    double hf;             // f_i/(2 f*)
    double da2[4], dae[4], dfo[4], fon;  // derivatives by f0 T, cos(theta), phi, fdot T^2; f_i/f*
};

// The three spacecraft of a sample (arg2 as ucb_slow_sample_to forms it).
template <bool TAN>
__device__ __forceinline__ void ucb_crafts(const UcbConst& c, const UcbDiff& dd, double t, const double (&x)[3],
                                           const double (&y)[3], const double (&z)[3], UcbCraft (&C)[3])
{
    double a2[3], xi[3];
    double dft;
    {
#pragma clang fp contract(off)
        dft = c.df * t;
    }
#pragma unroll
    for (int i = 0; i < 3; i++)
    {
#pragma clang fp contract(off)
        const double kdotx = div_by_recip(x[i] * c.k[0] + y[i] * c.k[1] + z[i] * c.k[2], kCLIGHT, kInvCLIGHT);
        xi[i] = t - kdotx;
        a2[i] = c.pi2f0 * xi[i] - c.phi0 - dft;
        a2[i] += c.pidfdt * xi[i] * xi[i];
    }
    double sn[3], cs[3];
    unsigned fl[3];
    sincos_half<3>(a2, sn, cs, fl);
    const double ca = 0.66666666666666666666;
#pragma unroll
    for (int i = 0; i < 3; i++)
    {
        UcbCraft& q = C[i];
        const double quarter = flip_sign(0.25, fl[i]);
        q.wr = quarter * cs[i];
        q.wi = quarter * sn[i];
        q.ae = fma(c.aevc, xi[i], 1.0);
        q.hf = fma(c.dfh, xi[i], c.f0h);
        if constexpr (TAN)
        {
            const double p = x[i] * dd.cph + y[i] * dd.sph, v = x[i] * dd.sph - y[i] * dd.cph;
            const double dx1 = -(dd.cot * p - z[i]) * kInvCLIGHT, dx2 = -(dd.st * v) * kInvCLIGHT;
            const double w = kPI2 * fma(c.dfdt, xi[i], dd.f0);
            const double xT = xi[i] * dd.invT;
            q.da2[0] = kPI2 * xT;
            q.da2[1] = w * dx1;
            q.da2[2] = w * dx2;
            q.da2[3] = kPI * xT * xT;
            const double g = c.dfdt * c.invfstar;
            q.dfo[0] = dd.invT * c.invfstar;
            q.dfo[1] = g * dx1;
            q.dfo[2] = g * dx2;
            q.dfo[3] = xT * dd.invT * c.invfstar;
            q.fon = fma(c.dfdt, xi[i], c.f0) * c.invfstar;
            q.dae[1] = c.aevc * dx1;
            q.dae[2] = c.aevc * dx2;
            q.dae[0] = -c.aevc * xT / dd.f0;
            q.dae[3] = ca * xT * dd.invT / dd.f0;
        }
    }
}

// Series sets [S0, S0+NS) of one slow sample at time t: out(set, series,
// value) for every set of the range and the five series (links 12, 21, 31,
// 13, 32 less link 23).  Sets 0, 1: the plus / cross basis (the sample is DP
// s0 + DC s1, complex products); 2..5: d/d(f0 T), d/dcos(theta), d/dphi,
// d/d(fdot T^2).
template <int S0, int NS, typename Out>
__device__ __forceinline__ void ucb_sample_sets_to(const UcbConst& c, const UcbDiff& dd, double t,
                                                   const double* __restrict__ pos, Out&& out)
{
    constexpr bool W01 = S0 <= 1;      // any basis set
    constexpr bool WT = S0 + NS > 2;   // any tangent set
    const double x[3] = {pos[0], pos[1], pos[2]}, y[3] = {pos[3], pos[4], pos[5]}, z[3] = {pos[6], pos[7], pos[8]};
    UcbCraft C[3];
    ucb_crafts<WT>(c, dd, t, x, y, z, C);
    const UcbArm<WT> arm[3] = {{c, dd, x[1] - x[0], y[1] - y[0], z[1] - z[0]},
                               {c, dd, x[2] - x[0], y[2] - y[0], z[2] - z[0]},
                               {c, dd, x[2] - x[1], y[2] - y[1], z[2] - z[1]}};
    double2 d23[NS];
#pragma unroll
    for (int w = 0; w < 3; w++)
    {
        const int i = w == 0 ? 1 : (w == 1 ? 0 : 2);  // spacecraft 2 first: link 23
        const UcbCraft& q = C[i];
        const int am[2] = {i == 2 ? 1 : 0, i == 0 ? 1 : 2};
        const double sg[2] = {i == 0 ? 1.0 : -1.0, i == 2 ? -1.0 : 1.0};
        const double xx[2] = {q.hf + sg[0] * q.hf * arm[am[0]].kr, q.hf + sg[1] * q.hf * arm[am[1]].kr};
        double s[2], cc[2], ds[2];
        sinc_values<WT>(xx, c.wide, s, cc, ds);
        // link 23 (h = 1 of spacecraft 2) before 21
#pragma unroll
        for (int hh = 0; hh < 2; hh++)
        {
            const int h = i == 1 ? 1 - hh : hh;
            const UcbArm<WT>& A = arm[am[h]];
            // S exp(-i arg1) (times 4) and its derivative
            const double fr = s[h] * cc[h], fi = -(xx[h] * s[h]) * s[h];
            const double2 B = make_double2(q.wr * fr - q.wi * fi, q.wr * fi + q.wi * fr);
            auto emit = [&](int k, double2 v) {
                if (i == 1 && h == 1)
                    d23[k - S0] = v;
                else
                    out(k, i == 1 ? 1 : (i == 0 ? (h ? 3 : 0) : (h ? 4 : 2)),
                        make_double2(v.x - d23[k - S0].x, v.y - d23[k - S0].y));
            };
            if constexpr (W01)
            {
#pragma unroll
                for (int k = 0; k < 2; k++)
                {
                    if (k < S0 || k >= S0 + NS) continue;
                    const double g = q.ae * (k == 0 ? A.dp : A.dc);
                    emit(k, make_double2(g * B.x, g * B.y));
                }
            }
            if constexpr (WT)
            {
                const double br = ds[h] * cc[h] - xx[h] * s[h] * s[h], bi = -(ds[h] * xx[h] * s[h] + s[h] * cc[h]);
                // exp(-i x) = c - i x s: (ds - i s)(c - i x s)
                const double2 B1 = make_double2(q.wr * br - q.wi * bi, q.wr * bi + q.wi * br);
                const double2 M = cmulc(A.T, B), M1 = cmulc(A.T, B1);
                const double kp = 1.0 + sg[h] * A.kr;
#pragma unroll
                for (int k = 2; k < 6; k++)
                {
                    if (k < S0 || k >= S0 + NS) continue;
                    const int v = k - 2;  // 0: f0 T, 1: cos(theta), 2: phi, 3: fdot T^2
                    double da = q.dfo[v] * kp;
                    if (v == 1) da += q.fon * (sg[h] * A.k1);
                    if (v == 2) da += q.fon * (sg[h] * A.k2);
                    const double g = q.ae * (0.5 * da), b = q.ae * q.da2[v];
                    double2 o = make_double2(q.dae[v] * M.x - b * M.y + g * M1.x, q.dae[v] * M.y + b * M.x + g * M1.y);
                    if (v == 1 || v == 2)
                    {
                        const double2 dT = v == 1 ? A.T1 : A.T2;
                        const double2 e = cmulc(make_double2(q.ae * dT.x, q.ae * dT.y), B);
                        o.x += e.x;
                        o.y += e.y;
                    }
                    emit(k, o);
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// The contraction of one sample's tangents with the adjoint series: sb(l) =
// adjoint of link l (12, 21, 31, 13, 23, 32).  acc[0..3] gains Re conj(dV) Sb
// for f0 T, cos(theta), phi, fdot T^2 and acc[4..7] the complex basis sums
// P0, P1 (Sb against the plus and cross basis).  The tangents themselves are
// not formed: conj(B) Sb and conj(B1) Sb per link, then real factors.
template <typename Sb>
__device__ __forceinline__ void ucb_sample_adjoint(const UcbConst& c, const UcbDiff& dd, double t,
                                                   const double* __restrict__ pos, Sb&& sb, double* acc)
{
    const double x[3] = {pos[0], pos[1], pos[2]}, y[3] = {pos[3], pos[4], pos[5]}, z[3] = {pos[6], pos[7], pos[8]};
    UcbCraft C[3];
    ucb_crafts<true>(c, dd, t, x, y, z, C);
    const UcbArm<true> arm[3] = {{c, dd, x[1] - x[0], y[1] - y[0], z[1] - z[0]},
                                 {c, dd, x[2] - x[0], y[2] - y[0], z[2] - z[0]},
                                 {c, dd, x[2] - x[1], y[2] - y[1], z[2] - z[1]}};
    auto cj = [](double2 a, double2 b) { return make_double2(a.x * b.x + a.y * b.y, a.x * b.y - a.y * b.x); };
#pragma unroll
    for (int i = 0; i < 3; i++)
    {
        const UcbCraft& q = C[i];
        const int am[2] = {i == 2 ? 1 : 0, i == 0 ? 1 : 2};
        const double sg[2] = {i == 0 ? 1.0 : -1.0, i == 2 ? -1.0 : 1.0};
        const double xx[2] = {q.hf + sg[0] * q.hf * arm[am[0]].kr, q.hf + sg[1] * q.hf * arm[am[1]].kr};
        double s[2], cc[2], ds[2];
        sinc_values<true>(xx, c.wide, s, cc, ds);
#pragma unroll
        for (int h = 0; h < 2; h++)
        {
            const UcbArm<true>& A = arm[am[h]];
            const double fr = s[h] * cc[h], fi = -(xx[h] * s[h]) * s[h];
            const double br = ds[h] * cc[h] - xx[h] * s[h] * s[h], bi = -(ds[h] * xx[h] * s[h] + s[h] * cc[h]);
            const double2 B = make_double2(q.wr * fr - q.wi * fi, q.wr * fi + q.wi * fr);
            const double2 B1 = make_double2(q.wr * br - q.wi * bi, q.wr * bi + q.wi * br);
            const double2 S = sb(i + 3 * h);
            const double2 Z = cj(B, S), Z1 = cj(B1, S), Q = cj(A.T, Z);
            const double q1 = A.T.x * Z1.x + A.T.y * Z1.y;  // Re conj(T B1) Sb
            const double kp = 1.0 + sg[h] * A.kr;
            // Re conj(M (dae + i b)) Sb = dae Re Q + b Im Q, Q = conj(M) Sb
            const double az[4] = {0.0, A.T1.x * Z.x + A.T1.y * Z.y, A.T2.x * Z.x + A.T2.y * Z.y, 0.0};
            const double dk[4] = {0.0, sg[h] * A.k1, sg[h] * A.k2, 0.0};
#pragma unroll
            for (int v = 0; v < 4; v++)
            {
                const double da = q.dfo[v] * kp + (v == 1 || v == 2 ? q.fon * dk[v] : 0.0);
                acc[v] += q.dae[v] * Q.x + q.ae * (q.da2[v] * Q.y + 0.5 * da * q1 + (v == 1 || v == 2 ? az[v] : 0.0));
            }
            const double g0 = q.ae * A.dp, g1 = q.ae * A.dc;
            acc[4] += g0 * Z.x;
            acc[5] += g0 * Z.y;
            acc[6] += g1 * Z.x;
            acc[7] += g1 * Z.y;
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

}  // namespace glass
