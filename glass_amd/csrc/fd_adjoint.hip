// fd_adjoint.hip -- reverse-mode (adjoint) gradient of one galactic binary's
// likelihood contribution, for many sources at once (no reference
// counterpart: the reference differences whole waveforms in ucb_fisher,
// ucb/src/glass_ucb_waveform.c:364-522).
//
// With L = (R|h) - (h|h)/2 (R the residual without the source) and h the
// TDI of the series spectra d_l = FFT(s_l)/(2N) (fftshifted), the
// gradient is
//   dL/dtheta = (R - h | dh/dtheta) = 2 Re sum_n sum_l conj(ds_l[n]/dtheta) Sb_l[n]
// where the adjoint of the slow series Sb is obtained from the residual in
// three linear steps run backwards:
//   G_b[m]  = sum_a w_ab[j] (R - h)_a[m]            (weighted residual, per bin)
//   Db_l[m] = sum_b conj(T_bl[m]) G_b[m]            (TDI transposed)
//   Sb_l[n] = sum_m exp(+2 pi i n s(m)/N) Db_l[m] / (2N)
//           = conj(FFT(conj(Db_l at index s(m))))[n] / (2N)   (FFT transposed)
// One workgroup per source: the forward pass (fd_link_bins) gives h and L;
// the five adjoint series go back through the same LDS buffer and FFT, the
// P-point step of fd_link_bins transposed after it; a last pass contracts
// each slow sample's tangents with Sb (ucb_sample_adjoint; link 23, which the
// series subtract, has minus the sum of the five).  The four parameters that
// enter linearly (ln A, cos iota, psi, phi0) follow from the basis sums.
// Cost: one waveform, five more FFTs and one tangent pass over the samples
// (the forward-mode Fisher kernel runs six series sets through FFT and TDI).
// The tangents are contracted as they are formed, none is stored; registers
// bound it (201: two waves per SIMD).  1501 sources of 512 bins 182 -> 123 us.
#include <cmath>

#include "../../include/glass_hip_batch.h"
#include "fd_derivs.h"
#include "fd_tangent.h"
#include "reduce.h"
#include "runtime.h"

namespace glass {

int parse_format(const char* format);

namespace {

constexpr int kNAdj = 9;  // L, four tangent gradients, basis sums P0, P1 (complex)

// TDI of bin m as channel = alpha a + beta b with a = d_ij - d_ik and
// b = d_ji - d_ki (fd_tdi: beta = P, alpha = P exp(-ix)).
template <int N>
__device__ inline void tdi_coef(const UcbConst& c, int m, int fmt, double2& alpha, double2& beta)
{
    double s1, c1;
    fd_tdi_phase<N>(c, m, c1, s1);
    beta = fd_tdi_prefactor<N>(c, m, fmt, c1, s1);
    alpha = make_double2(beta.x * c1 + beta.y * s1, beta.y * c1 - beta.x * s1);
}

__device__ inline double2 cconj(double2 a) { return make_double2(a.x, -a.y); }
__device__ inline double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
// conj(a) b
__device__ inline double2 cjmul(double2 a, double2 b)
{
    return make_double2(a.x * b.x + a.y * b.y, a.x * b.y - a.y * b.x);
}

template <int N, bool GRAD>
__global__ __launch_bounds__(fd_threads(N)) void adjoint_kernel(DerivArgs A)
{
    using S = FdShape<N>;
    constexpr int P = S::P, NT = S::NT, PN = S::PN, NTHR = S::NTHR;
    __shared__ double2 lds[S::LDS];
    __shared__ UcbDiff sdd;
    const int e = blockIdx.x;
    const int t = threadIdx.x;
    const double* p = A.params + (size_t)(A.pidx ? A.pidx[e] : e) * 8;
    // the template constants and their derivatives on lanes of two waves,
    // so the two serial setups overlap (one wave at 32/64 bins: in turn)
    __shared__ UcbConst sc;
    if (t == 0) ucb_setup(p, 8, A.T, A.t0, A.L, A.fstar, A.reach, sc);
    if (GRAD && t == (NTHR >= 128 ? 64 : 0)) ucb_diff_setup(p, A.T, sdd);
    __syncthreads();
    UcbConst c = sc;  // into scalar registers for the passes
    c.np = 8;
    make_uniform(c);
    const int posstride = 4096 / N;
    const double2* R = A.iroff ? A.resid + A.iroff[e] : A.resid + (size_t)e * (A.rstride / 2);
    const double* iC = A.iioff ? A.invC + A.iioff[e] : A.invC + (size_t)e * A.istride;
    const int W = A.iW ? A.iW[e] : A.W, imin = A.imin[e];
    double acc[kNAdj];
#pragma unroll
    for (int q = 0; q < kNAdj; q++) acc[q] = 0.0;
    double2 db[P][kNLink];
    // forward: the series of each bin, h, L and the transposed TDI
    fd_link_bins<N, false>(
        HeldConst{c}, lds, opaque(A.pos), posstride, opaque(A.tw), kTwN / N, [](int) {},
        [&](int r, int m, const double2* d) {
            const int j = imin + m;
            const bool used = (A.mode == 0 || m < W) && j >= 0 && j < W;
            double2 G[3] = {make_double2(0.0, 0.0), make_double2(0.0, 0.0), make_double2(0.0, 0.0)};
            if (used)
            {
                double2 h[5];
                fd_tdi<N>(c, m, A.fmt, d, h);
                double w[6];
#pragma unroll
                for (int q = 0; q < 6; q++) w[q] = iC[(size_t)q * W + j];
                double2 res[3], y[3];
#pragma unroll
                for (int ch = 0; ch < 3; ch++)
                {
                    res[ch] = A.resid ? R[(size_t)ch * W + j] : make_double2(0.0, 0.0);
                    y[ch] = make_double2(fma(-0.5, h[ch].x, res[ch].x), fma(-0.5, h[ch].y, res[ch].y));
                }
                // (R|h) - (h|h)/2 = (R - h/2|h)
                auto re = [](double2 a, double2 b) { return a.x * b.x + a.y * b.y; };
                acc[0] += 2.0 * (w[0] * re(y[0], h[0]) + w[1] * re(y[1], h[1]) + w[2] * re(y[2], h[2]) +
                                 w[3] * (re(y[0], h[1]) + re(y[1], h[0])) + w[4] * (re(y[0], h[2]) + re(y[2], h[0])) +
                                 w[5] * (re(y[1], h[2]) + re(y[2], h[1])));
                if constexpr (GRAD)
                {
                    const double2 x0 = csub(res[0], h[0]), x1 = csub(res[1], h[1]), x2 = csub(res[2], h[2]);
                    // G_b = sum_a w_ab (R - h)_a, w symmetric: XX,YY,ZZ,XY,XZ,YZ
                    G[0] = make_double2(w[0] * x0.x + w[3] * x1.x + w[4] * x2.x, w[0] * x0.y + w[3] * x1.y + w[4] * x2.y);
                    G[1] = make_double2(w[3] * x0.x + w[1] * x1.x + w[5] * x2.x, w[3] * x0.y + w[1] * x1.y + w[5] * x2.y);
                    G[2] = make_double2(w[4] * x0.x + w[5] * x1.x + w[2] * x2.x, w[4] * x0.y + w[5] * x1.y + w[2] * x2.y);
                }
            }
            if constexpr (GRAD)
            {
                double2 al, be;
                tdi_coef<N>(c, m, A.fmt, al, be);
                // X = al (d0 - d3) + be (d1 - d2), Y = -al d1 + be (d4 - d0),
                // Z = al (d2 - d4) + be d3; conj(Db_l) = conj(sum_b conj(T_bl) G_b)
                const double2 aX = cconj(cjmul(al, G[0])), bX = cconj(cjmul(be, G[0]));
                const double2 aY = cconj(cjmul(al, G[1])), bY = cconj(cjmul(be, G[1]));
                const double2 aZ = cconj(cjmul(al, G[2])), bZ = cconj(cjmul(be, G[2]));
                double2(&o)[kNLink] = db[r];
                o[0] = csub(aX, bY);
                o[1] = csub(bX, aY);
                o[2] = csub(aZ, bX);
                o[3] = csub(bZ, aX);
                o[4] = csub(bY, aZ);
            }
        });
    if constexpr (GRAD)
    {
        // bin m = P t + r is FFT index P k + r: per residue r the NT-point
        // transform over k, then sample n = t + NT p sums the residues with
        // w_N^{r t} w_P^{r p}
        const int k = S::place(t + NT / 2), ts = S::place(t);
        const bool on = NT >= 64 || t < NT;
#pragma unroll
        for (int r = 0; r < P; r++)
        {
            __syncthreads();  // the LDS reads of the pass before
            if (on)
#pragma unroll
                for (int l = 0; l < kNLink; l++) lds[l * PN + k] = db[r][l];
            __syncthreads();
            wave_fft<NT, kNLink, NTHR>(lds, opaque(A.tw), P * (kTwN / N));
            const double2 w = r ? A.tw[(r * t) * (kTwN / N)] : make_double2(1.0, 0.0);
#pragma unroll
            for (int l = 0; l < kNLink; l++) db[r][l] = r ? cmul(lds[l * PN + ts], w) : lds[l * PN + ts];
        }
        if constexpr (P > 1)
#pragma unroll
            for (int l = 0; l < kNLink; l++)
            {
                double2 v[P], y[P];
#pragma unroll
                for (int r = 0; r < P; r++) v[r] = db[r][l];
                radix_butterfly<P>(v, y);
#pragma unroll
                for (int q = 0; q < P; q++) db[q][l] = y[q];
            }
        // one sample's temporaries at a time (unrolled, the 1024-bin kernel
        // spilled 560 bytes): the samples move down to db[0]
        if (on)
#pragma unroll 1
            for (int q = 0; q < P; q++)
            {
                const int n = t + NT * q;
                double2 Sb[6];
                double2 sum = make_double2(0.0, 0.0);
#pragma unroll
                for (int l = 0; l < kNLink; l++)
                {
                    const double2 v = cconj(db[0][l]);
                    Sb[l < 4 ? l : 5] = v;
                    sum = make_double2(sum.x - v.x, sum.y - v.y);
                }
                Sb[4] = sum;
                ucb_sample_adjoint(c, sdd, ucb_sample_time(c.T, c.t0, n, N), A.pos + (size_t)n * posstride * 9,
                                   [&](int l) { return Sb[l]; }, acc + 1);
#pragma unroll
                for (int i = 0; i + 1 < P; i++)
#pragma unroll
                    for (int l = 0; l < kNLink; l++) db[i][l] = db[i + 1][l];
            }
    }
    // workgroup sums of the nine partials
    constexpr int NS = GRAD ? kNAdj : 1;
    __shared__ double tot[NS];
    double part[NS];
#pragma unroll
    for (int q = 0; q < NS; q++) part[q] = acc[q];
    block_sum_many<NTHR, NS>(part, tot);
    if (t == 0)
    {
        A.outL[e] = tot[0];
        if constexpr (GRAD)
        {
            const UcbDiff& dd = sdd;
            const double2 P0 = make_double2(tot[5], tot[6]), P1 = make_double2(tot[7], tot[8]);
            // s = DP s0 + DC s1: conj(ds) Sb summed = conj(dDP) P0 + conj(dDC) P1
            auto lin = [&](double2 a, double2 b) {
                const double2 u = cjmul(a, P0), v = cjmul(b, P1);
                return make_double2(u.x + v.x, u.y + v.y);
            };
            const double2 sP = lin(make_double2(c.DPr, c.DPi), make_double2(c.DCr, c.DCi));
            double* g = A.grad + (size_t)e * 8;
            g[0] = 2.0 * tot[1];                                                    // f0 T
            g[1] = 2.0 * tot[2];                                                    // cos(theta)
            g[2] = 2.0 * tot[3];                                                    // phi
            g[3] = 2.0 * sP.x;                                                      // ln A: ds = s
            g[4] = 2.0 * lin(make_double2(dd.DPr4, dd.DPi4), make_double2(dd.DCr4, dd.DCi4)).x;  // cos(iota)
            g[5] = 2.0 * lin(make_double2(dd.DPr5, dd.DPi5), make_double2(dd.DCr5, dd.DCi5)).x;  // psi
            g[6] = -2.0 * sP.y;                                                     // phi0: ds = -i s
            g[7] = 2.0 * tot[4];                                                    // fdot T^2
        }
    }
}

}  // namespace

int launch_adjoint(int N, const DerivArgs& A, int n, bool want_grad, hipStream_t s)
{
    if (n <= 0) return GLASS_HIP_OK;
    switch (N)
    {
#define GH_A(NN)                                                                                   \
    case NN:                                                                                       \
        if (want_grad)                                                                             \
            adjoint_kernel<NN, true><<<n, fd_threads(NN), 0, s>>>(A);                              \
        else                                                                                       \
            adjoint_kernel<NN, false><<<n, fd_threads(NN), 0, s>>>(A);                             \
        break;
        GH_A(32) GH_A(64) GH_A(128) GH_A(256) GH_A(512) GH_A(1024)
#undef GH_A
        default: set_error("fd adjoint: BW=%d unsupported (power of two 32..1024)", N); return GLASS_HIP_EINVAL;
    }
    GH_CHECK(hipGetLastError());
    return GLASS_HIP_OK;
}

}  // namespace glass

using namespace glass;

extern "C" int glass_hip_fd_source_grad(const glass_hip_orbit* orbit, const char* format, double T, double t0, int n,
                                        const double* d_params, int BW, const int* d_imin, int W,
                                        const double* d_resid, long long resid_stride, const double* d_invC,
                                        long long invC_stride, int mode, double* d_logL, double* d_grad,
                                        void* stream)
{
    int fmt = parse_format(format);
    if (fmt < 0)
    {
        set_error("Unsupported data format %s", format ? format : "(null)");
        return GLASS_HIP_EINVAL;
    }
    if (!orbit || n < 0 || !d_params || !d_imin || W < 1 || !d_invC || !d_logL || (mode != 0 && mode != 1) ||
        resid_stride < 0 || invC_stride < 0)
    {
        set_error("fd_source_grad: bad arguments");
        return GLASS_HIP_EINVAL;
    }
    if (n == 0) return GLASS_HIP_OK;
    const double* pos;
    const double2* tw;
    int rc;
    if ((rc = positions(*orbit, T, t0, 4096, &pos)) || (rc = twiddles(&tw))) return rc;
    DerivArgs A{};
    A.params = d_params;
    A.imin = d_imin;
    A.W = W;
    A.resid = (const double2*)d_resid;
    A.rstride = resid_stride;
    A.invC = d_invC;
    A.istride = invC_stride;
    A.mode = mode;
    A.T = T;
    A.t0 = t0;
    A.L = orbit->L;
    A.fstar = orbit->fstar;
    A.reach = analytic_reach(orbit->L, orbit->fstar, orbit->R, T, t0);
    A.pos = pos;
    A.tw = tw;
    A.fmt = fmt;
    A.outL = d_logL;
    A.grad = d_grad;
    return launch_adjoint(BW, A, n, d_grad != nullptr, (hipStream_t)stream);
}
