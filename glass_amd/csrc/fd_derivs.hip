// fd_derivs.hip -- exact gradient and Fisher matrix of one galactic binary's
// likelihood contribution, for many sources at once (no reference
// counterpart: the reference's ucb_fisher, ucb/src/glass_ucb_waveform.c:
// 364-522, uses forward differences of 8 extra waveforms).
//
// For a source with template h(theta) over a residual R that excludes it,
// logL = const + L(theta),  L = (R|h) - (h|h)/2,  so
//   dL/dtheta_k = (R - h | dh/dtheta_k),   Gamma_kl = (dh_k | dh_l),
// with ( | ) the 3-channel noise-weighted product of gaussian_log_likelihood
// (utils/src/glass_model.c:758-767).  One workgroup per source: the six
// series sets of fd_tangent.h go through LDS and FFT in passes of a few sets,
// each TDI'd into per-bin values u_q; every thread then adds its bins'
// Hermitian Gram G_qr = u_q^H W u_r (36 real numbers) and projections
// P_q = (W (R - h))^H u_q (12), and the workgroup reduces the 48 sums.  All
// eight dh/dtheta are fixed complex combinations of the six u_q, so L, the
// gradient and the Fisher matrix follow from them: 420 multiply-adds a bin
// where the 45 real products of the dh/dtheta took 1250.  Registers bound it:
// the bin's 18 complex values are held through the sample passes, so two waves
// per SIMD are resident (253 vector registers; three waves spill, and were
// slower).  8192 sources of 256 bins 0.57 -> 0.41 ms; 16,384 sources of a
// sampler's chains, 32 to 4096 bins, 4.4 -> 3.2 ms.
#include <cmath>

#include "../../include/glass_hip_batch.h"
#include "fd_derivs.h"
#include "fd_tangent.h"
#include "reduce.h"
#include "runtime.h"

namespace glass {

int parse_format(const char* format);

// Sums of one source: G_qq (6), Re and Im of G_qr for q < r (15 pairs), Re
// and Im of P_q (6 pairs), and in mode 1 h^H W h with the likelihood's weights.
constexpr int kNSum = 49, kNMain = 48, kGOff = 6, kPOff = 36;
__host__ __device__ constexpr int gram_index(int q, int r) { return kGOff + 2 * (q * 5 - q * (q - 1) / 2 + r - q - 1); }

// Series sets per pass.  Three up to 512 bins (two passes; 138 KB of LDS at
// 512, two workgroups per CU at 256): each pass evaluates the sample's
// common part again.  One above, where a thread holds P results of every
// series through its samples.
constexpr int deriv_sets(int N) { return N <= 512 ? 3 : 1; }

// One pass: series sets [S0, S0+NS) of the slow samples -> LDS -> FFT ->
// TDI: out(r, set, X, Y, Z) for the thread's bins m = P t + r.
template <int N, int S0, int NS, typename Out>
__device__ __forceinline__ void deriv_pass(const UcbConst& c, const UcbDiff& dd, double2* lds, const DerivArgs& A,
                                           Out&& out)
{
    using S = FdShape<N, 1>;
    constexpr int P = S::P, NT = S::NT, PN = S::PN, L = NS * kNLink;
    const int t = threadIdx.x;
    const bool on = NT >= 64 || t < NT;
    const int ts = wave_fft_slot(t);
    const double2* tw = opaque(A.tw);
    const double* pos = opaque(A.pos);
    double2 x[P][L];
    if constexpr (P == 1)
    {
        if (on)
            ucb_sample_sets_to<S0, NS>(c, dd, ucb_sample_time(c.T, c.t0, t, N), pos + (size_t)t * (4096 / N) * 9,
                                       [&](int q, int l, double2 v) { lds[((q - S0) * kNLink + l) * PN + ts] = v; });
    }
    else
    {
#pragma unroll
        for (int p = 0; p < P; p++)
#pragma unroll
            for (int l = 0; l < L; l++) x[p][l] = make_double2(0.0, 0.0);
#pragma unroll 1
        for (int p = 0; p < P; p++)
        {
            const int n = t + NT * p;
            ucb_sample_sets_to<S0, NS>(c, dd, ucb_sample_time(c.T, c.t0, n, N), pos + (size_t)n * (4096 / N) * 9,
                                       [&](int q, int l, double2 v) {
                                           const int k = (q - S0) * kNLink + l;
#pragma unroll
                                           for (int j = 0; j + 1 < P; j++) x[j][k] = x[j + 1][k];
                                           x[P - 1][k] = v;
                                       });
        }
        fd_dif<N, L>(x, tw, kTwN / N, t);
#pragma unroll
        for (int l = 0; l < L; l++) lds[l * PN + ts] = x[0][l];
    }
    __syncthreads();
    const int k = wave_fft_slot((t + NT / 2) & (NT - 1));
#pragma unroll
    for (int r = 0; r < P; r++)
    {
        wave_fft<NT, L, S::NTHR>(lds, opaque(A.tw), P * (kTwN / N));
        double2 d[L];
        if (on)
#pragma unroll
            for (int l = 0; l < L; l++) d[l] = lds[l * PN + k];
        __syncthreads();
        if (r + 1 < P)
#pragma unroll
            for (int l = 0; l < L; l++) lds[l * PN + ts] = x[r + 1][l];
        if (on)
        {
            const int m = P * t + r;
            double s1, c1;
            fd_tdi_phase<N>(c, m, c1, s1);
            const double2 pf = fd_tdi_prefactor<N>(c, m, A.fmt, c1, s1);
#pragma unroll
            for (int q = 0; q < NS; q++)
            {
                double2 X, Y, Z;
                fd_tdi_xyz(c1, s1, pf, d + q * kNLink, X, Y, Z);
                out(r, S0 + q, X, Y, Z);
            }
        }
        if (r + 1 < P) __syncthreads();
    }
}

// All passes, the highest sets first: the tangent sets (2-5, the costly
// samples) run while few TDI values of earlier passes are held in registers.
template <int N, int S1, typename Out>
__device__ __forceinline__ void deriv_passes(const UcbConst& c, const UcbDiff& dd, double2* lds, const DerivArgs& A,
                                             Out&& out)
{
    constexpr int NS = S1 < deriv_sets(N) ? S1 : deriv_sets(N);
    deriv_pass<N, S1 - NS, NS>(c, dd, lds, A, out);
    if constexpr (S1 - NS > 0) deriv_passes<N, S1 - NS>(c, dd, lds, A, out);
}

// The window and residual of item e.
struct DerivItem
{
    const double2* R;   // residual, 3 x W complex
    const double* iC;   // invC, 6 x W
    const double2* Ha;  // stored template added back (or NULL)
    int W, imin, hcap;
};

__device__ __forceinline__ DerivItem deriv_item(const DerivArgs& A, int e)
{
    DerivItem it;
    it.R = A.iroff ? A.resid + A.iroff[e] : A.resid + (size_t)e * (A.rstride / 2);
    it.iC = A.iioff ? A.invC + A.iioff[e] : A.invC + (size_t)e * A.istride;
    it.W = A.iW ? A.iW[e] : A.W;
    it.imin = A.imin[e];
    it.Ha = A.tadd ? A.tadd + A.taddoff[e] : nullptr;
    it.hcap = A.tadd ? A.taddcap[e] : 0;
    return it;
}

// y = W u for the symmetric weights w = XX, YY, ZZ, XY, XZ, YZ
__device__ __forceinline__ void wmul(const double* w, const double2* u, double2* y)
{
    y[0] = make_double2(w[0] * u[0].x + w[3] * u[1].x + w[4] * u[2].x, w[0] * u[0].y + w[3] * u[1].y + w[4] * u[2].y);
    y[1] = make_double2(w[3] * u[0].x + w[1] * u[1].x + w[5] * u[2].x, w[3] * u[0].y + w[1] * u[1].y + w[5] * u[2].y);
    y[2] = make_double2(w[4] * u[0].x + w[5] * u[1].x + w[2] * u[2].x, w[4] * u[0].y + w[5] * u[1].y + w[2] * u[2].y);
}

// Adds template bin m's terms to the sums from its six sets' TDI values u.
__device__ __forceinline__ void deriv_bin(const UcbConst& c, const DerivArgs& A, const DerivItem& it, int m,
                                          const double2 (&u)[6][3], double (&acc)[kNSum])
{
    const int W = it.W, j = it.imin + m;
    const int wi = A.mode == 1 ? m : j;  // Fisher weight index
    const bool inwin = j >= 0 && j < W;
    if (wi < 0 || wi >= W) return;
    double w[6];
#pragma unroll
    for (int q = 0; q < 6; q++) w[q] = it.iC[(size_t)q * W + wi];
    if (inwin)
    {
        // likelihood terms only where the template lands in the window
        double2 h[3], x[3], z[3];
#pragma unroll
        for (int ch = 0; ch < 3; ch++)
        {
            const double2 a = u[0][ch], b = u[1][ch];
            h[ch] = make_double2(c.DPr * a.x - c.DPi * a.y + c.DCr * b.x - c.DCi * b.y,
                                 c.DPr * a.y + c.DPi * a.x + c.DCr * b.y + c.DCi * b.x);
            double2 r = A.resid ? it.R[(size_t)ch * W + j] : make_double2(0.0, 0.0);
            if (it.Ha)
            {
                // the residual of the whole model plus this source's stored
                // template: the residual without the source
                r.x += it.Ha[(size_t)ch * it.hcap + m].x;
                r.y += it.Ha[(size_t)ch * it.hcap + m].y;
            }
            x[ch] = make_double2(r.x - h[ch].x, r.y - h[ch].y);
        }
        if (A.mode == 1)
        {
            double wj[6];
#pragma unroll
            for (int q = 0; q < 6; q++) wj[q] = it.iC[(size_t)q * W + j];
            wmul(wj, x, z);
            double2 y[3];
            wmul(wj, h, y);
#pragma unroll
            for (int ch = 0; ch < 3; ch++) acc[kNMain] += h[ch].x * y[ch].x + h[ch].y * y[ch].y;
        }
        else
            wmul(w, x, z);
#pragma unroll
        for (int q = 0; q < 6; q++)
#pragma unroll
            for (int ch = 0; ch < 3; ch++)
            {
                acc[kPOff + 2 * q] += z[ch].x * u[q][ch].x + z[ch].y * u[q][ch].y;
                acc[kPOff + 2 * q + 1] += z[ch].x * u[q][ch].y - z[ch].y * u[q][ch].x;
            }
    }
#pragma unroll
    for (int r = 0; r < 6; r++)
    {
        double2 y[3];
        wmul(w, u[r], y);
#pragma unroll
        for (int ch = 0; ch < 3; ch++) acc[r] += u[r][ch].x * y[ch].x + u[r][ch].y * y[ch].y;
#pragma unroll
        for (int q = 0; q < r; q++)
#pragma unroll
            for (int ch = 0; ch < 3; ch++)
            {
                acc[gram_index(q, r)] += u[q][ch].x * y[ch].x + u[q][ch].y * y[ch].y;
                acc[gram_index(q, r) + 1] += u[q][ch].x * y[ch].y - u[q][ch].y * y[ch].x;
            }
    }
}

// Workgroup sums of the per-thread sums into red[kNSum]; buf: the FFT buffer
// (its readers have passed a barrier).
template <int NTHR, int CH>
__device__ __forceinline__ void deriv_reduce(const double (&acc)[kNSum], double* buf, double* red, bool extra)
{
    block_sum_rows<NTHR, CH, kNMain>(acc, buf, red);
    const double s = extra ? block_sum<NTHR>(acc[kNMain]) : 0.0;
    if (threadIdx.x == 0) red[kNMain] = s;
    __syncthreads();
}

// L, gradient and Fisher matrix of item e from the reduced sums: dh/dtheta_a
// = A u_q + B u_s with at most two sets.
__device__ __forceinline__ void deriv_write(const UcbConst& c, const UcbDiff& dd, const DerivArgs& A, int e,
                                            const double* red)
{
    if (threadIdx.x >= 64) return;
    auto coef = [&](int a, int& q, double2& ca, double2& cb) {
        const int set[8] = {2, 3, 4, 0, 0, 0, 0, 5};
        q = set[a];
        ca = make_double2(1.0, 0.0);
        cb = make_double2(0.0, 0.0);
        const double2 DP = make_double2(c.DPr, c.DPi), DC = make_double2(c.DCr, c.DCi);
        if (a == 3) ca = DP, cb = DC;                                                        // ln A: h
        if (a == 4) ca = make_double2(dd.DPr4, dd.DPi4), cb = make_double2(dd.DCr4, dd.DCi4);
        if (a == 5) ca = make_double2(dd.DPr5, dd.DPi5), cb = make_double2(dd.DCr5, dd.DCi5);
        if (a == 6) ca = make_double2(DP.y, -DP.x), cb = make_double2(DC.y, -DC.x);          // phi0: -i h
    };
    auto G = [&](int q, int r) {
        if (q == r) return make_double2(red[q], 0.0);
        const int k = gram_index(q < r ? q : r, q < r ? r : q);
        return make_double2(red[k], q < r ? red[k + 1] : -red[k + 1]);
    };
    // Re conj(a) g b
    auto re3 = [](double2 a, double2 g, double2 b) {
        const double2 ab = make_double2(a.x * b.x + a.y * b.y, a.x * b.y - a.y * b.x);
        return ab.x * g.x - ab.y * g.y;
    };
    const int a = threadIdx.x / 8, b = threadIdx.x % 8;
    const int lo = a < b ? a : b, hi = a < b ? b : a;  // both triangles alike, bit for bit
    int qa, qb;
    double2 a0, a1, b0, b1;
    coef(lo, qa, a0, a1);
    coef(hi, qb, b0, b1);
    double f = re3(a0, G(qa, qb), b0);
    if (qb == 0) f += re3(a0, G(qa, 1), b1);
    if (qa == 0) f += re3(a1, G(1, qb), b0);
    if (qa == 0 && qb == 0) f += re3(a1, G(1, 1), b1);
    A.fisher[(size_t)e * 64 + threadIdx.x] = 2.0 * f;
    auto proj = [&](int k) {
        int q;
        double2 ca, cb;
        coef(k, q, ca, cb);
        double g = ca.x * red[kPOff + 2 * q] - ca.y * red[kPOff + 2 * q + 1];
        if (q == 0) g += cb.x * red[kPOff + 2] - cb.y * red[kPOff + 3];
        return 2.0 * g;
    };
    if (threadIdx.x < 8) A.grad[(size_t)e * 8 + threadIdx.x] = proj(threadIdx.x);
    // (R|h) - (h|h)/2 = (R - h|h) + (h|h)/2; thread 27 holds (3, 3) = (h|h)
    if (threadIdx.x == 27) A.outL[e] = proj(3) + (A.mode == 1 ? red[kNMain] : f);
}

// Waves per SIMD the register allocation must allow (1 = the compiler's
// choice, at least the two that eight waves per CU need).
#ifndef GH_DERIV_WAVES
#define GH_DERIV_WAVES 1
#endif

// The constants of the workgroup's source and their derivatives on lanes of
// two waves, so the two serial setups overlap.
template <int NTHR>
__device__ __forceinline__ void deriv_setup(const double* p, const DerivArgs& A, UcbConst& sc, UcbDiff& sdd)
{
    if (threadIdx.x == 0) ucb_setup(p, 8, A.T, A.t0, A.L, A.fstar, A.reach, sc);
    if (threadIdx.x == (NTHR >= 128 ? 64 : 0)) ucb_diff_setup(p, A.T, sdd);
    __syncthreads();
}

template <int N>
__global__ __launch_bounds__(fd_threads(N), GH_DERIV_WAVES) void deriv_kernel(DerivArgs A)
{
    using S = FdShape<N, 1>;
    constexpr int P = S::P, NTHR = S::NTHR;
    constexpr int LDS = deriv_sets(N) * kNLink * S::PN;
    constexpr int CH = 16 * (NTHR + 1) <= 2 * LDS ? 16 : 8;
    static_assert(CH * (NTHR + 1) <= 2 * LDS, "the reduction's rows fit the FFT buffer");
    __shared__ double2 lds[LDS];
    __shared__ UcbDiff sdd;
    __shared__ UcbConst sc;
    __shared__ double red[kNSum];
    int e = blockIdx.x;
    if (A.list)
    {
        if (e >= *A.count) return;  // uniform over the workgroup
        e = A.list[e];
    }
    deriv_setup<NTHR>(A.params + (size_t)(A.pidx ? A.pidx[e] : e) * 8, A, sc, sdd);
    // the constants into scalar registers for the passes (the derivative
    // constants stay in LDS, where the scalar copies would spill)
    UcbConst c = sc;
    c.np = 8;
    make_uniform(c);
    double2 u[P][6][3];
    deriv_passes<N, 6>(c, sdd, lds, A, [&](int r, int q, double2 X, double2 Y, double2 Z) {
        u[r][q][0] = X;
        u[r][q][1] = Y;
        u[r][q][2] = Z;
    });
    double acc[kNSum];
#pragma unroll
    for (int k = 0; k < kNSum; k++) acc[k] = 0.0;
    const DerivItem it = deriv_item(A, e);
    if (S::NT >= 64 || threadIdx.x < S::NT)
#pragma unroll
        for (int r = 0; r < P; r++) deriv_bin(c, A, it, P * threadIdx.x + r, u[r], acc);
    deriv_reduce<NTHR, CH>(acc, (double*)lds, red, A.mode == 1);
    deriv_write(c, sdd, A, e, red);
}

// N = 2048, 4096: the same with the TDI values of a source (18 N complex) in
// the workgroup's slice of hs, read back bin by bin for the sums (each
// thread reads only what it wrote).  Grid-striding over the class list.
template <int N>
__global__ __launch_bounds__(fd_threads(N, 1)) void deriv_kernel_long(DerivArgs A, double2* __restrict__ hs)
{
    using S = FdShape<N, 1>;
    constexpr int P = S::P, NTHR = S::NTHR;
    constexpr int LDS = deriv_sets(N) * kNLink * S::PN;
    constexpr int CH = 8;
    static_assert(CH * (NTHR + 1) <= 2 * LDS, "the reduction's rows fit the FFT buffer");
    __shared__ double2 lds[LDS];
    __shared__ UcbDiff sdd;
    __shared__ UcbConst sc;
    __shared__ double red[kNSum];
    double2* H = hs + (size_t)blockIdx.x * deriv_scratch(N);
    const int cnt = A.list ? *A.count : A.nitems;
    const int t = threadIdx.x;
    for (int w = blockIdx.x; w < cnt; w += gridDim.x)
    {
        const int e = A.list ? A.list[w] : w;
        __syncthreads();  // the last item's readers of sc, sdd and red
        deriv_setup<NTHR>(A.params + (size_t)(A.pidx ? A.pidx[e] : e) * 8, A, sc, sdd);
        const UcbConst& c = sc;
        deriv_passes<N, 6>(c, sdd, lds, A, [&](int r, int q, double2 X, double2 Y, double2 Z) {
            double2* o = H + (size_t)(q * 3 * P + r) * NTHR + t;
            o[0] = X;
            o[P * NTHR] = Y;
            o[2 * P * NTHR] = Z;
        });
        double acc[kNSum];
#pragma unroll
        for (int k = 0; k < kNSum; k++) acc[k] = 0.0;
        const DerivItem it = deriv_item(A, e);
#pragma unroll 1
        for (int r = 0; r < P; r++)
        {
            double2 u[6][3];
#pragma unroll
            for (int q = 0; q < 6; q++)
#pragma unroll
                for (int ch = 0; ch < 3; ch++) u[q][ch] = H[(size_t)((q * 3 + ch) * P + r) * NTHR + t];
            deriv_bin(c, A, it, P * t + r, u, acc);
        }
        deriv_reduce<NTHR, CH>(acc, (double*)lds, red, A.mode == 1);
        deriv_write(c, sdd, A, e, red);
    }
}

int launch_derivs_2048(const DerivArgs& A, int grid, double2* hs, hipStream_t s)
{
    if (grid <= 0) return GLASS_HIP_OK;
    if ((!A.list && A.nitems <= 0) || (A.list && !A.count) || !hs)
    {
        set_error("fd derivs: BW 2048 needs a class list or an item count, and scratch");
        return GLASS_HIP_EINVAL;
    }
    deriv_kernel_long<2048><<<grid, fd_threads(2048, 1), 0, s>>>(A, hs);
    GH_CHECK(hipGetLastError());
    return GLASS_HIP_OK;
}

int launch_derivs_4096(const DerivArgs& A, int grid, double2* hs, hipStream_t s)
{
    if (grid <= 0) return GLASS_HIP_OK;
    if ((!A.list && A.nitems <= 0) || (A.list && !A.count) || !hs)
    {
        set_error("fd derivs: BW 4096 needs a class list or an item count, and scratch");
        return GLASS_HIP_EINVAL;
    }
    deriv_kernel_long<4096><<<grid, fd_threads(4096, 1), 0, s>>>(A, hs);
    GH_CHECK(hipGetLastError());
    return GLASS_HIP_OK;
}

int launch_derivs(int N, const DerivArgs& A, int grid, hipStream_t s)
{
    if (grid <= 0) return GLASS_HIP_OK;
    switch (N)
    {
#define GH_D(NN)                                                                   \
    case NN:                                                                       \
        deriv_kernel<NN><<<grid, fd_threads(NN), 0, s>>>(A);       \
        break;
        GH_D(32) GH_D(64) GH_D(128) GH_D(256) GH_D(512) GH_D(1024)
#undef GH_D
        default: set_error("fd derivs: BW=%d unsupported (power of two 32..1024)", N); return GLASS_HIP_EINVAL;
    }
    GH_CHECK(hipGetLastError());
    return GLASS_HIP_OK;
}

}  // namespace glass

using namespace glass;

extern "C" int glass_hip_fd_source_derivs(const glass_hip_orbit* orbit, const char* format, double T, double t0,
                                          int n, const double* d_params, int BW, const int* d_imin, int W,
                                          const double* d_resid, long long resid_stride, const double* d_invC,
                                          long long invC_stride, int mode, double* d_logL, double* d_grad,
                                          double* d_fisher, void* stream)
{
    int fmt = parse_format(format);
    if (fmt < 0)
    {
        set_error("Unsupported data format %s", format ? format : "(null)");
        return GLASS_HIP_EINVAL;
    }
    if (!orbit || n < 0 || !d_params || !d_imin || W < 1 || !d_invC || !d_logL || !d_grad || !d_fisher ||
        (mode != 0 && mode != 1) || resid_stride < 0 || invC_stride < 0)
    {
        set_error("fd_source_derivs: bad arguments");
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
    A.fisher = d_fisher;
    if (BW <= 1024) return launch_derivs(BW, A, n, (hipStream_t)stream);
    if (BW != 2048 && BW != 4096)
    {
        set_error("fd derivs: BW=%d unsupported (power of two 32..4096)", BW);
        return GLASS_HIP_EINVAL;
    }
    // the decimated kernels stride over the items with a scratch slice per
    // workgroup (one workgroup per CU at most), held by the calling thread
    ThreadCtx* cx;
    if ((rc = ctx_get(&cx))) return rc;
    int ncu = 0;
    GH_CHECK(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, cx->device));
    const int grid = n < ncu ? n : ncu;
    if ((rc = cx->dscr.ensure(sizeof(double2) * deriv_scratch(BW) * (size_t)grid))) return rc;
    A.nitems = n;
    double2* hs = (double2*)cx->dscr.p;
    return BW == 2048 ? launch_derivs_2048(A, grid, hs, (hipStream_t)stream)
                      : launch_derivs_4096(A, grid, hs, (hipStream_t)stream);
}
