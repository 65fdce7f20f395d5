// fd_waveform.h -- device building blocks of the frequency-domain UCB
// template: slow series -> LDS FFTs -> fftshift/normalise -> TDI.
// ucb/src/glass_ucb_waveform.c:738-1001; TDI utils/src/glass_lisa.c:458-710.
//
// Five series, not six: every TDI channel is made of differences of link
// series, so the series e_l = d_l - d_23 of the other five links carry them
// all (a sixth of the FFT work, LDS and TDI reads less).  Order: 12, 21, 31,
// 13, 32.
//
// Work split: one workgroup per template of N = P NT bins, NT <= 512
// threads (64 at least).  Thread t evaluates the samples n = t + NT p; a
// P-point decimation-in-frequency step in registers turns them into P series
// of NT points (X[P k + r] = FFT_NT(w_N^{r t} sum_p x_p w_P^{r p})[k]), which
// are transformed in LDS one after the other, the others waiting in
// registers.  Each pass hands one bin per thread to the caller (m = P t + r),
// so one bin's five values are live at a time.  NT = 512 is the length that
// one wave transforms in three radix-8 passes (wave_fft).  At 2048 bins two
// groups of threads share the P samples (FdShape); at 4096 the template is cut
// by its samples instead of its bins (fd_bins_by_sample).
#pragma once
#include "fft_lds.h"
#include "runtime.h"
#include "ucb_common.h"

namespace glass {

constexpr int kNLink = 5;  // series of a template

// Groups of 512 threads per template: two from 2048 bins, where the four or
// eight series of one group would take 233 VGPRs and more (one workgroup of
// eight waves per CU, the vector units 34% busy); each group holds half.
// 23,671 fused evaluations of 2048 bins 2.93 -> 2.81 ms, 379 of 4096 bins 0.39
// -> 0.24 ms (0.17 cut by samples).
constexpr int fd_groups(int N) { return N >= 2048 ? 2 : 1; }

// Series of a template of N bins (P).
constexpr int fd_series(int N) { return N <= 512 ? 1 : N / 512; }

// Workgroup size for a template of N bins.
constexpr int fd_threads(int N, int G) { return N < 64 ? 64 : (N <= 512 ? N : 512 * G); }
constexpr int fd_threads(int N) { return fd_threads(N, fd_groups(N)); }

template <int N, int GROUPS = fd_groups(N)>
struct FdShape
{
    static_assert(N >= 16 && N <= 4096 && (N & (N - 1)) == 0, "16 to 4096 bins");
    static_assert(GROUPS == 1 || (GROUPS == 2 && N >= 2048), "two groups: two or four samples a thread");
    static constexpr int G = GROUPS;
    static constexpr int P = fd_series(N);
    static constexpr int Q = P / G;                   // samples and bins per thread
    static constexpr int NT = N / P;                  // points of an LDS series
    static constexpr int NTHR = fd_threads(N, G);
    static constexpr int PN = wave_fft_stride(NT);
    static constexpr int LDS = G * kNLink * PN;       // double2 elements
    // the template is cut by its samples
    static constexpr bool BYSAMPLE = G == 2 && Q >= 4;
    // the thread's place in its group, and its bin in pass s: P t + the
    // residue, of which the group g of two takes j = g Q/2 .. and j + Q; cut
    // by samples, t + NT (j + P/2) modulo N
    static __device__ __forceinline__ int lane() { return G == 1 ? threadIdx.x : threadIdx.x & 511; }
    static __device__ __forceinline__ int group() { return G == 1 ? 0 : threadIdx.x >> 9; }
    __host__ __device__ static constexpr int residue(int g, int s) { return G == 1 ? s : g * (Q / 2) + s / 2 + Q * (s % 2); }
    __host__ __device__ static constexpr int bin(int t, int g, int s)
    {
        return BYSAMPLE ? t + NT * ((residue(g, s) + P / 2) & (P - 1)) : P * t + residue(g, s);
    }
    static __device__ __forceinline__ int bin(int s) { return bin(lane(), group(), s); }
    // LDS place of thread t's point of a series.  A series of 16 or 32 points
    // has fewer than its workgroup's 64 threads: the others get a place of it
    // too, so that a read without a test stays within the series.
    __host__ __device__ static constexpr int place(int t) { return wave_fft_slot(t & (NT - 1)); }
    // where the series of pass s waits
    static constexpr int slot(int s) { return G == 1 ? s : s / 2 + (Q / 2) * (s % 2); }
};

// Move a value that every lane holds identically into a scalar register.
__device__ inline double uniform(double x)
{
    int lo = __builtin_amdgcn_readfirstlane(__double2loint(x));
    int hi = __builtin_amdgcn_readfirstlane(__double2hiint(x));
    return __hiloint2double(hi, lo);
}

__device__ inline void make_uniform(UcbConst& c)
{
    double* f = &c.T;
    // every double member up to (not including) q
    constexpr int nd = (int)((offsetof(UcbConst, q)) / sizeof(double));
#pragma unroll
    for (int i = 0; i < nd; i++) f[i] = uniform(f[i]);
    c.q = ((long)__builtin_amdgcn_readfirstlane((int)(c.q >> 32)) << 32) |
          (unsigned)__builtin_amdgcn_readfirstlane((int)(c.q & 0xffffffff));
    c.np = __builtin_amdgcn_readfirstlane(c.np);
    c.wide = __builtin_amdgcn_readfirstlane(c.wide);
}

// A pointer that every lane holds identically, in scalar registers.
template <typename T>
__device__ __forceinline__ const T* uniform_ptr(const T* p)
{
    const unsigned long long v = (unsigned long long)p;
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
    return (const T*)(((unsigned long long)hi << 32) | lo);
}

// The constants of one template as the building blocks below take them: a
// callable that returns them.  One that is held (in LDS or registers):
struct HeldConst
{
    const UcbConst& c;
    __device__ const UcbConst& operator()() const { return c; }
};
// ... and one read again by scalar loads at each use (8 parameters).  The
// constants, pointers and masks of a fused kernel are more than the ~100
// scalar registers; held throughout, 370 moves a wave go to spilling them
// into vector lanes.  The pointer passes through an empty asm, so that no
// value of one use stays live until the next.
struct LoadedConst
{
    const UcbConst* p;
    __device__ __forceinline__ UcbConst operator()() const
    {
        auto g = (const __attribute__((address_space(4))) double*)uniform_ptr(p);
        asm volatile("" : "+s"(g));
        UcbConst c;
        double* f = &c.T;
        constexpr int nd = (int)((offsetof(UcbConst, q)) / sizeof(double));
#pragma unroll
        for (int i = 0; i < nd; i++) f[i] = g[i];
        auto w = (const __attribute__((address_space(4))) int*)g;
        c.q = (long)c.qd;
        c.np = 8;
        c.wide = w[offsetof(UcbConst, wide) / sizeof(int)];
        return c;
    }
};

// Per-template constants computed once per workgroup (by thread 0) into
// LDS; every thread reads them from there.  Synchronises the workgroup on
// entry (readers of the previous template are done) and on exit.
__device__ inline const UcbConst& ucb_setup_shared(const double* p, int np, double T, double t0, double L,
                                                   double fstar, OrbitReach reach)
{
    __shared__ UcbConst sc;
    __syncthreads();
    if (threadIdx.x == 0) ucb_setup(p, np, T, t0, L, fstar, reach, sc);
    __syncthreads();
    return sc;
}

// The P-point decimation-in-frequency step of thread t's samples x_p (sample
// t + NT p) in place: x[r] becomes the thread's point of series r.
template <int N, int L>
__device__ __forceinline__ void fd_dif(double2 (&x)[fd_series(N)][L], const double2* __restrict__ tw, int tws, int t)
{
    constexpr int P = fd_series(N);
    double2 w[P > 1 ? P - 1 : 1];
#pragma unroll
    for (int r = 1; r < P; r++) w[r - 1] = tw[(r * t) * tws];
#pragma unroll
    for (int l = 0; l < L; l++)
    {
        double2 v[P], y[P];
#pragma unroll
        for (int p = 0; p < P; p++) v[p] = x[p][l];
        radix_butterfly<P>(v, y);
        x[0][l] = y[0];
#pragma unroll
        for (int r = 1; r < P; r++) x[r][l] = cmul(y[r], w[r - 1]);
    }
}

// The same with the samples of a point on two threads: group g of two holds
// x_{g + 2q}, q < Q.  Each thread transforms its own (A_j from the even samples,
// B_j from the odd, j < Q), hands half of the results to its partner through
// LDS and combines the other half: X_j = A_j + w_P^j B_j, X_{j+Q} = A_j - w_P^j B_j,
// left in the slots of FdShape.  lds: the groups' series rows.  TURN: and times
// w_N^{j t}, the points of the series to transform.
template <int N, bool TURN = true>
__device__ __forceinline__ void fd_dif2(double2 (&x)[fd_series(N) / 2][kNLink], double2* lds,
                                        const double2* __restrict__ tw, int tws)
{
    using S = FdShape<N, 2>;
    constexpr int Q = S::Q, H = Q / 2;
    const bool g = S::group() != 0;
    const int t = S::lane();
    // by value: a choice between array elements would put the array in memory
    auto pick = [](bool c, double2 a, double2 b) { return make_double2(c ? a.x : b.x, c ? a.y : b.y); };
    double2* mine = lds + g * kNLink * S::PN;
    const double2* other = lds + (1 - g) * kNLink * S::PN;
#pragma unroll
    for (int l = 0; l < kNLink; l++)
    {
        double2 v[Q], y[Q];
#pragma unroll
        for (int q = 0; q < Q; q++) v[q] = x[q][l];
        radix_butterfly<Q>(v, y);
#pragma unroll
        for (int q = 0; q < Q; q++) x[q][l] = y[q];
    }
#pragma unroll
    for (int i = 0; i < H; i++)
    {
        if (i) __syncthreads();
#pragma unroll
        for (int l = 0; l < kNLink; l++) mine[l * S::PN + t] = pick(g, x[i][l], x[H + i][l]);
        __syncthreads();
        const int j = g * H + i;
        const double2 wp = tw[j * S::NT * tws];  // w_P^j
        double2 w1, w2;
        if constexpr (TURN) w1 = tw[(j * t) * tws], w2 = tw[((j + Q) * t) * tws];
#pragma unroll
        for (int l = 0; l < kNLink; l++)
        {
            const double2 o = other[l * S::PN + t], h = pick(g, x[H + i][l], x[i][l]);
            const double2 a = pick(g, o, h), b = cmul(pick(g, h, o), wp);
            x[i][l] = make_double2(a.x + b.x, a.y + b.y);
            x[H + i][l] = make_double2(a.x - b.x, a.y - b.y);
            if constexpr (TURN) x[i][l] = cmul(x[i][l], w1), x[H + i][l] = cmul(x[H + i][l], w2);
        }
    }
    __syncthreads();
}

// fd_link_bins (below) cut by the samples: series p is the samples n = P j + p,
// whose transform Y_p enters bin j + NT r (FFT index) as w_N^{p j} w_P^{p r}
// Y_p[j].  Each pass evaluates, transforms and turns one series a group, and the
// groups' P sums come last (fd_dif2's exchange), so a thread's bins are 512
// apart and the lanes of a wave read and write consecutive bins.  Cut by bins, a
// thread's bins are P apart: each pass reads every line of the window, the stored
// template and the weights for 16 of its 128 bytes, eight times 0.8 MB an item,
// past the L2.  4080 evaluations of 4096 bins 2.67 -> 1.42 ms (1.65 with radix-4
// transforms and bins 512 apart), 20,000 9.6 -> 5.9 ms; 300 in one launch 302 ->
// 164 us.
template <int N, bool SOA, typename K, typename Pre, typename F>
__device__ __forceinline__ void fd_bins_by_sample(const K& kget, double2* lds, const double* __restrict__ pos,
                                                  int posstride, const double2* __restrict__ tw, int tws, Pre&& pre,
                                                  F&& f)
{
    using S = FdShape<N>;
    constexpr int P = S::P, Q = S::Q, NT = S::NT, PN = S::PN;
    constexpr int KS = SOA ? N : 1;
    static_assert(S::BYSAMPLE && pos_soa_place(N, P * 5 + 3) == 3 * NT + 5, "positions in the samples' order");
    const int t = S::lane();
    // this thread's place of a series: it alone writes and, transformed, reads it
    double2* own = lds + S::group() * kNLink * PN + S::place(t);
    double2 x[Q][kNLink];
#pragma unroll
    for (int q = 0; q < Q; q++)
#pragma unroll
        for (int l = 0; l < kNLink; l++) x[q][l] = make_double2(0.0, 0.0);
#pragma unroll 1
    for (int q = 0; q < Q; q++)
    {
        const int p = S::group() + S::G * q, n = P * t + p;
        const UcbConst& c = kget();
        ucb_slow_sample_to<KS>(c, ucb_sample_time(c.T, c.t0, n, N),
                               SOA ? pos + pos_soa_place(N, n) : pos + (size_t)n * posstride * 9,
                               [&](int l, double2 v) { own[l * PN] = v; });
        __syncthreads();
        wave_fft<NT, S::G * kNLink, S::NTHR, true>(lds, opaque(tw), P * tws);
        const double2 w = tw[(p * t) * tws];
#pragma unroll
        for (int l = 0; l < kNLink; l++)
        {
#pragma unroll
            for (int i = 0; i + 1 < Q; i++) x[i][l] = x[i + 1][l];
            x[Q - 1][l] = cmul(own[l * PN], w);
        }
    }
    __syncthreads();
    fd_dif2<N, false>(x, lds, tw, tws);
#pragma unroll
    for (int s = 0; s < Q; s++)
    {
        int u = t;  // fresh indices per bin
        asm volatile("" : "+v"(u));
        const int m = S::bin(u, S::group(), s);
        pre(m);
        f(s, m, x[S::slot(s)]);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// ... and cut by the bins.
template <int N, bool SOA, int GROUPS, typename K, typename Pre, typename F>
__device__ __forceinline__ void fd_bins_by_bin(const K& kget, double2* lds, const double* __restrict__ pos,
                                               int posstride, const double2* __restrict__ tw, int tws, Pre&& pre,
                                               F&& f)
{
    using S = FdShape<N, GROUPS>;
    constexpr int P = S::P, Q = S::Q, NT = S::NT, PN = S::PN;
    constexpr int KS = SOA ? N : 1;
    const int t = S::lane();
    const bool on = NT >= 64 || t < NT;
    const int ts = wave_fft_slot(t);
    double2* rows = lds + S::group() * kNLink * PN;
    auto sample = [&](int n, auto&& out) {
        const UcbConst& c = kget();
        ucb_slow_sample_to<KS>(c, ucb_sample_time(c.T, c.t0, n, N), SOA ? pos + n : pos + (size_t)n * posstride * 9,
                               out);
    };
    double2 x[Q][kNLink];
    if constexpr (P == 1)
    {
        if (on) sample(t, [&](int l, double2 v) { rows[l * PN + ts] = v; });
    }
    else
    {
        // the samples shifted in: a loop whose body is one sample, so that
        // one sample's temporaries are live beside the Q results
#pragma unroll
        for (int p = 0; p < Q; p++)
#pragma unroll
            for (int l = 0; l < kNLink; l++) x[p][l] = make_double2(0.0, 0.0);
#pragma unroll 1
        for (int p = 0; p < Q; p++)
            sample(t + NT * (S::group() + S::G * p), [&](int l, double2 v) {
#pragma unroll
                for (int q = 0; q + 1 < Q; q++) x[q][l] = x[q + 1][l];
                x[Q - 1][l] = v;
            });
        if constexpr (S::G == 2)
            fd_dif2<N>(x, lds, tw, tws);
        else
            fd_dif<N, kNLink>(x, tw, tws, t);
#pragma unroll
        for (int l = 0; l < kNLink; l++) rows[l * PN + ts] = x[0][l];
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < Q; s++)
    {
        // fresh indices per pass (as in wave_fft): kept, they fill registers
        int u = t;
        if constexpr (P > 1) asm volatile("" : "+v"(u));
        // bin m = P t + r is FFT index (m + N/2) mod N = P k + r
        const int k = wave_fft_slot((u + NT / 2) & (NT - 1));
        const int m = S::bin(u, S::group(), s);
        if (on) pre(m);
        wave_fft<NT, S::G * kNLink, S::NTHR, (P > 1)>(lds, opaque(tw), P * tws);
        double2 d[kNLink];
#pragma unroll
        for (int l = 0; l < kNLink; l++) d[l] = rows[l * PN + k];
        if (s + 1 < Q)
        {
            __syncthreads();
            // the next series takes the LDS before this bin's work, so it is
            // not held in registers across that work
#pragma unroll
            for (int l = 0; l < kNLink; l++) rows[l * PN + wave_fft_slot(u)] = x[S::slot(s + 1)][l];
        }
        if (on) f(s, m, d);
        if (s + 1 < Q) __syncthreads();
    }
}

// f(s, m, d) for every output bin m = FdShape::bin(s) of this thread: d[l] =
// series l at bin m, FFT_l[(m + N/2) mod N] (glass_ucb_waveform.c:940-962);
// the reference's 1/(2N) is part of fd_tdi's prefactor.  SOA: pos is the
// N-sample structure-of-arrays block (9 rows of N samples, pos_soa_place); else
// the record table read with stride posstride.  tws = entries of tw per N-th root.
// pre(m) is called before the transform of bin m's pass, so that global
// loads the caller issues there are in flight during it.  No barrier after
// the last LDS reads: the caller passes one of its own before anything
// writes lds again.
template <int N, bool SOA, int GROUPS = fd_groups(N), typename K, typename Pre, typename F>
__device__ __forceinline__ void fd_link_bins(const K& kget, double2* lds, const double* __restrict__ pos,
                                             int posstride, const double2* __restrict__ tw, int tws, Pre&& pre, F&& f)
{
    using S = FdShape<N, GROUPS>;
    if constexpr (S::BYSAMPLE)
        fd_bins_by_sample<N, SOA>(kget, lds, pos, posstride, tw, tws, pre, f);
    else
        fd_bins_by_bin<N, SOA, GROUPS>(kget, lds, pos, posstride, tw, tws, pre, f);
}

// exp(-i x) of x = f/f* at template bin m (f = (q + m - N/2)/T,
// glass_lisa.c:664): the template's own value at bin q (ucb_setup) turned by
// the few bins between, a small angle, 14 instructions instead of a full
// sine and cosine per bin (50).  Where N/2 bins are more than 1/64 rad (a
// T below ~1e7 s for long templates) the angle is evaluated directly.  The
// reference steps it with a rotation recurrence (glass_lisa.c:403-415),
// which agrees to ~N ulp.
template <int N>
__device__ __forceinline__ void fd_tdi_phase(const UcbConst& c, int m, double& c1, double& s1)
{
    const double dm = (double)(m - N / 2);
    if (c.tdx * (N / 2) <= 0.015625)
    {
        const double d = dm * c.tdx, z = d * d;
        const double sd = d * fma(z, fma(z, 1.0 / 120.0, -1.0 / 6.0), 1.0);
        const double cd = fma(z, fma(z, fma(z, -1.0 / 720.0, 1.0 / 24.0), -0.5), 1.0);
        c1 = c.ttc * cd - c.tts * sd;
        s1 = c.tts * cd + c.ttc * sd;
    }
    else
        sincos_red((c.qd + dm) * c.invT * c.invfstar, &s1, &c1);
}

// The prefactor P of a channel P (a exp(-ix) + b), a = d_ij - d_ik and b =
// d_ji - d_ki, with the 1/(2N) of the link spectra (a power of two):
//   sangria (glass_lisa.c:645-710): pf [a e^{-2ix} + b e^{-ix}],
//     pf = 4 sqrt(T) (f/f*) sin(f/f*), so P = pf e^{-ix};
//   phase, frequency (:458-643): pf [a e^{-3ix} + b e^{-2ix} - a e^{-ix} - b],
//     pf = sqrt(T) or sqrt(T) 2 f/f*, so P = pf (e^{-2ix} - 1).
template <int N>
__device__ __forceinline__ double2 fd_tdi_prefactor(const UcbConst& c, int m, int fmt, double c1, double s1)
{
    constexpr double inv2N = 1. / (double)(2 * N);
    const double x = (c.qd + (double)(m - N / 2)) * c.tdx;
    if (fmt == TDI_SANGRIA)
    {
        const double pf = x * (4.0 * inv2N * c.sqT) * s1;
        return make_double2(pf * c1, -pf * s1);
    }
    const double pf = -2.0 * inv2N * c.sqT * s1 * (fmt == TDI_PHASE ? 1.0 : 2.0 * x);
    return make_double2(pf * s1, pf * c1);
}

// The channel combinations of the series (kNLink order): aX = d12 - d13, bX
// = d21 - d31, aY = d23 - d21, bY = d32 - d12, aZ = d31 - d32, bZ = d13 - d23.
// TDI of template bin m from its five series values.  out: X, Y, Z, A, E.
// From exp(-ix) and the prefactor P of the bin.
__device__ __forceinline__ void fd_tdi_xyz(double c1, double s1, double2 P, const double2* d, double2& X, double2& Y,
                                           double2& Z)
{
    auto ch = [&](double ax, double ay, double bx, double by) {
        const double vx = fma(ax, c1, fma(ay, s1, bx)), vy = fma(ay, c1, fma(-ax, s1, by));
        return make_double2(vx * P.x - vy * P.y, vx * P.y + vy * P.x);
    };
    X = ch(d[0].x - d[3].x, d[0].y - d[3].y, d[1].x - d[2].x, d[1].y - d[2].y);
    Y = ch(-d[1].x, -d[1].y, d[4].x - d[0].x, d[4].y - d[0].y);
    Z = ch(d[2].x - d[4].x, d[2].y - d[4].y, d[3].x, d[3].y);
}

__device__ __forceinline__ void fd_tdi_channels(double c1, double s1, double2 P, int fmt, const double2* d,
                                                double2* out)
{
    double2 X, Y, Z;
    fd_tdi_xyz(c1, s1, P, d, X, Y, Z);
    double2 A = make_double2((Z.x - X.x) * kSQRT1_2, (Z.y - X.y) * kSQRT1_2);
    double2 E = make_double2((X.x - 2 * Y.x + Z.x) * kINVSQ6, (X.y - 2 * Y.y + Z.y) * kINVSQ6);
    if (fmt == TDI_PHASE)
    {
        A.y = -A.y;
        E.y = -E.y;
    }
    out[0] = X;
    out[1] = Y;
    out[2] = Z;
    out[3] = A;
    out[4] = E;
}

template <int N>
__device__ __forceinline__ void fd_tdi(const UcbConst& c, int m, int fmt, const double2* d, double2* out)
{
    double s1, c1;
    fd_tdi_phase<N>(c, m, c1, s1);
    fd_tdi_channels(c1, s1, fd_tdi_prefactor<N>(c, m, fmt, c1, s1), fmt, d, out);
}

}  // namespace glass
