// fstat.hip -- the F-statistic of the UCB sampler's F-statistic proposal,
// batched over grid cells.
//
// Reference (paths relative to the reference root):
//   get_Fstat_logL                 ucb/src/glass_ucb_fstatistic.c:646-703
//   get_filters (the 4 filters)    ucb/src/glass_ucb_fstatistic.c:231-348
//   get_N, get_M, init_M_matrix    ucb/src/glass_ucb_fstatistic.c:172-517
//   calc_Fstat_logL, calc_a_i      ucb/src/glass_ucb_fstatistic.c:599-644
//   get_F_params                   ucb/src/glass_ucb_fstatistic.c:525-597
//   setup_ / build_fstatistic_proposal  ucb/src/glass_ucb_proposal.c:916-1180
//
// One workgroup per grid cell (f0, fdot, theta, phi): the four filter
// templates A^i (ucb_waveform at amplitude 2, iota = pi/2 and the four
// (psi, phase) pairs) go through the batched template pipeline (slow series
// -> LDS FFTs -> TDI) one after another and stay in registers, one bin per
// thread; then the projections N^i = (s|A^i) and the Gram M^ij = (A^i|A^j)
// for X and for A+E are summed over the workgroup.  Cells are bucketed by
// their filter length N = ucb_bandwidth(f0, fdot, cos theta, A = 1e-22) into
// one kernel per power-of-two class, as the proposal evaluations are.
//
// Vector issue bounds it, and at the usual 64 bins a cell is one wave, so
// what one lane does costs as much as what all do: the constants of a cell
// before the filters, and after them the inverses of its two 4x4 Grams, F =
// N^T M^-1 N / 2 and the maximum-likelihood extrinsic parameters, are kernels
// of one thread per cell.  The filters share their sample (FilterSample).
// 102,400 cells of 64 bins: 1.28 -> 0.53 ms.
//
// The 4x4 inverse is Gauss-Jordan elimination with partial pivoting in
// place of LAPACKE dgetrf/dgetri (utils/src/glass_math.c:501-523); the two
// agree to rounding.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <vector>

#include "../../include/glass_hip_fstat.h"
#include "fd_waveform.h"
#include "reduce.h"
#include "runtime.h"

namespace glass {

int parse_format(const char* format);

namespace {

constexpr int kFsClass = 8;  // filter lengths 16 .. 2048
constexpr int kPosNF = 4096;

struct FstatDev
{
    const double2* X;
    const double2* A;
    const double2* E;
    const double* C00;
    int NFFT, qmin0;
    double T, t0, L, fstar;
    OrbitReach reach;
    int fmt;
    const double* pos;
    const double2* tw;
    // per filter: the factors of the plus and cross tensors as ucb_setup
    // forms them, the phase (0 for the first) with its cosine and sine
    struct Filter
    {
        double DPr, DPi, DCr, DCi, phase, cph, sph;
    } f[4];
};

struct Cells
{
    const double* cell;  // [n][4]: f0, fdot, theta, phi
    double* lx;          // [n] F-statistic of X
    double* lae;         // [n] F-statistic of A, E
    double* fpar;        // [n][4]: A, iota, psi, phase of the A,E fit
    UcbConst* pc;        // [n] template constants of the first filter
    double* sums;        // [n][kFsSum]
    int* cls;            // [n] class (kFsClass: none)
};

// Sums of one cell: N of X and of A, E, then the upper triangles of M.
constexpr int kFsSum = 28;

// Cells that a new plan has work buffers for (constants, sums, class and lists, 692
// bytes a cell).  A call with more grows them; where there is no memory for that it
// evaluates the cells in turns (408,800 cells 2.02 ms at once, 2.12 in four turns).
// With buffers for its whole capacity a plan of 2^20 cells, the Python default,
// held 0.8 GB and took 12 ms to create and close; now 0.2 GB and 1 to 3 ms.
constexpr int kFsTurn = 131072;

// Gauss-Jordan inverse with partial pivoting of a 4x4 matrix (in place)
__host__ __device__ inline void invert4(double m[4][4])
{
#pragma clang fp contract(off)
    double a[4][8];
    for (int i = 0; i < 4; i++)
        for (int j = 0; j < 4; j++)
        {
            a[i][j] = m[i][j];
            a[i][4 + j] = i == j ? 1.0 : 0.0;
        }
    for (int c = 0; c < 4; c++)
    {
        int p = c;
        for (int r = c + 1; r < 4; r++)
            if (fabs(a[r][c]) > fabs(a[p][c])) p = r;
        if (p != c)
            for (int j = 0; j < 8; j++)
            {
                double t = a[c][j];
                a[c][j] = a[p][j];
                a[p][j] = t;
            }
        const double piv = a[c][c];
        for (int j = 0; j < 8; j++) a[c][j] = a[c][j] / piv;
        for (int r = 0; r < 4; r++)
        {
            if (r == c) continue;
            const double f = a[r][c];
            for (int j = 0; j < 8; j++) a[r][j] = a[r][j] - f * a[c][j];
        }
    }
    for (int i = 0; i < 4; i++)
        for (int j = 0; j < 4; j++) m[i][j] = a[i][4 + j];
}

__host__ __device__ inline int sgn(double v) { return v < 0 ? -1 : (v > 0 ? 1 : 0); }

// calc_Fstat_logL for one channel set (the reference's term order)
__host__ __device__ inline double fstat_value(const double M[4][4], const double* N)
{
#pragma clang fp contract(off)
    return 0.5 * (M[0][0] * N[0] * N[0] + 2 * M[0][1] * N[0] * N[1] + 2 * M[0][2] * N[0] * N[2] +
                  2 * M[0][3] * N[0] * N[3] + M[1][1] * N[1] * N[1] + 2 * M[1][2] * N[1] * N[2] +
                  2 * M[1][3] * N[1] * N[3] + M[2][2] * N[2] * N[2] + 2 * M[2][3] * N[2] * N[3] +
                  M[3][3] * N[3] * N[3]);
}

// calc_a_i + get_F_params for the A,E channels
__device__ inline void fstat_params(const double M[4][4], const double* N, double* out)
{
#pragma clang fp contract(off)
    double a[4];
    for (int i = 0; i < 4; i++) a[i] = M[i][0] * N[0] + M[i][1] * N[1] + M[i][2] * N[2] + M[i][3] * N[3];
    const double a1p4 = a[0] + a[3], a2m3 = a[1] - a[2], a1m4 = a[0] - a[3], a2p3 = a[1] + a[2];
    const double s1 = sqrt(a1p4 * a1p4 + a2m3 * a2m3), s2 = sqrt(a1m4 * a1m4 + a2p3 * a2p3);
    const double Ap = s1 + s2, Ac = s1 - s2;
    double psi = atan2(Ap * a[3] - Ac * a[0], -(Ac * a[1] + Ap * a[2]));
    psi *= 0.5;
    const double c = (double)sgn(sin(2.0 * psi));
    const double r = sqrt(Ap * Ap - Ac * Ac);
    out[0] = 0.5 * (Ap + r);
    out[1] = acos(-Ac / (Ap + r));
    out[2] = psi;
    out[3] = atan2(c * (Ap * a[3] - Ac * a[0]), -c * (Ac * a[2] + Ap * a[1]));
}

// filter length of each cell and the per-class lists.  Slots are reserved
// per block (an LDS histogram, then one global atomic per class per
// block): the cells of a segment mostly share one filter length, and one
// global atomic per cell on that class's counter serialises the launch.
__global__ __launch_bounds__(256) void fstat_align_kernel(int n, FstatDev D,
                                                          Cells C, int* __restrict__ cls, int* __restrict__ list,
                                                          int cap, int* __restrict__ err)
{
    __shared__ int hist[kFsClass + 1], base[kFsClass + 1];
    if (threadIdx.x <= kFsClass) hist[threadIdx.x] = 0;
    __syncthreads();
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    int k = -1, slot = 0;
    if (e < n)
    {
        const double f0 = C.cell[(size_t)e * 4], fdot = C.cell[(size_t)e * 4 + 1];
        const double theta = C.cell[(size_t)e * 4 + 2], phi = C.cell[(size_t)e * 4 + 3];
        const int N = ucb_bandwidth(D.L, D.fstar, f0, fdot, cos(theta), 1.e-22, D.T, D.NFFT);
        k = 31 - __clz(N) - 4;  // log2(N) - 4
        if (k < 0 || k >= kFsClass || (N & (N - 1))) k = kFsClass;
        C.cls[e] = k;
        // amplitude and polarisation come with each filter
        const double p[8] = {f0 * D.T, cos(theta), phi, 0.0, 0.0, 0.0, D.f[0].phase, fdot * (D.T * D.T)};
        ucb_setup(p, 8, D.T, D.t0, D.L, D.fstar, D.reach, C.pc[e]);
        slot = atomicAdd(&hist[k], 1);
    }
    __syncthreads();
    if (threadIdx.x < kFsClass && hist[threadIdx.x]) base[threadIdx.x] = atomicAdd(&cls[threadIdx.x], hist[threadIdx.x]);
    if (threadIdx.x == kFsClass && hist[kFsClass]) atomicAdd(err, hist[kFsClass]);
    __syncthreads();
    if (k >= 0 && k < kFsClass) list[(size_t)k * cap + base[k] + slot] = e;
}

// One slow sample of all four filters.  They differ in the polarisation
// tensor's factors and in the constant phase subtracted in arg2, whose rounding
// (~1e-10 rad at 3 mHz and 2 yr, independent in each filter) the results keep:
// with the quadrature filters as exact quarter turns of the others F moves by
// up to 1e-9.  arg2 of filter k is that of the first less phase_k plus a
// delta, so its factor exp(i arg2) is the first's turned by phase_k times 1 +
// i delta (delta^2 < 1e-18).  What the filters share is formed once: ~350
// instructions, and 90 for each filter instead of 400.
struct FilterSample
{
    double2 B[3][2];      // spacecraft i, link h: amplitude exp(i arg2) S exp(-i arg1) (the first's arg2)
    double dp[3], dc[3];  // arms 12, 13, 23
    double delta[3][3];   // filter 1..3, spacecraft

    __device__ __forceinline__ FilterSample(const UcbConst& c, const FstatDev& D, double t,
                                            const double* __restrict__ pos)
    {
        const double x[3] = {pos[0], pos[1], pos[2]}, y[3] = {pos[3], pos[4], pos[5]}, z[3] = {pos[6], pos[7], pos[8]};
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
                // as ucb_slow_sample_to forms it for each filter
#pragma clang fp contract(off)
                const double kdotx = div_by_recip(x[i] * c.k[0] + y[i] * c.k[1] + z[i] * c.k[2], kCLIGHT, kInvCLIGHT);
                xi = t - kdotx;
                const double w = c.pi2f0 * xi, chirp = c.pidfdt * xi * xi;
                a2[i] = w - c.phi0 - dft;
                a2[i] += chirp;
#pragma unroll
                for (int k = 1; k < 4; k++)
                {
                    double a = w - D.f[k].phase - dft;
                    a += chirp;
                    delta[k - 1][i] = (a - a2[i]) + D.f[k].phase;
                }
            }
            hf[i] = fma(c.dfh, xi, c.f0h);
            ae[i] = fma(c.aevq, xi, 0.25);
        }
        double kr[3];
#pragma unroll
        for (int m = 0; m < 3; m++)
        {
            const int i0 = m < 2 ? 0 : 1, i1 = m == 0 ? 1 : 2;
            const double r0 = x[i1] - x[i0], r1 = y[i1] - y[i0], r2 = z[i1] - z[i0];
            const double ru = r0 * c.ua[0] + r1 * c.ua[1] + r2 * c.ua[2];
            const double rv = r0 * c.va[0] + r1 * c.va[1];
            kr[m] = r0 * c.ka[0] + r1 * c.ka[1] + r2 * c.ka[2];
            dp[m] = rv * rv - ru * ru;
            dc[m] = 2.0 * ru * rv;
        }
        __builtin_amdgcn_sched_barrier(0);
        double sn[3], cs[3];
        unsigned fl[3];
        sincos_half<3>(a2, sn, cs, fl);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 3; i++)
        {
            const double a = flip_sign(ae[i], fl[i]), wr = a * cs[i], wi = a * sn[i];
            const double ka = i == 0 ? kr[0] : (i == 1 ? -kr[0] : -kr[1]);
            const double kb = i == 0 ? kr[1] : (i == 1 ? kr[2] : -kr[2]);
            const double arg[2] = {fma(hf[i], ka, hf[i]), fma(hf[i], kb, hf[i])};
            double fr[2], fi[2];
            sinc_phase<2>(arg, c.wide, fr, fi);
#pragma unroll
            for (int h = 0; h < 2; h++) B[i][h] = make_double2(wr * fr[h] - wi * fi[h], wr * fi[h] + wi * fr[h]);
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    // out(l, value) of filter k's five series, as ucb_slow_sample_to
    template <typename Out>
    __device__ __forceinline__ void filter(const FstatDev::Filter& f, int k, Out&& out) const
    {
        double2 T1[3];
#pragma unroll
        for (int m = 0; m < 3; m++)
            T1[m] = make_double2(dp[m] * f.DPr + dc[m] * f.DCr, dp[m] * f.DPi + dc[m] * f.DCi);
        double2 d23;
#pragma unroll
        for (int q = 0; q < 3; q++)
        {
            const int i = q == 0 ? 1 : (q == 1 ? 0 : 2);
            double2 r = make_double2(1.0, 0.0);
            if (k > 0)
            {
                const double e = delta[k > 0 ? k - 1 : 0][i];
                r = make_double2(fma(e, f.sph, f.cph), fma(e, f.cph, -f.sph));
            }
            double2 d[2];
#pragma unroll
            for (int h = 0; h < 2; h++)
            {
                const int m = i == 0 ? h : (i == 1 ? 2 * h : 1 + h);
                const double2 b = k > 0 ? cmul(B[i][h], r) : B[i][h];
                d[h] = cmul(T1[m], b);
            }
            if (i == 1) d23 = d[1];
            out(i, make_double2(d[0].x - d23.x, d[0].y - d23.y));
            if (i != 1) out(i == 0 ? 3 : 4, make_double2(d[1].x - d23.x, d[1].y - d23.y));
        }
    }
};

// The constants of a cell's filter: the first's with its own amplitude and phase.
struct FilterConst
{
    LoadedConst base;
    const FstatDev& D;
    int k;
    __device__ __forceinline__ UcbConst operator()() const
    {
        UcbConst c = base();
        const FstatDev::Filter& f = D.f[k];
        c.DPr = f.DPr;
        c.DPi = f.DPi;
        c.DCr = f.DCr;
        c.DCi = f.DCi;
        c.phi0 = f.phase;
        return c;
    }
};

// Terms of one bin from the filters' X, A, E, with the weight 1/c.
__device__ __forceinline__ void fstat_bin(const FstatDev& D, long kb, const double2 (&h)[4][3], double (&v)[kFsSum])
{
    const double w = 1.0 / D.C00[kb];
    const double2 dX = D.X[kb], dA = D.A[kb], dE = D.E[kb];
    auto re = [](double2 a, double2 b) { return a.x * b.x + a.y * b.y; };
    int t = 8;
#pragma unroll
    for (int i = 0; i < 4; i++)
    {
        double2 u[3];
#pragma unroll
        for (int ch = 0; ch < 3; ch++) u[ch] = make_double2(w * h[i][ch].x, w * h[i][ch].y);
        v[i] += re(dX, u[0]);
        v[4 + i] += re(dA, u[1]) + re(dE, u[2]);
#pragma unroll
        for (int j = i; j < 4; j++, t++)
        {
            v[t] += 4.0 * re(u[0], h[j][0]);
            v[10 + t] += 4.0 * (re(u[1], h[j][1]) + re(u[2], h[j][2]));
        }
    }
}

// Three waves per SIMD up to 512 bins: the compiler's choice is a few vector
// registers above the 168 that allows.
template <int N>
__global__ __launch_bounds__(fd_threads(N)) __attribute__((amdgpu_waves_per_eu(N <= 512 ? 3 : 1, 8))) void fstat_kernel(
    const int* __restrict__ list, const int* __restrict__ count, FstatDev D, Cells C)
{
    using S = FdShape<N>;
    constexpr int CH = 8, ROWS = CH * (S::NTHR + 1) / 2 + 1;
    __shared__ double2 lds[S::LDS > ROWS ? S::LDS : ROWS];
    if ((int)blockIdx.x >= *count) return;
    const int e = list[blockIdx.x];
    const LoadedConst k{C.pc + e};
    const long qo = (long)(C.cell[(size_t)e * 4] * D.T) - D.qmin0 - N / 2;  // segment bin of template bin 0
    double v[kFsSum];
#pragma unroll
    for (int i = 0; i < kFsSum; i++) v[i] = 0.0;
    if constexpr (S::P == 1)
    {
        const int t = S::lane();
        const bool on = t < N;
        const int ts = wave_fft_slot(t), tb = wave_fft_slot((t + N / 2) & (N - 1));
        const int n = on ? t : 0;
        const FilterSample s(k(), D, ucb_sample_time(D.T, D.t0, n, N), D.pos + (size_t)n * (kPosNF / N) * 9);
        double2 h[4][3], P;
        double c1, s1;
        {
            const UcbConst& c = k();
            fd_tdi_phase<N>(c, t, c1, s1);
            P = fd_tdi_prefactor<N>(c, t, D.fmt, c1, s1);
        }
#pragma unroll
        for (int f = 0; f < 4; f++)
        {
            if (f) __syncthreads();  // the last filter's LDS reads
            if (on) s.filter(D.f[f], f, [&](int l, double2 x) { lds[l * S::PN + ts] = x; });
            __syncthreads();
            wave_fft<N, kNLink, S::NTHR, true>(lds, opaque(D.tw), kTwN / N);
            double2 d[kNLink], o[5];
#pragma unroll
            for (int l = 0; l < kNLink; l++) d[l] = lds[l * S::PN + tb];
            fd_tdi_channels(c1, s1, P, D.fmt, d, o);
            h[f][0] = o[0];
            h[f][1] = o[3];
            h[f][2] = o[4];
        }
        const long kb = qo + t;
        if (on && kb > 0 && kb < D.NFFT) fstat_bin(D, kb, h, v);
    }
    else
    {
        double2 h[S::Q][4][3];
#pragma unroll
        for (int f = 0; f < 4; f++)
        {
            if (f) __syncthreads();  // the last filter's LDS reads
            fd_link_bins<N, false>(
                FilterConst{k, D, f}, lds, D.pos, kPosNF / N, D.tw, kTwN / N, [](int) {},
                [&](int s, int m, const double2* dl) {
                    double2 o[5];
                    fd_tdi<N>(k(), m, D.fmt, dl, o);
                    h[s][f][0] = o[0];
                    h[s][f][1] = o[3];
                    h[s][f][2] = o[4];
                });
        }
#pragma unroll
        for (int s = 0; s < S::Q; s++)
        {
            const long kb = qo + S::bin(s);
            if (kb > 0 && kb < D.NFFT) fstat_bin(D, kb, h[s], v);
        }
    }
    __syncthreads();
    block_sum_rows<S::NTHR, CH, kFsSum>(v, (double*)lds, C.sums + (size_t)e * kFsSum);
}

// F-statistics and extrinsic parameters of the cells, one thread each; cells
// no class holds get NaN.
__global__ __launch_bounds__(64) void fstat_fit_kernel(int n, Cells C)
{
    const int e = blockIdx.x * 64 + threadIdx.x;
    if (e >= n) return;
    if (C.cls[e] >= kFsClass)
    {
        C.lx[e] = C.lae[e] = NAN;
        for (int k = 0; k < 4; k++) C.fpar[(size_t)e * 4 + k] = NAN;
        return;
    }
    const double* v = C.sums + (size_t)e * kFsSum;
    double nx[4], nae[4], MX[4][4], MA[4][4];
#pragma unroll
    for (int i = 0; i < 4; i++)
    {
        nx[i] = 4.0 * v[i];
        nae[i] = 4.0 * v[4 + i];
    }
    int t = 8;
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = i; j < 4; j++, t++)
        {
            MX[i][j] = MX[j][i] = v[t];
            MA[i][j] = MA[j][i] = v[10 + t];
        }
    invert4(MX);
    C.lx[e] = fstat_value(MX, nx);
    invert4(MA);
    C.lae[e] = fstat_value(MA, nae);
    fstat_params(MA, nae, C.fpar + (size_t)e * 4);
}

}  // namespace

}  // namespace glass

using namespace glass;

struct glass_hip_fstat
{
    int device = 0;
    FstatDev D{};
    int cap = 0, turn = 0;  // cells a call, and at a time
    std::vector<void*> allocs;
    double* cells = nullptr;
    double *lx = nullptr, *lae = nullptr, *fpar = nullptr;
    int *cls = nullptr, *list = nullptr, *kcls = nullptr;
    // per cell constants, sums and class (Cells) and the class lists of turn
    // cells, one allocation
    char* work = nullptr;
    UcbConst* pc = nullptr;
    double* sums = nullptr;
};

template <typename T>
static int falloc(glass_hip_fstat* F, T** p, size_t n)
{
    void* q = nullptr;
    if (hipMalloc(&q, sizeof(T) * (n ? n : 1)) != hipSuccess)
    {
        set_error("fstat: hipMalloc of %zu bytes failed", sizeof(T) * (n ? n : 1));
        return GLASS_HIP_ERUNTIME;
    }
    F->allocs.push_back(q);
    *p = (T*)q;
    return GLASS_HIP_OK;
}

// Work buffers for n cells in place of the ones the plan has, which stay if there
// is no memory for them.
static bool work_buffers(glass_hip_fstat* F, int n)
{
    const size_t c = n;
    char* w = nullptr;
    if (hipMalloc(&w, c * (sizeof(UcbConst) + sizeof(double) * kFsSum + sizeof(int) * (1 + kFsClass))) != hipSuccess)
    {
        (void)hipGetLastError();
        return false;
    }
    if (F->work)
    {
        (void)hipDeviceSynchronize();  // an earlier call's kernels use them
        (void)hipFree(F->work);
    }
    F->work = w;
    F->turn = n;
    F->pc = (UcbConst*)w;
    F->sums = (double*)(F->pc + c);
    F->kcls = (int*)(F->sums + kFsSum * c);
    F->list = F->kcls + c;
    return true;
}

extern "C" int glass_hip_fstat_destroy(glass_hip_fstat* F)
{
    if (!F) return GLASS_HIP_OK;
    (void)hipSetDevice(F->device);
    (void)hipDeviceSynchronize();
    for (void* p : F->allocs) (void)hipFree(p);
    if (F->work) (void)hipFree(F->work);
    delete F;
    return GLASS_HIP_OK;
}

extern "C" int glass_hip_fstat_create(glass_hip_fstat** out, const glass_hip_orbit* orbit, const char* format,
                                      double T, double t0, int NFFT, int qmin0, const double* X, const double* A,
                                      const double* E, const double* C00, int max_cells, void* stream)
{
    if (!out || !orbit || !format || NFFT <= 0 || !X || !A || !E || !C00 || max_cells <= 0 || !(T > 0))
    {
        set_error("fstat_create: bad arguments");
        return GLASS_HIP_EINVAL;
    }
    const int fmt = parse_format(format);
    if (fmt < 0)
    {
        set_error("fstat_create: unsupported format '%s'", format);
        return GLASS_HIP_EINVAL;
    }
    *out = nullptr;
    auto* F = new glass_hip_fstat();
    GH_CHECK(hipGetDevice(&F->device));
    hipStream_t s = (hipStream_t)stream;
    FstatDev& D = F->D;
    D.NFFT = NFFT;
    D.qmin0 = qmin0;
    D.T = T;
    D.t0 = t0;
    D.L = orbit->L;
    D.fstar = orbit->fstar;
    D.reach = analytic_reach(orbit->L, orbit->fstar, orbit->R, T, t0);
    D.fmt = fmt;
    // the four filters of get_filters: amplitude 2, iota = pi/2 and
    // (psi, phase) = (0, 0), (pi/4, pi), (0, 3 pi/2), (pi/4, pi/2), mapped
    // to the waveform's ln A and cos iota on the host as the reference does
    const double psi[4] = {0.0, M_PI_4, 0.0, M_PI_4}, ph[4] = {0.0, M_PI, 3.0 * M_PI_2, M_PI_2};
    for (int i = 0; i < 4; i++)
    {
        const double p[8] = {1.0, 0.0, 0.0, log(2.0), cos(M_PI_2), psi[i], ph[i], 0.0};
        UcbConst c;
        ucb_setup(p, 8, T, t0, orbit->L, orbit->fstar, D.reach, c);
        D.f[i] = {c.DPr, c.DPi, c.DCr, c.DCi, ph[i], cos(ph[i]), sin(ph[i])};
    }
    F->cap = max_cells;
    const size_t nb = sizeof(double) * 2 * (size_t)NFFT;
    double *dX = nullptr, *dA = nullptr, *dE = nullptr, *dC = nullptr;
    int rc;
    if ((rc = falloc(F, &dX, 2 * (size_t)NFFT)) || (rc = falloc(F, &dA, 2 * (size_t)NFFT)) ||
        (rc = falloc(F, &dE, 2 * (size_t)NFFT)) || (rc = falloc(F, &dC, NFFT)) ||
        (rc = falloc(F, &F->cells, 4 * (size_t)max_cells)) || (rc = falloc(F, &F->lx, max_cells)) ||
        (rc = falloc(F, &F->lae, max_cells)) || (rc = falloc(F, &F->fpar, 4 * (size_t)max_cells)) ||
        (rc = falloc(F, &F->cls, kFsClass + 1)))
    {
        glass_hip_fstat_destroy(F);
        return rc;
    }
    if (!work_buffers(F, max_cells < kFsTurn ? max_cells : kFsTurn))
    {
        set_error("fstat: no memory for the work buffers of %d cells", max_cells < kFsTurn ? max_cells : kFsTurn);
        glass_hip_fstat_destroy(F);
        return GLASS_HIP_ERUNTIME;
    }
    const double* pos = nullptr;
    const double2* tw = nullptr;
    if ((rc = positions(*orbit, T, t0, kPosNF, &pos)) || (rc = twiddles(&tw)))
    {
        glass_hip_fstat_destroy(F);
        return rc;
    }
    D.pos = pos;
    D.tw = tw;
    D.X = (const double2*)dX;
    D.A = (const double2*)dA;
    D.E = (const double2*)dE;
    D.C00 = dC;
    if (hipMemcpyAsync(dX, X, nb, hipMemcpyHostToDevice, s) || hipMemcpyAsync(dA, A, nb, hipMemcpyHostToDevice, s) ||
        hipMemcpyAsync(dE, E, nb, hipMemcpyHostToDevice, s) ||
        hipMemcpyAsync(dC, C00, sizeof(double) * NFFT, hipMemcpyHostToDevice, s) || hipStreamSynchronize(s))
    {
        set_error("fstat_create: upload failed");
        glass_hip_fstat_destroy(F);
        return GLASS_HIP_ERUNTIME;
    }
    *out = F;
    return GLASS_HIP_OK;
}

__global__ void fs_zero_kernel(int* p, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

// n <= F->turn cells; first: the count of cells without a class starts at zero.
static int fstat_turn(glass_hip_fstat* F, int n, const double* cells, double* lx, double* lae, double* fpar, bool first,
                      hipStream_t s)
{
    fs_zero_kernel<<<1, 64, 0, s>>>(F->cls, first ? kFsClass + 1 : kFsClass);
    const Cells C{cells, lx, lae, fpar, F->pc, F->sums, F->kcls};
    fstat_align_kernel<<<(n + 255) / 256, 256, 0, s>>>(n, F->D, C, F->cls, F->list, F->turn, F->cls + kFsClass);
    // the class counts decide the grids: only non-empty classes launch, one
    // workgroup per cell (an empty class's full grid of immediately
    // exiting workgroups costs 80-160 us)
    int cnt[kFsClass + 1];
    GH_CHECK(hipMemcpyAsync(cnt, F->cls, sizeof(cnt), hipMemcpyDeviceToHost, s));
    GH_CHECK(hipStreamSynchronize(s));
#define FS_L(kk, NN)                                                                                        \
    if (cnt[kk] > 0)                                                                                        \
        fstat_kernel<NN><<<cnt[kk], fd_threads(NN), 0, s>>>(F->list + (size_t)kk * F->turn, F->cls + kk,    \
                                                            F->D, C);
    FS_L(0, 16) FS_L(1, 32) FS_L(2, 64) FS_L(3, 128) FS_L(4, 256) FS_L(5, 512) FS_L(6, 1024) FS_L(7, 2048)
#undef FS_L
    fstat_fit_kernel<<<(n + 63) / 64, 64, 0, s>>>(n, C);
    GH_CHECK(hipGetLastError());
    return GLASS_HIP_OK;
}

static int fstat_launch(glass_hip_fstat* F, int n, const double* cells, double* lx, double* lae, double* fpar,
                        hipStream_t s)
{
    if (n > F->turn) work_buffers(F, n);
    for (int o = 0; o < n; o += F->turn)
        if (int rc = fstat_turn(F, n - o < F->turn ? n - o : F->turn, cells + 4 * (size_t)o, lx + o, lae + o,
                                fpar + 4 * (size_t)o, o == 0, s))
            return rc;
    return GLASS_HIP_OK;
}

extern "C" int glass_hip_fstat_eval(glass_hip_fstat* F, int n, const double* d_cells, double* d_logL_X,
                                    double* d_logL_AE, double* d_Fparams, void* stream)
{
    if (!F || n < 0 || n > F->cap || (n && (!d_cells || !d_logL_X || !d_logL_AE || !d_Fparams)))
    {
        set_error("fstat_eval: bad arguments (n %d, capacity %d)", n, F ? F->cap : 0);
        return GLASS_HIP_EINVAL;
    }
    if (n == 0) return GLASS_HIP_OK;
    GH_CHECK(hipSetDevice(F->device));
    return fstat_launch(F, n, d_cells, d_logL_X, d_logL_AE, d_Fparams, (hipStream_t)stream);
}

// the fdot of a chirp mass, ucb_fdot (ucb/src/glass_ucb_waveform.c:307-314)
static double ucb_fdot_host(double Mc, double f0)
{
    const double TSUN = 4.92569043916e-6;
    double M = Mc * TSUN;
    double Q = 19.2;
    return Q * pow(pow(M_PI, 8) * pow(M, 5) * pow(f0, 11), 1. / 3.);
}

static int eval_host_cells(glass_hip_fstat* F, const std::vector<double>& cells, std::vector<double>& lae,
                           hipStream_t s)
{
    const int n = (int)(cells.size() / 4);
    lae.assign(n, 0.0);
    for (int o = 0; o < n; o += F->cap)
    {
        const int m = std::min(F->cap, n - o);
        GH_CHECK(hipMemcpyAsync(F->cells, cells.data() + (size_t)o * 4, sizeof(double) * 4 * m,
                                hipMemcpyHostToDevice, s));
        if (int rc = fstat_launch(F, m, F->cells, F->lx, F->lae, F->fpar, s)) return rc;
        GH_CHECK(hipMemcpyAsync(lae.data() + o, F->lae, sizeof(double) * m, hipMemcpyDeviceToHost, s));
        int err = 0;
        GH_CHECK(hipMemcpyAsync(&err, F->cls + kFsClass, sizeof(int), hipMemcpyDeviceToHost, s));
        GH_CHECK(hipStreamSynchronize(s));
        if (err)
        {
            set_error("fstat: %d cells with a filter length outside 16..2048", err);
            return GLASS_HIP_EINVAL;
        }
    }
    return GLASS_HIP_OK;
}

extern "C" int glass_hip_fstat_proposal(glass_hip_fstat* F, double fmin, double fmax, int n_theta, int n_phi,
                                        double* tensor, int* n_f_out, double* d_f_out, double* norm_out,
                                        double* maxp_out, void* stream)
{
    if (!F || !(fmax > fmin) || n_theta <= 0 || n_phi <= 0)
    {
        set_error("fstat_proposal: bad arguments");
        return GLASS_HIP_EINVAL;
    }
    GH_CHECK(hipSetDevice(F->device));
    hipStream_t s = (hipStream_t)stream;
    const double T = F->D.T;
    // setup_fstatistic_proposal (ucb/src/glass_ucb_proposal.c:928-936)
    const int n_f = (int)((fmax - fmin) * T);
    if (n_f <= 0)
    {
        set_error("fstat_proposal: empty band");
        return GLASS_HIP_EINVAL;
    }
    const double d_f = (int)((fmax - fmin) * T) / (double)n_f / T;
    const double d_theta = 2. / (double)n_theta;
    const double d_phi = 6.283185307179586 / (double)n_phi;
    if (n_f_out) *n_f_out = n_f;
    if (d_f_out) *d_f_out = d_f;
    if (!tensor) return GLASS_HIP_OK;
    // build_fstatistic_proposal (:1086-1180): every cell at fdot = 0, then
    // for cells with logL_AE > 1 the chirp-mass scan of fdot
    const size_t ncell = (size_t)n_f * n_theta * n_phi;
    std::vector<double> cells(4 * ncell);
    for (int i = 0; i < n_f; i++)
    {
        double f = fmin + i * d_f;
        f += d_f / 2;
        for (int j = 0; j < n_theta; j++)
            for (int k = 0; k < n_phi; k++)
            {
                const size_t c = ((size_t)i * n_theta + j) * n_phi + k;
                cells[4 * c] = f;
                cells[4 * c + 1] = 0.0;
                cells[4 * c + 2] = acos((-1. + (double)j * d_theta + d_theta / 2));
                cells[4 * c + 3] = (double)k * d_phi + d_phi / 2;
            }
    }
    std::vector<double> l0;
    if (int rc = eval_host_cells(F, cells, l0, s)) return rc;
    const int n_fdot = 10;
    const double d_fdot = (1.1 - 0.1) / n_fdot;
    std::vector<size_t> loud;
    for (size_t c = 0; c < ncell; c++)
        if (l0[c] > 1) loud.push_back(c);
    std::vector<double> cells2(4 * loud.size() * n_fdot);
    for (size_t u = 0; u < loud.size(); u++)
        for (int nn = 0; nn < n_fdot; nn++)
        {
            const double* src = &cells[4 * loud[u]];
            double* dst = &cells2[4 * (u * n_fdot + nn)];
            dst[0] = src[0];
            dst[1] = ucb_fdot_host(0.1 + nn * d_fdot, src[0]);
            dst[2] = src[2];
            dst[3] = src[3];
        }
    std::vector<double> l1;
    if (!loud.empty())
        if (int rc = eval_host_cells(F, cells2, l1, s)) return rc;
    for (size_t c = 0; c < ncell; c++) tensor[c] = l0[c] * l0[c];
    for (size_t u = 0; u < loud.size(); u++)
    {
        double lmax = l0[loud[u]];
        for (int nn = 0; nn < n_fdot; nn++)
        {
            const double v = l1[u * n_fdot + nn];
            if (v > lmax) lmax = v;
            if (v < 1) break;
        }
        tensor[loud[u]] = lmax * lmax;
    }
    double norm = 0.0;
    for (size_t c = 0; c < ncell; c++) norm += tensor[c];
    norm = (n_f * n_theta * n_phi) / norm;
    double maxp = -1.e60;
    for (size_t c = 0; c < ncell; c++)
    {
        tensor[c] *= norm;
        if (tensor[c] > maxp) maxp = tensor[c];
    }
    if (norm_out) *norm_out = norm;
    if (maxp_out) *maxp_out = maxp;
    return GLASS_HIP_OK;
}

extern "C" int glass_hip_get_Fstat_logL(const glass_hip_orbit* orbit, const char* format, double T, double t0,
                                        int NFFT, int qmin0, const double* X, const double* A, const double* E,
                                        const double* C00, double f0, double fdot, double theta, double phi,
                                        double* logL_X, double* logL_AE, double* Fparams)
{
    if (!logL_X || !logL_AE || !Fparams)
    {
        set_error("get_Fstat_logL: null output");
        return GLASS_HIP_EINVAL;
    }
    ThreadCtx* cx;
    int rc;
    if ((rc = ctx_get(&cx))) return rc;
    glass_hip_fstat* F = nullptr;
    if ((rc = glass_hip_fstat_create(&F, orbit, format, T, t0, NFFT, qmin0, X, A, E, C00, 1, cx->stream)))
        return rc;
    const double cell[4] = {f0, fdot, theta, phi};
    double res[6];
    if (hipMemcpyAsync(F->cells, cell, sizeof(cell), hipMemcpyHostToDevice, cx->stream) != hipSuccess)
        rc = GLASS_HIP_ERUNTIME;
    if (!rc) rc = fstat_launch(F, 1, F->cells, F->lx, F->lae, F->fpar, cx->stream);
    int err = 0;
    if (!rc && (hipMemcpyAsync(res, F->lx, sizeof(double), hipMemcpyDeviceToHost, cx->stream) ||
                hipMemcpyAsync(res + 1, F->lae, sizeof(double), hipMemcpyDeviceToHost, cx->stream) ||
                hipMemcpyAsync(res + 2, F->fpar, sizeof(double) * 4, hipMemcpyDeviceToHost, cx->stream) ||
                hipMemcpyAsync(&err, F->cls + kFsClass, sizeof(int), hipMemcpyDeviceToHost, cx->stream) ||
                hipStreamSynchronize(cx->stream)))
    {
        set_error("get_Fstat_logL: kernel or copy failed");
        rc = GLASS_HIP_ERUNTIME;
    }
    glass_hip_fstat_destroy(F);
    if (rc) return rc;
    if (err)
    {
        set_error("get_Fstat_logL: filter length outside 16..2048");
        return GLASS_HIP_EINVAL;
    }
    *logL_X = res[0];
    *logL_AE = res[1];
    for (int i = 0; i < 4; i++) Fparams[i] = res[2 + i];
    return GLASS_HIP_OK;
}
