// wdm_ucb.hip -- galactic-binary templates in the WDM wavelet domain on
// gfx950: ucb_waveform_wavelet (ucb/src/glass_ucb_waveform.c:1061-1240),
// wavelet_nwip-based inner products, snr_wavelet and the wavelet
// likelihood, as drop-ins and as a batched device API.
//
// Layout of the computation:
//  hdr_kernel       : one thread per template, its header (layers, heterodyne).
//  K1 resp_kernel   : one workgroup per template, on the Norb orbit knots --
//                     barycentre amplitude and phase splines, phase at
//                     spacecraft 1, the 24 delayed one-arm terms of X,Y,Z
//                     (LISA_spline_response), their amplitude/phase
//                     (extract_amplitude_and_phase, unwrap_phase) and the six
//                     TDI splines.
//  K2               : the heterodyned series at NT*(L+1) samples, a packed
//                     real FFT (X+iY in one complex FFT, Z as half-length),
//                     per layer the Meyer-windowed band and an inverse FFT of
//                     NT, the pixel list, then the inner products against data
//                     and invC.  NT of 256 and 512: layer_kernel, one workgroup
//                     per template, from LDS.  NT of 1024 to 4096: series_,
//                     fft_, band_ and sum_kernel_big, several workgroups per
//                     template, through a global slice.  Forced layer counts:
//                     layer_kernel_big, ping-pong transforms through L2.
// Everything that depends only on the orbit and the time grids (knots,
// spline x-terms, spacecraft geometry at the knots, spacecraft 1 at the
// downsampled times, interval indices) is tabulated once on the host with
// the reference's operation order and lives on the device.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <mutex>
#include <vector>

#include "../../include/glass_hip_wdm.h"
#include "fft_lds.h"
#include "reduce.h"
#include "runtime.h"
#include "wdm_common.h"

namespace glass {
namespace wdm {

// ------------------------------------------------------------ TDI table --

constexpr TdiTerm kTdi[8] = {
    {0, 2, 1, +1, 0, 1, -1, 1, 2, 2.0, 2.0},
    {1, 2, 1, -1, 0, 2, +1, 1, 2, 1.0, 2.0},
    {2, 1, 2, +1, 1, 1, -1, 0, 1, 1.0, 2.0},
    {0, 1, 0, -1, 0, 1, +1, 0, 2, 2.0, 0.0},
    {0, 2, 0, +1, 1, 2, -1, 1, 1, 2.0, 0.0},
    {2, 1, 0, -1, 1, 1, +1, 0, 1, 1.0, 0.0},
    {1, 2, 0, +1, 0, 2, -1, 1, 2, 1.0, 0.0},
    {0, 0, 0, -1, 0, 2, +1, 1, 1, 0.0, 0.0},
};

// ----------------------------------------------------- host: splines ----

// Natural cubic spline coefficients c = y0|y1|y2|y3 (N each), the
// recurrence of spline_coefficients (utils/src/glass_math.c:98-178).
void spline_host(int N, const double* x, const double* y, double* c)
{
#pragma clang fp contract(off)
    std::vector<double> dx(N, 0.0), alpha(N, 0.0), l(N, 0.0), z(N, 0.0), mu(N, 0.0);
    double *y0 = c, *y1 = c + N, *y2 = c + 2 * N, *y3 = c + 3 * N;
    dx[0] = x[1] - x[0];
    for (int i = 1; i < N - 1; i++)
    {
        dx[i] = x[i + 1] - x[i];
        alpha[i] = 3.0 * ((y[i + 1] - y[i]) / dx[i] - (y[i] - y[i - 1]) / dx[i - 1]);
    }
    l[0] = l[N - 1] = 1.0;
    for (int i = 1; i < N - 1; i++)
    {
        l[i] = 2.0 * (x[i + 1] - x[i - 1]) - dx[i - 1] * mu[i - 1];
        mu[i] = dx[i] / l[i];
        z[i] = (alpha[i] - dx[i - 1] * z[i - 1]) / l[i];
    }
    y0[N - 1] = y[N - 1];
    y1[N - 1] = y2[N - 1] = y3[N - 1] = 0.0;
    for (int i = N - 2; i >= 0; i--)
    {
        y0[i] = y[i];
        y2[i] = z[i] - mu[i] * y2[i + 1];
        y1[i] = (y0[i + 1] - y0[i]) / dx[i] - dx[i] * (y2[i + 1] + 2.0 * y2[i]) / 3.0;
        y3[i] = (y2[i + 1] - y2[i]) / (3.0 * dx[i]);
    }
}

// x-only terms of the recurrence: dx | l | mu | 1/l (N each; the
// reciprocals correctly rounded, for spline_sweep's division)
static void spline_prep_host(int N, const double* x, double* p, int* warm)
{
#pragma clang fp contract(off)
    double *dx = p, *l = p + N, *mu = p + 2 * N, *rl = p + 3 * N;
    for (int i = 0; i < 4 * N; i++) p[i] = 0.0;
    dx[0] = x[1] - x[0];
    for (int i = 1; i < N - 1; i++) dx[i] = x[i + 1] - x[i];
    l[0] = l[N - 1] = 1.0;
    for (int i = 1; i < N - 1; i++)
    {
        l[i] = 2.0 * (x[i + 1] - x[i - 1]) - dx[i - 1] * mu[i - 1];
        mu[i] = dx[i] / l[i];
    }
    for (int i = 0; i < N; i++) rl[i] = 1.0 / l[i];
    // knots after which either recurrence holds less than 2^-80 of what it
    // started from (42 on even knots)
    *warm = 1;
    for (int i = 1; i < N - 1; i++)
    {
        double f = 1.0, b = 1.0;
        int n = 0;
        for (int j = i; j < N - 1 && (f > 0x1p-80 || b > 0x1p-80); j++, n++)
        {
            f *= dx[j - 1] / l[j];
            b *= mu[j];
        }
        if (n > *warm) *warm = n;
    }
}

// ------------------------------------------------------ host: geometry --

static double incomplete_beta(double a, double b, double x)
{
#pragma clang fp contract(off)
    // incomplete_beta_function (utils/src/glass_math.c:1214-1242): the
    // Gauss series 2F1(a, 1-b; a+1; x) to |term| <= 1e-8
    double aa = a, bb = 1 - b, cc = a + 1;
    double term = aa * bb * x / cc;
    double value = 1.0 + term;
    int n = 1;
    while (fabs(term) > 1e-8)
    {
        aa++, bb++, cc++, n++;
        term *= aa * bb * x / cc / n;
        value += term;
    }
    double B = exp(lgamma(a) + lgamma(b) - lgamma(a + b));
    return pow(x, a) * value / B / a;
}

// build_wdm_filter_freq (utils/src/glass_wavelet.c:305-349), forward
void wdm_window(int Nf, int Nt, double A, double* phif)
{
#pragma clang fp contract(off)
    const double DeltaOmega = M_PI / Nf;
    const double domega = 2 * DeltaOmega / (double)Nt;
    for (int i = 0; i < Nt / 2 + 1; i++)
    {
        double omega = domega * i;
        double B = DeltaOmega - 2 * A;
        double insDOM = 1.0 / sqrt(DeltaOmega);
        double z = 0.0;
        if (fabs(omega) >= A && fabs(omega) < A + B)
        {
            double x = (fabs(omega) - A) / B;
            double y = incomplete_beta(6.0, 6.0, x);
            z = insDOM * cos(y * M_PI_2);
        }
        if (fabs(omega) < A) z = insDOM;
        phif[i] = z;
    }
    double norm = 0.0;
    for (int i = 0; i < Nt / 2 + 1; i++)
    {
        if (i == 0) norm += phif[i] * phif[i];
        else norm += 2 * phif[i] * phif[i];
    }
    norm *= domega * M_1_PI;
    norm = sqrt(norm);
    norm *= Nf / 2.0;
    for (int i = 0; i < Nt / 2 + 1; i++) phif[i] /= norm;
}

// Device tables of one (wdm grid, orbit knots, Tobs, t0) combination.
struct Geo
{
    int Norb, NT, NF, kmin, kmax, imin, imax;
    double Tobs, t0, dt, df, A, ot0, ods;
    const double* ot;      // Norb orbit knots
    const double* oc;      // 9 x 4 x Norb position splines (row 3*sc+coord)
    const double* prep_o;  // 4 x Norb  dx | l | mu | 1/l on the orbit knots
    const double* tssb;    // Norb response times t0 + i Tobs/(Norb-1)
    const double* prep_s;  // 4 x Norb  on the response times
    int warm_o, warm_s;    // spline_prep_host's warm of both
    const double* resp;    // Norb x 24: x[3][3]/c, n[3][3], L[3] at tssb
    // per layer count L (slot L; a forced count Lf in slot kForcedSlot):
    const double* ds[kForcedSlot + 1];   // N_ds x 5: t, r0x, r0y, r0z, dx
    const int* dsi[kForcedSlot + 1];     // response-time interval
    const double* win[kForcedSlot + 1];  // window of L+1 layers
    int Lf;                // forced layer count of every template (0: ucb_wavelet_layers' own)
    const double2* tw;     // 4096-entry twiddles
    const double2* tw3;    // 12288-entry twiddles
    const double2* tw16;   // 16384-entry twiddles (template series of NT >= 1024)
    const double2* tw32;   // 32768-entry twiddles (forced layer counts)
};

struct GeoHost
{
    Geo g;
    std::vector<void*> bufs;
    ~GeoHost()
    {
        for (void* p : bufs) (void)hipFree(p);
    }
};

template <typename T>
static int upload(GeoHost& G, const std::vector<T>& v, const T** out)
{
    void* d = nullptr;
    GH_CHECK(hipMalloc(&d, sizeof(T) * std::max<size_t>(v.size(), 1)));
    G.bufs.push_back(d);
    GH_CHECK(hipMemcpy(d, v.data(), sizeof(T) * v.size(), hipMemcpyHostToDevice));
    *out = (const T*)d;
    return GLASS_HIP_OK;
}

static double spline_host_at(const std::vector<double>& x, const double* c, int N, double t)
{
#pragma clang fp contract(off)
    int n = knot_index(x.data(), N, t);
    double dx = t - x[n];
    return c[n] + c[N + n] * dx + c[2 * N + n] * dx * dx + c[3 * N + n] * dx * dx * dx;
}

// Fills the tables.  pos: 9 x Norb positions (row 3*sc + coord); Lf > 0
// adds the tables of that forced layer count.
static int geo_build(GeoHost& G, const glass_hip_wdm& w, int Norb, const double* ot_in,
                     const double* pos, double Tobs, double t0, int Lf)
{
#pragma clang fp contract(off)
    Geo& g = G.g;
    const int N = Norb;
    g.Norb = N;
    g.NT = w.NT;
    g.NF = w.NF;
    g.kmin = w.kmin;
    g.kmax = w.kmax;
    g.imin = w.imin;
    g.imax = w.imax;
    g.Tobs = Tobs;
    g.t0 = t0;
    g.dt = w.dt;
    g.df = w.df;
    g.A = w.A;
    std::vector<double> ot(ot_in, ot_in + N);
    g.ot0 = ot[0];
    g.ods = ot[1] - ot[0];
    std::vector<double> oc(9 * 4 * N), prep_o(4 * N), tssb(N), prep_s(4 * N), resp(24 * N, 0.0);
    for (int s = 0; s < 9; s++) spline_host(N, ot.data(), pos + s * N, oc.data() + 4 * s * N);
    spline_prep_host(N, ot.data(), prep_o.data(), &g.warm_o);
    const double dts = Tobs / (double)(N - 1);
    for (int i = 0; i < N; i++) tssb[i] = t0 + i * dts;
    spline_prep_host(N, tssb.data(), prep_s.data(), &g.warm_s);
    if (tssb[0] < ot[0] || tssb[N - 1] > ot[N - 1])
    {
        set_error("wavelet waveform: response times [%g, %g] outside the orbit knots [%g, %g]",
                  tssb[0], tssb[N - 1], ot[0], ot[N - 1]);
        return GLASS_HIP_EINVAL;
    }
    // spacecraft geometry at the response times (LISA_spline_response,
    // utils/src/glass_lisa.c:976-1016)
    for (int m = 0; m < N; m++)
    {
        double x[3][3], n[3][3], L[3];
        for (int i = 0; i < 3; i++)
            for (int d = 0; d < 3; d++)
                x[i][d] = spline_host_at(ot, oc.data() + 4 * (3 * i + d) * N, N, tssb[m]) / CLIGHT;
        for (int i = 0; i < 3; i++)
        {
            n[0][i] = x[1][i] - x[2][i];
            n[1][i] = x[2][i] - x[0][i];
            n[2][i] = x[0][i] - x[1][i];
        }
        for (int i = 0; i < 3; i++)
        {
            L[i] = 0.0;
            for (int j = 0; j < 3; j++) L[i] += n[i][j] * n[i][j];
            L[i] = sqrt(L[i]);
        }
        for (int i = 0; i < 3; i++)
            for (int j = 0; j < 3; j++) n[i][j] /= L[i];
        double* r = resp.data() + 24 * m;
        for (int i = 0; i < 3; i++)
            for (int j = 0; j < 3; j++)
            {
                r[3 * i + j] = x[i][j];
                r[9 + 3 * i + j] = n[i][j];
            }
        for (int i = 0; i < 3; i++) r[18 + i] = L[i];
    }
    int rc;
    if ((rc = upload(G, ot, &g.ot)) || (rc = upload(G, oc, &g.oc)) || (rc = upload(G, prep_o, &g.prep_o)) ||
        (rc = upload(G, tssb, &g.tssb)) || (rc = upload(G, prep_s, &g.prep_s)) ||
        (rc = upload(G, resp, &g.resp)))
        return rc;
    // per layer count L: the downsampled times, spacecraft 1 there, the
    // response-time interval and offset of each sample, and the window
    g.Lf = Lf;
    for (int slot = 1; slot <= (Lf > 0 ? kForcedSlot : kMaxLayers); slot++)
    {
        const int L = slot == kForcedSlot ? Lf : slot;
        const int Nds = w.NT * (L + 1);
        const double dt_ds = w.dt / (double)(L + 1);
        std::vector<double> ds(5 * (size_t)Nds);
        std::vector<int> dsi(Nds);
        for (int i = 0; i < Nds; i++)
        {
            double t = t0 + i * dt_ds;
            if (t < tssb[0] || t > tssb[N - 1] || t < ot[0] || t > ot[N - 1])
            {
                set_error("wavelet waveform: sample time %g of the %d-layer grid (NT*dt = %g) lies "
                          "outside [t0, t0+Tobs] = [%g, %g]",
                          t, L, w.NT * w.dt, tssb[0], tssb[N - 1]);
                return GLASS_HIP_EINVAL;
            }
            double* e = ds.data() + 5 * (size_t)i;
            e[0] = t;
            for (int d = 0; d < 3; d++) e[1 + d] = spline_host_at(ot, oc.data() + 4 * d * N, N, t) / CLIGHT;
            int k = knot_index(tssb.data(), N, t);
            dsi[i] = k;
            e[4] = t - tssb[k];
        }
        std::vector<double> win(w.NT / 2 + 1);
        wdm_window(L + 1, w.NT, w.A, win.data());
        if ((rc = upload(G, ds, &g.ds[slot])) || (rc = upload(G, dsi, &g.dsi[slot])) ||
            (rc = upload(G, win, &g.win[slot])))
            return rc;
    }
    g.ds[0] = nullptr;
    g.dsi[0] = nullptr;
    g.win[0] = nullptr;
    if (Lf <= 0)
    {
        g.ds[kForcedSlot] = nullptr;
        g.dsi[kForcedSlot] = nullptr;
        g.win[kForcedSlot] = nullptr;
    }
    g.tw32 = nullptr;
    if ((rc = twiddles(&g.tw)) || (rc = twiddles3(&g.tw3)) || (rc = twiddles16(&g.tw16)) ||
        (Lf > 0 && (rc = twiddles32(&g.tw32))))
        return rc;
    return GLASS_HIP_OK;
}

// Validates the grid for the template kernels.
static int check_grid(const glass_hip_wdm* w, int Norb)
{
    if (!w) return set_error("NULL wdm"), GLASS_HIP_EINVAL;
    if (w->NT != 256 && w->NT != 512 && w->NT != 1024 && w->NT != 2048 && w->NT != 4096)
    {
        set_error("wavelet templates: NT = %d unsupported (this build computes templates for NT = 256, 512, "
                  "1024, 2048 or 4096)",
                  w->NT);
        return GLASS_HIP_EINVAL;
    }
    if (w->NF < 4 || w->dt <= 0 || w->df <= 0)
        return set_error("wavelet templates: bad grid NF=%d dt=%g df=%g", w->NF, w->dt, w->df), GLASS_HIP_EINVAL;
    if (Norb < 4 || Norb > kMaxKnots)
        return set_error("wavelet templates: %d orbit knots (supported 4..%d)", Norb, kMaxKnots),
               GLASS_HIP_EINVAL;
    return GLASS_HIP_OK;
}

// ------------------------------------------------------- K1: response ---

// Per-template scratch (global): header, barycentre phase spline (4N),
// TDI splines (6 x 4N: amp X, phase X, amp Y, phase Y, amp Z, phase Z).
__host__ __device__ inline size_t scratch_doubles(int N) { return 64 + 28 * (size_t)N; }

constexpr int kRespThreads = 256;

// LDS of K1 in doubles: sine table 512 | ssb 8N | M,Mf 6N | As 3N | z 3N |
// phase_sc N.  The splines' right-hand sides and sweeps live in regions dead by
// then: the two barycentre splines in M,Mf (not yet written), the six TDI
// splines in ssb (right-hand sides, then y2) and As + z (the forward sweeps),
// dead after the signed amplitude/phase step.  Then the sign-flip scan's knot
// flags: per channel the d2 and d3 tests and the flips, kMaxKnots bits each.
constexpr int kFlagWords = kMaxKnots / 64;
__host__ __device__ inline size_t resp_lds_bytes(int N)
{
    return sizeof(double) * (512 + 21 * (size_t)N) + sizeof(unsigned long long) * 9 * kFlagWords;
}

// Per-template constants, one thread per template, into each template's
// scratch header (read by K1 and K2).
__global__ void __launch_bounds__(256) hdr_kernel(Geo g, int n, const double* __restrict__ params,
                                                 double* __restrict__ scratch)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n) return;
    Hdr h;
    make_hdr(params + 8 * (size_t)e, g.Tobs, g.df, g.A, &h);
    if (g.Lf > 0) h.L = g.Lf;  // forced layer count: same first layer and heterodyne
    *(Hdr*)(scratch + scratch_doubles(g.Norb) * (size_t)e) = h;
}

// The right-hand side alpha_i (1 <= i <= N-2) of the natural spline
// through y (knots described by prep), into z[i]: independent per knot, so
// the whole workgroup computes them before one lane's sweep.
__device__ inline void spline_alpha(int N, const double* __restrict__ prep, const double* y, double* z, int i)
{
#pragma clang fp contract(off)
    const double* dx = prep;
    z[i] = 3.0 * ((y[i + 1] - y[i]) / dx[i] - (y[i] - y[i - 1]) / dx[i - 1]);
}

// The tridiagonal sweeps of that spline over chunk c of kSweepChunks, one lane
// each: alpha (spline_alpha) -> z, and after a barrier z -> y2.  Only the
// recurrence itself is serial (its division by l_i goes through the precomputed
// 1/l_i) and it forgets: each knot keeps 0.27 of the one before, so a chunk that
// starts `warm` knots early from zero holds the value of the whole sweep (2^-80
// of it is left out, 2^-27 of its last bit).  62 dependent steps for 202 knots
// instead of 202.  The x-only terms come from LDS: a step that waits for L2 takes
// 380 cycles, five times its arithmetic.
constexpr int kSweepChunks = 10;
struct SweepTerms
{
    double *dx, *l, *mu, *rl;
    // from prep (spline_prep_host), by the whole workgroup
    __device__ __forceinline__ void fill(int N, const double* __restrict__ prep) const
    {
        for (int i = threadIdx.x; i < N; i += kRespThreads)
        {
            dx[i] = prep[i];
            l[i] = prep[N + i];
            mu[i] = prep[2 * N + i];
            rl[i] = prep[3 * N + i];
        }
    }
};
__device__ inline void sweep_range(int N, int c, int* lo, int* hi)
{
    const int len = (N - 2 + kSweepChunks - 1) / kSweepChunks;
    *lo = 1 + c * len;
    *hi = min(N - 1, *lo + len);
}
__device__ inline void spline_forward(int N, const SweepTerms& s, const double* alpha, double* z, int c, int warm)
{
#pragma clang fp contract(off)
    int lo, hi;
    sweep_range(N, c, &lo, &hi);
    if (c == 0) z[0] = 0.0;
    double zp = 0.0;
#pragma unroll 4
    for (int i = max(1, lo - warm); i < hi; i++)
    {
        zp = div_by_recip(alpha[i] - s.dx[i - 1] * zp, s.l[i], s.rl[i]);
        if (i >= lo) z[i] = zp;
    }
}
__device__ inline void spline_backward(int N, const SweepTerms& s, const double* z, double* y2, int c, int warm)
{
#pragma clang fp contract(off)
    int lo, hi;
    sweep_range(N, c, &lo, &hi);
    if (c == 0) lo = 0;
    if (c == kSweepChunks - 1) y2[N - 1] = 0.0;
    double yn = 0.0;
#pragma unroll 4
    for (int i = min(N - 2, hi - 1 + warm); i >= lo; i--)
    {
        yn = z[i] - s.mu[i] * yn;
        if (i < hi) y2[i] = yn;
    }
}

// y1, y3 of knot i from y0 and y2
__device__ inline void spline_finish(int N, int i, const double* __restrict__ prep, const double* y0,
                                     const double* y2, double* y1o, double* y3o)
{
#pragma clang fp contract(off)
    if (i == N - 1)
    {
        *y1o = 0.0;
        *y3o = 0.0;
        return;
    }
    const double dx = prep[i];
    *y1o = (y0[i + 1] - y0[i]) / dx - dx * (y2[i + 1] + 2.0 * y2[i]) / 3.0;
    *y3o = (y2[i + 1] - y2[i]) / (3.0 * dx);
}

// A template's header by scalar loads.
__device__ __forceinline__ Hdr load_hdr(const double* scr)
{
    Hdr h;
    auto hs = (const __attribute__((address_space(4))) double*)scr;
#pragma unroll
    for (int i = 0; i < (int)(sizeof(Hdr) / sizeof(double)); i++) ((double*)&h)[i] = hs[i];
    return h;
}

// Vector issue bounds it (65% busy), most of it in the 24 delayed terms of
// a knot.  Their sine and cosine come from a table in LDS (sincos_tab); the
// vertices and arms are permuted for the channel as they are loaded, so the
// eight terms are written out without selects; and what is serial along the
// knots, which one wave worked while three waited, is cut into chunks (the
// splines), bits (the flips) and a prefix sum (the unwrapping).  4096 templates
// of 202 knots: 718 -> 338 us.  Four waves per SIMD (128 VGPRs): four 256-thread
// workgroups per CU, as many as the LDS allows.
__global__ void __launch_bounds__(kRespThreads) __attribute__((amdgpu_waves_per_eu(4, 8))) resp_kernel(
    Geo g, int n, double* __restrict__ scratch)
{
#pragma clang fp contract(off)
    const int e = blockIdx.x;
    if (e >= n) return;
    extern __shared__ double lds[];
    const int N = g.Norb;
    const int tid = threadIdx.x;
    dd_t* tab = (dd_t*)lds;          // sin_tab_entry
    double* ssb = lds + 512;         // amp y0..y3 | phase y0..y3
    double* Mx = ssb + 8 * N;        // M X,Y,Z | Mf X,Y,Z
    double* As = Mx + 6 * N;         // |M| X,Y,Z, and 3N more
    double* phsc = As + 6 * N;       // phase at spacecraft 1
    unsigned long long* flg = (unsigned long long*)(phsc + N);  // 9 x kFlagWords
    double* scr = scratch + scratch_doubles(N) * (size_t)e;

    // the header hdr_kernel wrote, by scalar loads
    const Hdr h = load_hdr(scr);
    for (int i = tid; i < 256; i += kRespThreads) tab[i] = sin_tab_entry(i);
    // barycentre amplitude and phase at the orbit knots
    for (int i = tid; i < N; i += kRespThreads)
    {
        const double t = g.ot[i];
        ssb[i] = ucb_amplitude(t, h.A0, h.f0, h.fdot);
        ssb[4 * N + i] = ucb_phase(t, h.f0, h.phi0, h.fdot);
    }
    __syncthreads();
    for (int it = tid; it < 2 * (N - 2); it += kRespThreads)
    {
        const int sp = it / (N - 2), i = 1 + it % (N - 2);
        spline_alpha(N, g.prep_o, ssb + 4 * N * sp, Mx + N * sp, i);
    }
    const SweepTerms to{As, As + N, As + 2 * N, As + 3 * N};  // not yet written
    to.fill(N, g.prep_o);
    __syncthreads();
    {
        const int sp = tid / kSweepChunks, c = tid % kSweepChunks;
        double* z = Mx + (2 + sp) * N;
        if (sp < 2) spline_forward(N, to, Mx + N * sp, z, c, g.warm_o);
        __syncthreads();
        if (sp < 2) spline_backward(N, to, z, ssb + 4 * N * sp + 2 * N, c, g.warm_o);
    }
    __syncthreads();
    for (int i = tid; i < 2 * N; i += kRespThreads)
    {
        const int s = i / N, k = i % N;
        double* c = ssb + 4 * N * s;
        spline_finish(N, k, g.prep_o, c, c + 2 * N, c + N + k, c + 3 * N + k);
    }
    __syncthreads();
    const double* cph = ssb + 4 * N;
    const double rds = 1.0 / g.ods;
    // even_index with the division by the knot spacing through its reciprocal
    auto knot = [&](double x) {
        const int j = (int)floor(div_by_recip(x - g.ot0, g.ods, rds));
        return min(max(j, 0), N - 1);
    };
    // export the barycentre phase spline for the layer kernel
    for (int i = tid; i < 4 * N; i += kRespThreads) scr[64 + i] = cph[i];
    // phase at spacecraft 1 (LISA_spacecraft_to_barycenter_time, flag -1)
    for (int m = tid; m < N; m += kRespThreads)
    {
        const double* r = g.resp + 24 * m;
        double kdotr = 0.0;
        for (int i = 0; i < 3; i++) kdotr += h.k[i] * r[i];
        const double tsc = g.tssb[m] - kdotr;
        const int j = knot(tsc);
        phsc[m] = spline_at(cph, N, j, tsc - g.ot[j]);
    }
    // the X, Y, Z responses: items (sample m, channel ch), vertex and arm i of
    // the channel's permutation being (ch + i) mod 3
    for (int it = tid; it < 3 * N; it += kRespThreads)
    {
        const int m = it / 3, ch = it % 3;
        const double* r = g.resp + 24 * m;
        double kr[3], L[3], App[3], Apm[3], Acp[3], Acm[3];
#pragma unroll
        for (int i = 0; i < 3; i++)
        {
            const int v = ch + i < 3 ? ch + i : ch + i - 3;
            const double *x = r + 3 * v, *nn = r + 9 + 3 * v;
            L[i] = r[18 + v];
            kr[i] = 0.0;
            double kn = 0.0;
#pragma unroll
            for (int j = 0; j < 3; j++)
            {
                kr[i] += h.k[j] * x[j];
                kn += h.k[j] * nn[j];
            }
            double dp = 0.0, dc = 0.0;
#pragma unroll
            for (int j = 0; j < 3; j++)
#pragma unroll
                for (int l = 0; l < 3; l++)
                {
                    dp += (nn[j] * nn[l]) * h.ep[3 * j + l];
                    dc += (nn[j] * nn[l]) * h.ec[3 * j + l];
                }
            const double bp = 1.0 + kn, bm = 1.0 - kn, rp = 1.0 / bp, rm = 1.0 / bm;
            App[i] = div_by_recip(dp, bp, rp);
            Apm[i] = div_by_recip(dp, bm, rm);
            Acp[i] = div_by_recip(dc, bp, rp);
            Acm[i] = div_by_recip(dc, bm, rm);
        }
        const double t = g.tssb[m];
        double M = 0.0, Mf = 0.0;
#pragma unroll
        for (int q = 0; q < 8; q++)
        {
            const TdiTerm T = kTdi[q];
            const double te = t - kr[T.v] - T.m1 * L[T.i1] - T.m2 * L[T.i2];
            const int j = knot(te);
            const double dx = te - g.ot[j];
            const double a = spline_at(ssb, N, j, dx);
            const double ph = spline_at(cph, N, j, dx);
            // correctly rounded: the channel sums cancel by (f/f*)^2, which
            // would magnify one-ulp differences of sin/cos
            const sc_t sc = sincos_tab(ph, tab);
            const double sp = sc.s, cp = sc.c;
            const double hp = a * (h.Ap * h.c2p * cp + h.Ac * h.s2p * sp);
            const double hc = a * (h.Ac * h.c2p * sp - h.Ap * h.s2p * cp);
            const double hpf = a * (-h.Ap * h.c2p * sp + h.Ac * h.s2p * cp);
            const double hcf = a * (h.Ac * h.c2p * cp + h.Ap * h.s2p * sp);
            const double P1 = T.pm1 ? App[T.j1] : Apm[T.j1], Q1 = T.pm1 ? Acp[T.j1] : Acm[T.j1];
            const double P2 = T.pm2 ? App[T.j2] : Apm[T.j2], Q2 = T.pm2 ? Acp[T.j2] : Acm[T.j2];
            double v;
            v = hp * P1 + hc * Q1;
            M = T.s1 > 0 ? M + v : M - v;
            v = hp * P2 + hc * Q2;
            M = T.s2 > 0 ? M + v : M - v;
            v = hpf * P1 + hcf * Q1;
            Mf = T.s1 > 0 ? Mf + v : Mf - v;
            v = hpf * P2 + hcf * Q2;
            Mf = T.s2 > 0 ? Mf + v : Mf - v;
            __builtin_amdgcn_sched_barrier(0);  // one term's temporaries at a time
        }
        Mx[ch * N + m] = M;
        Mx[(3 + ch) * N + m] = Mf;
        As[ch * N + m] = sqrt(M * M + Mf * Mf);
    }
    __syncthreads();
    // sign flips of the amplitude (extract_amplitude_and_phase,
    // utils/src/glass_math.c:1244-1296): at a local minimum of |M| the tests
    // |d2/d1| < 0.1 (the amplitude and its phase jump flip at the next knot,
    // which is then skipped) and |d3/d1| < 0.1 (they flip at this one).  The
    // tests need no state: every wave evaluates 64 knots of a channel into
    // ballot masks.  One lane per channel walks the knots that pass one, in
    // the reference's order, and leaves a mask of the flips.
    const int NWd = (N + 63) / 64, lane = tid & 63;
    for (int b = tid >> 6; b < 3 * NWd; b += kRespThreads / 64)
    {
        const int ch = b / NWd, w = b % NWd, i = w * 64 + lane;
        bool t2 = false, t3 = false;
        if (i >= 1 && i <= N - 2)
        {
            const double* A = As + ch * N;
            if (A[i] < A[i - 1] && A[i] < A[i + 1])
            {
                const double d1 = A[i + 1] + A[i - 1] - 2.0 * A[i];
                const double d2 = -A[i + 1] + A[i - 1] - 2.0 * A[i];
                const double d3 = -A[i + 1] + A[i - 1] + 2.0 * A[i];
                t2 = fabs(d2 / d1) < 0.1;
                t3 = fabs(d3 / d1) < 0.1;
            }
        }
        const unsigned long long m2 = __ballot(t2), m3 = __ballot(t3);
        if (lane == 0)
        {
            flg[(ch * 3 + 0) * kFlagWords + w] = m2;
            flg[(ch * 3 + 1) * kFlagWords + w] = m3;
            flg[(ch * 3 + 2) * kFlagWords + w] = 0;
        }
    }
    __syncthreads();
    if (tid < 3)
    {
        const unsigned long long *f2 = flg + tid * 3 * kFlagWords, *f3 = f2 + kFlagWords;
        unsigned long long* fl = flg + tid * 3 * kFlagWords + 2 * kFlagWords;
        int i = 1;
        while (i < N - 1)
        {
            const int w = i >> 6;
            const unsigned long long m = (f2[w] | f3[w]) >> (i & 63);
            if (!m)
            {
                i = (w + 1) * 64;
                continue;
            }
            i += __ffsll(m) - 1;
            const bool b2 = (f2[w] >> (i & 63)) & 1;  // else b3
            const int at = b2 ? i + 1 : i;
            if (at < N) fl[at >> 6] |= 1ull << (at & 63);
            i = at + 1;
        }
    }
    __syncthreads();
    // signed amplitude and phase relative to the spacecraft-1 carrier; the
    // last knot has the flips of the one before
    for (int it = tid; it < 3 * N; it += kRespThreads)
    {
        const int ch = it / N, i = it % N, k = min(i, N - 2);
        const unsigned long long* fl = flg + ch * 3 * kFlagWords + 2 * kFlagWords;
        int flips = __popcll(fl[k >> 6] << (63 - (k & 63)));
        for (int w = 0; w < k >> 6; w++) flips += __popcll(fl[w]);
        double pj = 0.0;
        for (int w = 0; w < flips; w++) pj += M_PI;
        const double M = Mx[ch * N + i], Mf = Mx[(3 + ch) * N + i];
        const double v = remainder(phsc[i], PI2);
        Mx[ch * N + i] = flips & 1 ? -As[ch * N + i] : As[ch * N + i];
        Mx[(3 + ch) * N + i] = -atan2_cr(Mf, M) + pj - v;
    }
    __syncthreads();
    // unwrap_phase (utils/src/glass_math.c:1034-1052), one wave per channel:
    // the turns added at a knot are those of the one before and the difference
    // of the two phases in turns, rounded, so they are a prefix sum.  Where a
    // difference is within 1e-6 of half a turn (or is NaN) the rounding of the
    // unwrapped phase decides, and one lane walks the knots.
    if (tid < 192)
    {
        constexpr double kInvPI2 = 1.0 / PI2;  // correctly rounded (compile time)
        double* ph = Mx + (3 + (tid >> 6)) * N;
        bool near = false;
        for (int i = 1 + lane; i < N; i += 64)
        {
            const double f = (ph[i - 1] - ph[i]) * kInvPI2;
            near = near || !(fabs(f - rint(f)) < 0.499999);
        }
        if (__ballot(near) == 0)
        {
            double turns = 0.0, last = ph[0];
            for (int i0 = 0; i0 < N; i0 += 64)
            {
                const int i = i0 + lane;
                const double p = ph[min(i, N - 1)];
                double b = __shfl_up(p, 1, 64);
                if (lane == 0) b = last;
                double d = rint((b - p) * kInvPI2);
#pragma unroll
                for (int w = 1; w < 64; w <<= 1)
                {
                    const double o = __shfl_up(d, w, 64);
                    if (lane >= w) d += o;
                }
                d += turns;
                if (i < N) ph[i] = p + d * PI2;
                turns = __shfl(d, 63, 64);
                last = __shfl(p, 63, 64);
            }
        }
        else if (lane == 0)
        {
            double v = ph[0];
#pragma unroll 4
            for (int i = 0; i < N; i++)
            {
                double u = ph[i];
                const double q = rint(div_by_recip(fabs(u - v), PI2, kInvPI2));
                if (q > 0.0)
                {
                    if (v > u) u += q * PI2;
                    else u -= q * PI2;
                }
                v = u;
                ph[i] = u;
            }
        }
    }
    __syncthreads();
    // six TDI splines on the response times: spline s = 2*ch + (0 amp, 1 phase)
    for (int it = tid; it < 6 * (N - 2); it += kRespThreads)
    {
        const int sp = it / (N - 2), i = 1 + it % (N - 2);
        const int ch = sp >> 1, ph = sp & 1;
        spline_alpha(N, g.prep_s, Mx + (3 * ph + ch) * N, ssb + sp * N, i);
    }
    static_assert(kMaxKnots <= 512, "mu in the sine table's place");
    const SweepTerms ts{ssb + 6 * N, ssb + 7 * N, lds, phsc};  // what they held is dead
    ts.fill(N, g.prep_s);
    __syncthreads();
    {
        const int sp = tid / kSweepChunks, c = tid % kSweepChunks;
        if (sp < 6) spline_forward(N, ts, ssb + sp * N, As + sp * N, c, g.warm_s);
        __syncthreads();
        if (sp < 6) spline_backward(N, ts, As + sp * N, ssb + sp * N, c, g.warm_s);
    }
    __syncthreads();
    for (int it = tid; it < 6 * N; it += kRespThreads)
    {
        const int s = it / N, i = it % N;
        const int ch = s >> 1, ph = s & 1;
        const double* y0 = Mx + (3 * ph + ch) * N;
        const double* y2 = ssb + s * N;
        double y1, y3;
        spline_finish(N, i, g.prep_s, y0, y2, &y1, &y3);
        double* c = scr + 64 + 4 * N + 4 * (size_t)N * s;
        c[i] = y0[i];
        c[N + i] = y1;
        c[2 * N + i] = y2[i];
        c[3 * N + i] = y3;
    }
}

// ---------------------------------------------------------- K2: layers --

struct LayerArgs
{
    const double* data;   // 3 planes of npix (NULL: no inner products)
    const double* invC;   // 6 planes XX,YY,ZZ,XY,XZ,YZ of npix
    int npix;
    int* nwave;           // [n]
    int* list;            // [n x vcap] (compact pixel list)
    double* values;       // [n x 3 x vcap]
    double* dlogL;        // [n] (with data)
    double* snr;          // [n] (with data)
    double2* big;         // long-series kernel: nbig global scratch slices of bigslice double2
    int nbig;
    int vcap;             // pixels per template: 3 NT (NT max(3, Lf) with a forced layer count)
    size_t bigslice;
};

// X, Y (packed in U) or Z (half-length V) spectrum at bin k, 0 < k < Nds/2
template <int NDS>
__device__ inline double2 spectrum(int ch, int k, const double2* U, const double2* V, const double2* tw,
                                   int twstride)
{
    if (ch < 2)
    {
        const double2 a = U[k], b = U[(NDS - k) % NDS];
        // X = (U[k] + conj U[N-k]) / 2 ; Y = (U[k] - conj U[N-k]) / (2i)
        if (ch == 0) return make_double2(0.5 * (a.x + b.x), 0.5 * (a.y - b.y));
        return make_double2(0.5 * (a.y + b.y), -0.5 * (a.x - b.x));
    }
    constexpr int M = NDS / 2;
    const double2 a = V[k % M], b = V[(M - k % M) % M];
    const double2 E = make_double2(0.5 * (a.x + b.x), 0.5 * (a.y - b.y));
    const double2 O = make_double2(0.5 * (a.y + b.y), -0.5 * (a.x - b.x));
    const double2 w = tw[k * twstride];  // exp(-2 pi i k / NDS)
    return make_double2(E.x + (w.x * O.x - w.y * O.y), E.y + (w.x * O.y + w.y * O.x));
}

// Exclusive prefix sum of v over the workgroup in thread order, by wave
// scans (__shfl_up) and one pass over the NTHR/64 wave totals; ws holds
// NTHR/64 + 1 ints of LDS and ends with the total in ws[NTHR/64].  Ends
// with a barrier.
template <int NTHR>
__device__ inline int block_exclusive_scan(int v, int* ws)
{
    static_assert(NTHR % 64 == 0, "wave64 workgroups");
    constexpr int NW = NTHR / 64;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int x = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1)
    {
        const int y = __shfl_up(x, d, 64);
        if (lane >= d) x += y;
    }
    if (lane == 63) ws[w] = x;
    __syncthreads();
    if (threadIdx.x == 0)
    {
        int sum = 0;
        for (int i = 0; i < NW; i++)
        {
            const int t = ws[i];
            ws[i] = sum;
            sum += t;
        }
        ws[NW] = sum;
    }
    __syncthreads();
    return ws[w] + x - v;
}

// Doubles of a template's splines (phase at the barycentre, six TDI splines)
// staged in LDS for its samples, where they fit: a sample gathers 29 of them,
// from L2 a vector-memory instruction each.
__host__ __device__ constexpr int spline_doubles(int N) { return 28 * N; }
constexpr int kStagedKnots = 320;  // 72 KB

// Sample i of the heterodyned X, Y, Z series (ds, dsi: tables of its layer
// count).
__device__ __forceinline__ void series_sample(const Geo& g, const Hdr& h, const double* __restrict__ ds,
                                              const int* __restrict__ dsi, int i, const double* cph,
                                              const double* ctdi, double rds, double (&x)[3])
{
#pragma clang fp contract(off)
    const int N = g.Norb;
    const double* e5 = ds + 5 * (size_t)i;
    const double t = e5[0];
    double kdotr = 0.0;
#pragma unroll
    for (int d = 0; d < 3; d++) kdotr += h.k[d] * e5[1 + d];
    const double tsc = t - kdotr;
    // even_index with the division by the knot spacing through its reciprocal
    int j = (int)floor(div_by_recip(tsc - g.ot0, g.ods, rds));
    j = min(max(j, 0), N - 1);
    const double phase_ds = spline_at(cph, N, j, tsc - g.ot[j]);
    const double phase_het = PI2 * h.fhet * t;
    const int si = dsi[i];
    const double sdx = e5[4];
#pragma unroll
    for (int ch = 0; ch < 3; ch++)
    {
        const double Amp = spline_at(ctdi + 4 * N * (2 * ch), N, si, sdx);
        double Phase = spline_at(ctdi + 4 * N * (2 * ch + 1), N, si, sdx);
        Phase += phase_ds;
        Phase -= phase_het;
        double s, c;
        sincos_red(Phase, &s, &c);
        x[ch] = Amp * c;
    }
}

// The first decimation of thread t's samples n = t + NT p, p < P, of the packed
// series: u (X + i Y, P NT points) into P series of NT points, U[P k + r] =
// FFT(ur)[k], and z (Z, two samples a point: lanes 2n and 2n + 1 hold one) into P
// of NT/2.  pu(r, v): point t of series r; pv(r, v): point t/2, called by one of
// the two lanes.  tw: P NT-th roots, tws apart.
template <int NT, int P, typename PU, typename PV>
__device__ __forceinline__ void series_dif(double2 (&u)[P], const double (&z)[P], int t,
                                           const double2* __restrict__ tw, int tws, PU&& pu, PV&& pv)
{
    double2 y[P], v[P];
    radix_butterfly<P>(u, y);
    pu(0, y[0]);
#pragma unroll
    for (int r = 1; r < P; r++) pu(r, cmul(y[r], tw[r * t * tws]));
    const bool odd = t & 1;
#pragma unroll
    for (int p = 0; p < P; p++)
    {
        const double o = __shfl_xor(z[p], 1, 64);
        v[p] = odd ? make_double2(o, z[p]) : make_double2(z[p], o);
    }
    radix_butterfly<P>(v, y);
#pragma unroll
    for (int r = 0; r < P; r++)
        if (odd == ((r & 1) != 0)) pv(r, r == 0 ? y[0] : cmul(y[r], tw[r * (t >> 1) * 2 * tws]));
}

// The windowed and conjugated X, Y, Z spectra of bin k (0 < k < NDS/2) from U
// and V.  w: exp(-2 pi i k / NDS).  The inverse transforms are forward ones of
// the conjugates.
__device__ __forceinline__ void band_bin(double2 ua, double2 ub, double2 va, double2 vb, double2 w, double wt,
                                         double2 (&o)[3])
{
    // X = (U[k] + conj U[NDS-k]) / 2 ; Y = (U[k] - conj U[NDS-k]) / (2i)
    wt *= 0.5;
    o[0] = make_double2(wt * (ua.x + ub.x), -wt * (ua.y - ub.y));
    o[1] = make_double2(wt * (ua.y + ub.y), wt * (ua.x - ub.x));
    const double2 E = make_double2(va.x + vb.x, va.y - vb.y), O = make_double2(va.y + vb.y, -(va.x - vb.x));
    o[2] = make_double2(wt * (E.x + (w.x * O.x - w.y * O.y)), -wt * (E.y + (w.x * O.y + w.y * O.x)));
}

// Pixel value at time n of layer m from the inverse transform r (conjugated).
__device__ __forceinline__ double pixel_value(double2 r, int NT, int NF, int m, int n, double norm)
{
    const double re = r.x / NT, im = -r.y / NT;  // a power of two
    if (m == 0 || m == NF) return (n % 2 == 0) ? re * M_SQRT2 * norm : 0.0;
    const int sgn = (m % 2 == 0) ? 1 : -1;
    return ((n + m) % 2 == 0) ? re * norm : sgn * im * norm;
}

// The pixel list of template e (ucb/src/glass_ucb_waveform.c:1189-1212):
// candidates in (time i, layer j) order, kept when kmin <= k < kmax; returns
// their count, which it stores.  cnt: NTHR/64 + 1 ints of LDS.
template <int NT, int L, int NTHR>
__device__ __forceinline__ int pixel_list(const Geo& g, const Hdr& h, int e, const LayerArgs& a, int* cnt)
{
    constexpr int NC = NT * L;
    int* lst = a.list + (size_t)e * a.vcap;
    const int tid = threadIdx.x, k0 = h.jmin * NT;
    if (k0 >= g.kmin && k0 + NC <= g.kmax)
    {
        // all of them, but for a band at the grid's edge
        for (int c = tid; c < NC; c += NTHR) lst[c] = c / L + (h.jmin + c % L) * NT - g.kmin;
        if (tid == 0) a.nwave[e] = NC;
        return NC;
    }
    constexpr int PER = (NC + NTHR - 1) / NTHR;
    const int c0 = tid * PER;
    int mine = 0;
    for (int c = c0; c < c0 + PER && c < NC; c++)
    {
        const int k = c / L + (h.jmin + c % L) * NT;
        mine += (k >= g.kmin && k < g.kmax);
    }
    int pos = block_exclusive_scan<NTHR>(mine, cnt);
    if (tid == 0) a.nwave[e] = cnt[NTHR / 64];
    for (int c = c0; c < c0 + PER && c < NC; c++)
    {
        const int k = c / L + (h.jmin + c % L) * NT;
        if (k >= g.kmin && k < g.kmax) lst[pos++] = k - g.kmin;
    }
    __threadfence_block();
    __syncthreads();
    return cnt[NTHR / 64];
}

// wavelet_nwip terms of pixel k (index into the data planes): snr^2 = sum h^T
// C h; the logL change of adding the template to a zero model with the
// reference's edge rule (gaussian_log_likelhood_wavelet,
// utils/src/glass_model.c:805-855).
struct PixelData
{
    double w[6], d[3];  // invC and data planes
    __device__ __forceinline__ void load(const LayerArgs& a, int k)
    {
#pragma unroll
        for (int p = 0; p < 6; p++) w[p] = a.invC[p * (size_t)a.npix + k];
#pragma unroll
        for (int p = 0; p < 3; p++) d[p] = a.data[p * (size_t)a.npix + k];
    }
};
__device__ __forceinline__ void pixel_terms(const Geo& g, const LayerArgs& a, int k, const PixelData& x,
                                            const double (&hv)[3], double& hh, double& dl)
{
    const double* d = x.d;
    double C[3][3];
    C[0][0] = x.w[0];
    C[1][1] = x.w[1];
    C[2][2] = x.w[2];
    C[0][1] = C[1][0] = x.w[3];
    C[0][2] = C[2][0] = x.w[4];
    C[1][2] = C[2][1] = x.w[5];
    double th = 0.0, tdh = 0.0, tdd = 0.0;
#pragma unroll
    for (int p = 0; p < 3; p++)
#pragma unroll
        for (int q = 0; q < 3; q++)
        {
            th += hv[p] * hv[q] * C[p][q];
            tdh += d[p] * hv[q] * C[p][q];
            tdd += d[p] * d[q] * C[p][q];
        }
    hh += th;
    const int i = (k + g.kmin) % g.NT;
    if (k >= 0 && k < a.npix) dl += (i < g.imin || i > g.imax) ? 0.5 * tdd : tdh - 0.5 * th;
}

// One template per workgroup of NT threads (NT 256, 512).  Barriers and latency
// bound it, not work: with transforms spread over the workgroup (152 barriers a
// template) the vector units were 28% busy.  So each thread holds its L + 1
// samples of the series through a first decimation, each wave transforms whole
// series of NT points by itself, and the pixels go from the inverse transforms
// to the inner products in registers; six barriers are left.  LDS: up to eight
// series; three layers' nine bands go in two turns.  4096 templates of 512
// time pixels: 457 -> 297 us.
template <int NT, int L>
__device__ __forceinline__ void layer_body(const Geo& g, const Hdr& h, int e, const LayerArgs& a, double2* lds,
                                           int* cnt, const double* __restrict__ scr)
{
    constexpr int P = L + 1, NDS = NT * P, NTHR = NT;
    constexpr int PU = wave_fft_stride(NT) + 1, PV = wave_fft_stride(NT / 2) + 1;
    constexpr int UU = (P * NT + 511) / 512;  // waves the X, Y series take
    const int t = threadIdx.x, N = g.Norb;
    const bool three = (NDS % 3) == 0;
    const double2* twU = three ? g.tw3 : g.tw;
    const int tsU = (three ? kTw3N : kTwN) / NDS;
    const int Nw = pixel_list<NT, L, NTHR>(g, h, e, a, cnt);
    double2 *U = lds, *V = lds + P * PU;
    {
        const double* cs = scr + 64;
        const double rds = 1.0 / g.ods;
        double2 u[P];
        double z[P];
        if (N <= kStagedKnots)
        {
            double* c = (double*)lds;
#pragma unroll 8
            for (int i = t; i < spline_doubles(N); i += NTHR) c[i] = cs[i];
            __syncthreads();
#pragma unroll
            for (int p = 0; p < P; p++)
            {
                double x[3];
                series_sample(g, h, g.ds[L], g.dsi[L], t + NT * p, c, c + 4 * N, rds, x);
                u[p] = make_double2(x[0], x[1]);
                z[p] = x[2];
            }
            __syncthreads();
        }
        else
#pragma unroll
            for (int p = 0; p < P; p++)
            {
                double x[3];
                series_sample(g, h, g.ds[L], g.dsi[L], t + NT * p, cs, cs + 4 * N, rds, x);
                u[p] = make_double2(x[0], x[1]);
                z[p] = x[2];
            }
        series_dif<NT, P>(
            u, z, t, twU, tsU, [&](int r, double2 v) { U[r * PU + wave_fft_slot(t)] = v; },
            [&](int r, double2 v) { V[r * PV + wave_fft_slot(t >> 1)] = v; });
    }
    __syncthreads();
    wave_fft_units<NT, P, NTHR, true, 1>(U, g.tw, kTwN / NT, 0);
    wave_fft_units<NT / 2, P, NTHR, true, 1>(V, g.tw, kTwN / (NT / 2), UU);
    __syncthreads();
    // the bands of the L layers: bin k = P j + r of U is point j of series r
    double2 b[L][3];
    const double* win = g.win[L];
#pragma unroll
    for (int off = 0; off < L; off++)
    {
        const int j = t - NT / 2, k = (off + 1) * NT / 2 + j, m = h.jmin + off;
        b[off][0] = b[off][1] = b[off][2] = make_double2(0.0, 0.0);
        if (t > 0)
        {
            double wt = win[j < 0 ? -j : j];
            if (j == 0 && (m == 0 || m == g.NF)) wt /= 2.0;
            auto at = [&](const double2* s, int stride, int q) { return s[(q % P) * stride + wave_fft_slot(q / P)]; };
            band_bin(at(U, PU, k), at(U, PU, NDS - k), at(V, PV, k), at(V, PV, NDS / 2 - k), twU[k * tsU], wt, b[off]);
        }
    }
    // the inverse transforms, CB channels at a time; thread t takes the pixels
    // c = t + NTHR i, time c / L of layer c % L
    constexpr int CB = 3 * L <= 8 ? 3 : 2;
    double hv[L][3];
    // the pixels' data, loaded during the inverse transforms (all registers are
    // taken where there are three layers)
    constexpr bool EARLY = L <= 2;
    PixelData x[L];
    auto pixel = [&](int i) {
        const int c = t + NTHR * i;
        return Nw == NT * L ? c / L + (h.jmin + c % L) * NT - g.kmin : a.list[(size_t)e * a.vcap + c];
    };
    const double norm = sqrt((double)g.NF) / (L + 1.0);
    double* vals = a.values + (size_t)e * 3 * a.vcap;
#pragma unroll
    for (int c0 = 0; c0 < 3; c0 += CB)
    {
        constexpr int kCh = CB;
        const int nch = c0 + kCh <= 3 ? kCh : 3 - c0;
        __syncthreads();  // the readers of what is in LDS
#pragma unroll
        for (int ch = 0; ch < 3; ch++)
            if (ch >= c0 && ch < c0 + nch)
#pragma unroll
                for (int off = 0; off < L; off++) lds[((ch - c0) * L + off) * PU + wave_fft_slot(t)] = b[off][ch];
        if (EARLY && a.data)
#pragma unroll
            for (int i = 0; i < L; i++)
                if (t + NTHR * i < Nw) x[i].load(a, pixel(i));
        __syncthreads();
        wave_fft_units<NT, kCh * L, NTHR, true, 1>(lds, g.tw, kTwN / NT, 0);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < L; i++)
        {
            const int c = t + NTHR * i, n = c / L, off = c % L;
#pragma unroll
            for (int ch = 0; ch < 3; ch++)
                if (ch >= c0 && ch < c0 + nch)
                {
                    const double2 r = lds[((ch - c0) * L + off) * PU + wave_fft_slot(n)];
                    hv[i][ch] = pixel_value(r, NT, g.NF, h.jmin + off, n, norm);
                    if (c < Nw) vals[ch * a.vcap + c] = hv[i][ch];
                }
        }
    }
    if (!a.data) return;
    double hh = 0.0, dl = 0.0;
#pragma unroll
    for (int i = 0; i < L; i++)
    {
        if (t + NTHR * i >= Nw) continue;
        const int k = pixel(i);
        if (!EARLY) x[i].load(a, k);
        pixel_terms(g, a, k, x[i], hv[i], hh, dl);
    }
    hh = block_sum<NTHR>(hh);
    dl = block_sum<NTHR>(dl);
    if (t == 0)
    {
        a.snr[e] = sqrt(hh);
        a.dlogL[e] = dl;
    }
}

template <int NT>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4, 8))) layer_kernel(
    Geo g, int n, LayerArgs a, const double* __restrict__ scratch)
{
    const int e = blockIdx.x;
    if (e >= n) return;
    extern __shared__ double2 lds2[];
    __shared__ int cnt[NT / 64 + 1];
    const double* scr = scratch + scratch_doubles(g.Norb) * (size_t)e;
    const Hdr h = load_hdr(scr);
    if (h.L == 1) layer_body<NT, 1>(g, h, e, a, lds2, cnt, scr);
    else if (h.L == 2) layer_body<NT, 2>(g, h, e, a, lds2, cnt, scr);
    else layer_body<NT, 3>(g, h, e, a, lds2, cnt, scr);
}

// eight series, or the staged splines of N knots
template <int NT>
static size_t layer_lds_bytes(int N)
{
    const size_t series = sizeof(double2) * 8 * (wave_fft_stride(NT) + 1);
    const size_t staged = N <= kStagedKnots ? sizeof(double) * spline_doubles(N) : 0;
    return series > staged ? series : staged;
}

// ---------------------------------------------- K2 for NT of 1024..4096 --
//
// The heterodyned series of NT (L+1) <= 16384 samples and its spectrum do not
// fit one workgroup's LDS: they live in a global slice per template (U = X + i
// Y, then V = Z packed as above), the L + 1 series of NT and NT/2 points that a
// first decimation in registers leaves.  Four kernels, each with a template's
// work on several workgroups: the samples and their decimation; one workgroup a
// series, cut once more to 512 points a wave; one a channel for the bands and
// their inverse transforms; the pixel list and inner products.  (One workgroup
// for all of a template, with ping-pong stages of the whole series through L2
// and a fifth of the CUs holding a second one, left the vector units 10% busy.)
// 300 templates of 4096 time pixels: 651 -> 271 us.

constexpr int kSeriesThreads = 512;
constexpr int kSumThreads = 1024;

// double2 per scratch slice: U (NDS) and V (NDS / 2), NDS = NT (L + 1) at
// three layers; with a forced count each with its partner (below)
__host__ __device__ inline size_t big_layer_slice(int NT, int Lf = 0)
{
    return Lf > 0 ? 3 * (size_t)NT * (size_t)(Lf + 1) : 6 * (size_t)NT;
}

// f(integral constant L) of a template's layer count
template <typename F>
__device__ __forceinline__ void with_layers(int L, F&& f)
{
    if (L == 1) f(std::integral_constant<int, 1>());
    else if (L == 2) f(std::integral_constant<int, 2>());
    else f(std::integral_constant<int, 3>());
}

template <int NT>
__global__ void __launch_bounds__(kSeriesThreads) __attribute__((amdgpu_waves_per_eu(4, 8))) series_kernel_big(
    Geo g, int e0, LayerArgs a, const double* __restrict__ scratch)
{
    extern __shared__ double ldss[];  // the splines, where staged
    const int N = g.Norb, t = blockIdx.x * kSeriesThreads + threadIdx.x;
    const double* scr = scratch + scratch_doubles(N) * (size_t)(e0 + blockIdx.y);
    const Hdr h = load_hdr(scr);
    double2* S = a.big + a.bigslice * (size_t)blockIdx.y;
    const double* cs = scr + 64;
    const bool staged = N <= kStagedKnots;
    if (staged)
    {
#pragma unroll 8
        for (int i = threadIdx.x; i < spline_doubles(N); i += kSeriesThreads) ldss[i] = cs[i];
        __syncthreads();
    }
    with_layers(h.L, [&](auto l) {
        constexpr int L = decltype(l)::value, P = L + 1, NDS = NT * P;
        const double rds = 1.0 / g.ods;
        double2 u[P];
        double z[P];
        if (staged)
#pragma unroll
            for (int p = 0; p < P; p++)
            {
                double x[3];
                series_sample(g, h, g.ds[L], g.dsi[L], t + NT * p, ldss, ldss + 4 * N, rds, x);
                u[p] = make_double2(x[0], x[1]);
                z[p] = x[2];
            }
        else
#pragma unroll
            for (int p = 0; p < P; p++)
            {
                double x[3];
                series_sample(g, h, g.ds[L], g.dsi[L], t + NT * p, cs, cs + 4 * N, rds, x);
                u[p] = make_double2(x[0], x[1]);
                z[p] = x[2];
            }
        const bool three = P == 3;
        series_dif<NT, P>(
            u, z, t, three ? g.tw3 : g.tw16, (three ? kTw3N : kTw16N) / NDS,
            [&](int r, double2 v) { S[r * NT + t] = v; },
            [&](int r, double2 v) { S[NDS + r * (NT / 2) + (t >> 1)] = v; });
    });
}

// A forward transform of M = 512 P points whose points t + 512 p thread t of
// 512 brings in x: P series of 512 in lds, one a wave; get(i) is point t + 512 i
// of the result, after the call (no barrier after the reads).
template <int M>
struct SplitFft
{
    static constexpr int P = M / 512, PN = wave_fft_stride(512) + 1;
    static constexpr size_t kBytes = sizeof(double2) * P * PN;
    double2* lds;
    __device__ __forceinline__ SplitFft(double2 (&x)[P], double2* buf, const double2* __restrict__ tw, int t) : lds(buf)
    {
        double2* o = lds + wave_fft_slot(t);
        if constexpr (P == 1)
            o[0] = x[0];
        else
        {
            double2 y[P];
            radix_butterfly<P>(x, y);
            o[0] = y[0];
#pragma unroll
            for (int r = 1; r < P; r++) o[r * PN] = cmul(y[r], tw[r * t * (kTwN / M)]);
        }
        __syncthreads();
        wave_fft_units<512, P, 512, true, 1>(lds, tw, kTwN / 512, 0);
        __syncthreads();
    }
    __device__ __forceinline__ double2 get(int b) const { return lds[(b % P) * PN + wave_fft_slot(b / P)]; }
};

template <int M>
__device__ __forceinline__ void fft_in_place(double2* S, double2* lds, const double2* __restrict__ tw)
{
    const int t = threadIdx.x;
    double2 x[M / 512];
#pragma unroll
    for (int p = 0; p < M / 512; p++) x[p] = S[t + 512 * p];
    const SplitFft<M> f(x, lds, tw, t);
#pragma unroll
    for (int p = 0; p < M / 512; p++) S[t + 512 * p] = f.get(t + 512 * p);
}

// blockIdx.x 0..3: series of U, 4..7: of V
template <int NT>
__global__ void __launch_bounds__(512) fft_kernel_big(Geo g, int e0, LayerArgs a, const double* __restrict__ scratch)
{
    extern __shared__ double2 ldsb[];
    const int P = load_hdr(scratch + scratch_doubles(g.Norb) * (size_t)(e0 + blockIdx.y)).L + 1, r = blockIdx.x & 3;
    if (r >= P) return;
    double2* S = a.big + a.bigslice * (size_t)blockIdx.y;
    if (blockIdx.x < 4)
        fft_in_place<NT>(S + r * NT, ldsb, g.tw);
    else
        fft_in_place<NT / 2>(S + P * NT + r * (NT / 2), ldsb, g.tw);
}

// Pixels of a template's list: its candidates inside the grid.
__device__ __forceinline__ int pixel_count(const Geo& g, const Hdr& h, int L)
{
    int n = 0;
    for (int off = 0; off < L; off++)
    {
        const int k0 = (h.jmin + off) * g.NT;
        n += max(0, min(g.kmax, k0 + g.NT) - max(g.kmin, k0));
    }
    return n;
}

// blockIdx.x: channel
template <int NT>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4, 8))) band_kernel_big(
    Geo g, int e0, LayerArgs a, const double* __restrict__ scratch)
{
    extern __shared__ double2 ldsb[];
    const int e = e0 + blockIdx.y, ch = blockIdx.x, t = threadIdx.x;
    const Hdr h = load_hdr(scratch + scratch_doubles(g.Norb) * (size_t)e);
    const double2* S = a.big + a.bigslice * (size_t)blockIdx.y;
    with_layers(h.L, [&](auto l) {
        constexpr int L = decltype(l)::value, P = L + 1, NDS = NT * P, Q = NT / 512;
        const double2 *U = S, *V = S + NDS;
        const bool three = P == 3;
        const double2* twU = three ? g.tw3 : g.tw16;
        const int tsU = (three ? kTw3N : kTw16N) / NDS;
        const double* win = g.win[L];
        const double norm = sqrt((double)g.NF) / (L + 1.0);
        const int Nw = pixel_count(g, h, L);
        double val[L][Q];
#pragma unroll
        for (int off = 0; off < L; off++)
        {
            const int m = h.jmin + off;
            double2 x[Q];
#pragma unroll
            for (int p = 0; p < Q; p++)
            {
                const int jj = t + 512 * p, j = jj - NT / 2, k = off * (NT / 2) + jj;
                x[p] = make_double2(0.0, 0.0);
                if (jj > 0)
                {
                    double wt = win[j < 0 ? -j : j];
                    if (j == 0 && (m == 0 || m == g.NF)) wt /= 2.0;
                    auto at = [&](const double2* s, int len, int q) { return s[(q % P) * len + q / P]; };
                    const double2 none = make_double2(0.0, 0.0);
                    double2 o[3];
                    if (ch < 2)
                    {
                        band_bin(at(U, NT, k), at(U, NT, NDS - k), none, none, none, wt, o);
                        x[p] = ch == 0 ? o[0] : o[1];
                    }
                    else
                    {
                        band_bin(none, none, at(V, NT / 2, k), at(V, NT / 2, NDS / 2 - k), twU[k * tsU], wt, o);
                        x[p] = o[2];
                    }
                }
            }
            if (off) __syncthreads();  // the last layer's reads
            const SplitFft<NT> f(x, ldsb, g.tw, t);
#pragma unroll
            for (int p = 0; p < Q; p++)
                val[off][p] = pixel_value(f.get(t + 512 * p), NT, g.NF, m, t + 512 * p, norm);
        }
        double* vals = a.values + (size_t)(3 * (size_t)e + ch) * a.vcap;
#pragma unroll
        for (int p = 0; p < Q; p++)
#pragma unroll
            for (int off = 0; off < L; off++)
            {
                const int pos = (t + 512 * p) * L + off;
                if (pos < Nw) vals[pos] = val[off][p];
            }
    });
}

template <int NT>
__global__ void __launch_bounds__(kSumThreads) sum_kernel_big(Geo g, int e0, LayerArgs a,
                                                              const double* __restrict__ scratch)
{
    __shared__ int cnt[kSumThreads / 64 + 1];
    const int e = e0 + blockIdx.x, t = threadIdx.x;
    const Hdr h = load_hdr(scratch + scratch_doubles(g.Norb) * (size_t)e);
    with_layers(h.L, [&](auto l) {
        constexpr int L = decltype(l)::value;
        const int Nw = pixel_list<NT, L, kSumThreads>(g, h, e, a, cnt);
        if (!a.data) return;
        const int* lst = a.list + (size_t)e * a.vcap;
        const double* vals = a.values + (size_t)e * 3 * a.vcap;
        double hh = 0.0, dl = 0.0;
        for (int c = t; c < Nw; c += kSumThreads)
        {
            const double hv[3] = {vals[c], vals[a.vcap + c], vals[2 * a.vcap + c]};
            const int k = Nw == NT * L ? c / L + (h.jmin + c % L) * NT - g.kmin : lst[c];
            PixelData x;
            x.load(a, k);
            pixel_terms(g, a, k, x, hv, hh, dl);
        }
        hh = block_sum<kSumThreads>(hh);
        dl = block_sum<kSumThreads>(dl);
        if (t == 0)
        {
            a.snr[e] = sqrt(hh);
            a.dlogL[e] = dl;
        }
    });
}

template <int NT>
static void launch_big(const Geo& g, int n, const LayerArgs& a, const double* d_scratch, hipStream_t s)
{
    const size_t staged = g.Norb <= kStagedKnots ? sizeof(double) * spline_doubles(g.Norb) : 0;
    for (int e0 = 0; e0 < n; e0 += a.nbig)
    {
        const int m = std::min(a.nbig, n - e0);
        series_kernel_big<NT><<<dim3(NT / kSeriesThreads, m), kSeriesThreads, staged, s>>>(g, e0, a, d_scratch);
        fft_kernel_big<NT><<<dim3(8, m), 512, SplitFft<NT>::kBytes, s>>>(g, e0, a, d_scratch);
        band_kernel_big<NT><<<dim3(3, m), 512, SplitFft<NT>::kBytes, s>>>(g, e0, a, d_scratch);
        sum_kernel_big<NT><<<m, kSumThreads, 0, s>>>(g, e0, a, d_scratch);
    }
}

// ------------------------------------------- K2 for forced layer counts --
//
// Series of up to 32768 samples: U and V with a partner buffer each in a
// global slice per workgroup, transformed by ping-pong Stockham stages through
// L2; each layer's band is inverse-transformed in LDS, one layer at a time.
// Workgroups stride over the templates.

constexpr int kBigLayerThreads = 512;

template <int NT, int L>
__device__ void layer_body_big(const Geo& g, const Hdr& h, int e, const LayerArgs& a, double2* G0, double2* B,
                               int* cnt, const double* __restrict__ scr)
{
    constexpr int NDS = NT * (L + 1);
    constexpr int M = NDS / 2;
    constexpr int NTHR = kBigLayerThreads;
    constexpr int SLOT = kForcedSlot;
    const int tid = threadIdx.x;
    const int N = g.Norb;
    const double* cph = scr + 64;
    const double* ctdi = scr + 64 + 4 * N;
    const double* ds = g.ds[SLOT];
    const int* dsi = g.dsi[SLOT];
    double2* Ua = G0;
    double2* Ub = G0 + NDS;
    double2* Va = G0 + 2 * NDS;
    double2* Vb = Va + M;
    {
#pragma clang fp contract(off)
        const double w0 = PI2 * h.fhet;
        for (int i = tid; i < NDS; i += NTHR)
        {
            const double* e5 = ds + 5 * (size_t)i;
            const double t = e5[0];
            double kdotr = 0.0;
            for (int d = 0; d < 3; d++) kdotr += h.k[d] * e5[1 + d];
            const double tsc = t - kdotr;
            const int j = even_index(tsc, g.ot0, g.ods, N);
            const double phase_ds = spline_at(cph, N, j, tsc - g.ot[j]);
            const double phase_het = w0 * t;
            const int si = dsi[i];
            const double sdx = e5[4];
            double x[3];
            for (int ch = 0; ch < 3; ch++)
            {
                const double* ca = ctdi + 4 * (size_t)N * (2 * ch);
                const double* cp = ctdi + 4 * (size_t)N * (2 * ch + 1);
                const double Amp = spline_at(ca, N, si, sdx);
                double Phase = spline_at(cp, N, si, sdx);
                Phase += phase_ds;
                Phase -= phase_het;
                double sn, c;
                sincos_red(Phase, &sn, &c);
                x[ch] = Amp * c;
            }
            Ua[i] = make_double2(x[0], x[1]);
            if (i & 1) Va[i >> 1].y = x[2];
            else Va[i >> 1].x = x[2];
        }
    }
    __threadfence_block();
    __syncthreads();
    const double2* twU = NDS > kTw16N ? g.tw32 : g.tw16;
    const int tsU = (NDS > kTw16N ? kTw32N : kTw16N) / NDS;
    const double2* U = pingpong_fft<NDS, NTHR>(Ua, Ub, twU, tsU);
    const double2* V = pingpong_fft<M, NTHR>(Va, Vb, twU, tsU * 2);
    int* lst = a.list + (size_t)e * a.vcap;
    {
        constexpr int NC = NT * L;
        constexpr int PER = (NC + NTHR - 1) / NTHR;
        const int c0 = tid * PER;
        int mine = 0;
        for (int c = c0; c < c0 + PER && c < NC; c++)
        {
            const int k = c / L + (h.jmin + c % L) * NT;
            mine += (k >= g.kmin && k < g.kmax);
        }
        int pos = block_exclusive_scan<NTHR>(mine, cnt);
        if (tid == 0) a.nwave[e] = cnt[NTHR / 64];
        for (int c = c0; c < c0 + PER && c < NC; c++)
        {
            const int k = c / L + (h.jmin + c % L) * NT;
            if (k >= g.kmin && k < g.kmax) lst[pos++] = k - g.kmin;
        }
    }
    __syncthreads();
    const int Nw = cnt[NTHR / 64];
    const double* win = g.win[SLOT];
    const double norm = sqrt((double)g.NF) / (L + 1.0);
    double* vals = a.values + (size_t)e * 3 * a.vcap;
    for (int ch = 0; ch < 3; ch++)
        for (int off = 0; off < L; off++)
        {
            const int m = h.jmin + off;
            const int center = (off + 1) * NT / 2;
            for (int jj = tid; jj < NT; jj += NTHR)
            {
                const int j = jj - NT / 2;
                const int idx = center + j;
                double2 v = make_double2(0.0, 0.0);
                if (jj > 0 && idx >= 0 && idx <= NDS / 2)
                {
                    double wt = win[j < 0 ? -j : j];
                    if (j == 0 && (m == 0 || m == g.NF)) wt /= 2.0;
                    const double2 S = spectrum<NDS>(ch, idx, U, V, twU, tsU);
                    v = make_double2(wt * S.x, -(wt * S.y));
                }
                B[jj] = v;
            }
            __syncthreads();
            lds_fft<NT, 1, NTHR>(B, g.tw, kTwN / NT);
            for (int nn = tid; nn < NT; nn += NTHR)
            {
                const double2 r = B[nn];
                const double re = r.x / NT, im = -r.y / NT;
                double val;
                if (m == 0 || m == g.NF) val = (nn % 2 == 0) ? re * M_SQRT2 * norm : 0.0;
                else
                {
                    const int sgn = (m % 2 == 0) ? 1 : -1;
                    val = ((nn + m) % 2 == 0) ? re * norm : sgn * im * norm;
                }
                const int pos = nn * L + off;
                if (pos < Nw) vals[ch * a.vcap + pos] = val;
            }
            __syncthreads();
        }
    if (a.data)
    {
        __threadfence_block();
        __syncthreads();
        double hh = 0.0, dl = 0.0;
        for (int t = tid; t < Nw; t += NTHR)
        {
            const int k = lst[t];
            const double hv[3] = {vals[t], vals[a.vcap + t], vals[2 * a.vcap + t]};
            double C[3][3];
            C[0][0] = a.invC[k];
            C[1][1] = a.invC[(size_t)a.npix + k];
            C[2][2] = a.invC[2 * (size_t)a.npix + k];
            C[0][1] = C[1][0] = a.invC[3 * (size_t)a.npix + k];
            C[0][2] = C[2][0] = a.invC[4 * (size_t)a.npix + k];
            C[1][2] = C[2][1] = a.invC[5 * (size_t)a.npix + k];
            const double d[3] = {a.data[k], a.data[(size_t)a.npix + k], a.data[2 * (size_t)a.npix + k]};
            double th = 0.0, tdh = 0.0, tdd = 0.0;
            for (int p = 0; p < 3; p++)
                for (int q = 0; q < 3; q++)
                {
                    th += hv[p] * hv[q] * C[p][q];
                    tdh += d[p] * hv[q] * C[p][q];
                    tdd += d[p] * d[q] * C[p][q];
                }
            hh += th;
            const int i = (k + g.kmin) % g.NT;
            if (k >= 0 && k < a.npix) dl += (i < g.imin || i > g.imax) ? 0.5 * tdd : tdh - 0.5 * th;
        }
        hh = block_sum<NTHR>(hh);
        dl = block_sum<NTHR>(dl);
        if (tid == 0)
        {
            a.snr[e] = sqrt(hh);
            a.dlogL[e] = dl;
        }
    }
}

template <int NT>
__global__ void __launch_bounds__(kBigLayerThreads) layer_kernel_big(Geo g, int n, LayerArgs a,
                                                                     const double* __restrict__ scratch)
{
    extern __shared__ double2 ldsb[];  // B: one layer's band, NT complex
    __shared__ Hdr H;
    __shared__ int cnt[kBigLayerThreads + 1];
    double2* G0 = a.big + a.bigslice * (size_t)blockIdx.x;
    for (int e = blockIdx.x; e < n; e += gridDim.x)
    {
        const double* scr = scratch + scratch_doubles(g.Norb) * (size_t)e;
        __syncthreads();  // the previous template is done with H, cnt and the slice
        if (threadIdx.x == 0) H = *(const Hdr*)scr;
        __syncthreads();
        const Hdr h = H;
        // the counts of forced_layers_ok
        if (h.L == 7) layer_body_big<NT, 7>(g, h, e, a, G0, ldsb, cnt, scr);
        else if (h.L == 15) layer_body_big<NT, 15>(g, h, e, a, G0, ldsb, cnt, scr);
        else if (h.L == 31) layer_body_big<NT, 31>(g, h, e, a, G0, ldsb, cnt, scr);
        else if (h.L == 63) layer_body_big<NT, 63>(g, h, e, a, G0, ldsb, cnt, scr);
    }
}

// ----------------------------------------------------------- launching --

static int launch_templates(const GeoHost& G, int n, const double* d_params, double* d_scratch,
                            const LayerArgs& a, hipStream_t s)
{
    const Geo& g = G.g;
    if (n <= 0) return GLASS_HIP_OK;
    hipLaunchKernelGGL(hdr_kernel, dim3((n + 255) / 256), dim3(256), 0, s, g, n, d_params, d_scratch);
    hipLaunchKernelGGL(resp_kernel, dim3(n), dim3(kRespThreads), resp_lds_bytes(g.Norb), s, g, n, d_scratch);
    GH_CHECK(hipGetLastError());
    if (g.NT >= 1024 || g.Lf > 0)
    {
        if (!a.big || a.nbig <= 0 || a.bigslice < big_layer_slice(g.NT, g.Lf) || a.vcap < g.NT * (g.Lf > 3 ? g.Lf : 3))
        {
            set_error("wavelet templates: NT = %d (forced layers %d) needs the long-series scratch", g.NT, g.Lf);
            return GLASS_HIP_EINVAL;
        }
        if (g.Lf > 0)
        {
            const int grid = n < a.nbig ? n : a.nbig;
            const size_t lds = sizeof(double2) * (size_t)g.NT;
            if (g.NT == 256)
                layer_kernel_big<256><<<grid, kBigLayerThreads, lds, s>>>(g, n, a, d_scratch);
            else
                layer_kernel_big<512><<<grid, kBigLayerThreads, lds, s>>>(g, n, a, d_scratch);
        }
        else if (g.NT == 1024)
            launch_big<1024>(g, n, a, d_scratch, s);
        else if (g.NT == 2048)
            launch_big<2048>(g, n, a, d_scratch, s);
        else
            launch_big<4096>(g, n, a, d_scratch, s);
    }
    else if (g.NT == 512)
        hipLaunchKernelGGL(layer_kernel<512>, dim3(n), dim3(512), layer_lds_bytes<512>(g.Norb), s, g, n, a, d_scratch);
    else
        hipLaunchKernelGGL(layer_kernel<256>, dim3(n), dim3(256), layer_lds_bytes<256>(g.Norb), s, g, n, a, d_scratch);
    GH_CHECK(hipGetLastError());
    return GLASS_HIP_OK;
}

// The calling thread's long-series scratch for n templates of grid NT
// (nothing below NT = 1024).  Sets the default pixel capacity 3 NT.
static int big_scratch(ThreadCtx* c, int NT, int n, LayerArgs& a)
{
    a.vcap = 3 * NT;
    if (NT < 1024) return GLASS_HIP_OK;
    a.bigslice = big_layer_slice(NT);
    if (int rc = c->dscr.ensure(sizeof(double2) * a.bigslice * (size_t)n)) return rc;
    a.big = (double2*)c->dscr.p;
    a.nbig = n;
    return GLASS_HIP_OK;
}

static int set_lds_limits()
{
    static std::once_flag once;
    static int rc = GLASS_HIP_OK;
    std::call_once(once, [] {
        auto allow_lds = [](auto* f, size_t bytes) {
            return hipFuncSetAttribute((const void*)f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) ==
                   hipSuccess;
        };
        const size_t staged = sizeof(double) * spline_doubles(kStagedKnots);
        if (!allow_lds(resp_kernel, resp_lds_bytes(kMaxKnots)) ||
            !allow_lds(layer_kernel<512>, layer_lds_bytes<512>(kStagedKnots)) ||
            !allow_lds(layer_kernel<256>, layer_lds_bytes<256>(kStagedKnots)) ||
            !allow_lds(series_kernel_big<1024>, staged) || !allow_lds(series_kernel_big<2048>, staged) ||
            !allow_lds(series_kernel_big<4096>, staged) || !allow_lds(fft_kernel_big<4096>, SplitFft<4096>::kBytes) ||
            !allow_lds(band_kernel_big<4096>, SplitFft<4096>::kBytes))
        {
            set_error("hipFuncSetAttribute (dynamic LDS) failed");
            rc = GLASS_HIP_ERUNTIME;
        }
    });
    return rc;
}

// ------------------------------------------------ K3: wavelet Fisher --
//
// ucb_fisher_wavelet (ucb/src/glass_ucb_waveform.c:524-696) before the
// eigensolve, for sources whose 16 perturbed templates (slot 16 s + 2 i:
// params[i] + eps/2, slot + 1: params[i] - eps/2) are already in the
// template buffers.  One workgroup per source: the layer band the 16 pixel
// lists span becomes a dense local window of NT x (band) pixels in scratch;
// per parameter the minus template is scattered into a zeroed window and
// the derivative (h+ - h-)/eps written at the plus template's pixels with
// time index strictly inside (imin, imax); the 36 Fisher elements are then
// reduced over the window with the nine invC terms per pixel.

constexpr int kFishThreads = 256;
constexpr int kFishMaxBand = 6;  // layers the 16 templates of a source may span

struct FishArgs
{
    const int* nwave;      // [16 n]
    const int* list;       // [16 n][3 NT]
    const double* values;  // [16 n][3][3 NT]
    const double* invC;    // plane p of channel pair (a,b) = pmap[3a+b], element k - koff
    long long pstride;     // doubles between planes
    int koff, klen;        // data index of element 0; elements per plane
    int pmap[9];
    int npix;
    double* D;             // scratch [n][8][3][kFishMaxBand NT]
    double* M;             // scratch [n][3][kFishMaxBand NT]
    double* fisher;        // [n][64]
};

__device__ inline double fisher_terms(const double (&u)[3], const double (&v)[3], const double (&C)[9])
{
    // XX, YY, ZZ, XY, XZ, YZ, YX, ZX, ZY (glass_ucb_waveform.c:608-617)
    double f = u[0] * v[0] * C[0];
    f += u[1] * v[1] * C[4];
    f += u[2] * v[2] * C[8];
    f += u[0] * v[1] * C[1];
    f += u[0] * v[2] * C[2];
    f += u[1] * v[2] * C[5];
    f += u[1] * v[0] * C[3];
    f += u[2] * v[0] * C[6];
    f += u[2] * v[1] * C[7];
    return f;
}

__global__ void __launch_bounds__(kFishThreads) fisher_kernel(Geo g, int n, FishArgs a)
{
    const int s = blockIdx.x;
    if (s >= n) return;
    const int NT = g.NT, tid = threadIdx.x, cap = 3 * NT;
    const double invstep = 1. / 1.0e-6;
    __shared__ int band[2];
    __shared__ double red[36][kFishThreads / 64];
    if (tid == 0)
    {
        band[0] = 0x7fffffff;
        band[1] = -1;
    }
    __syncthreads();
    int jlo = 0x7fffffff, jhi = -1;
    for (int t = 0; t < 16; t++)
    {
        const int e = 16 * s + t;
        const int nw = a.nwave[e];
        const int* L = a.list + (size_t)e * cap;
        for (int m = tid; m < nw; m += kFishThreads)
        {
            const int j = (L[m] + g.kmin) / NT;
            jlo = min(jlo, j);
            jhi = max(jhi, j);
        }
    }
    atomicMin(&band[0], jlo);
    atomicMax(&band[1], jhi);
    __syncthreads();
    jlo = band[0];
    jhi = band[1];
    double* F = a.fisher + (size_t)s * 64;
    if (jhi < jlo || jhi - jlo + 1 > kFishMaxBand)
    {
        // no pixels: a zero matrix; a band too wide: NaN marks the failure
        const double v = jhi < jlo ? 0.0 : __builtin_nan("");
        for (int q = tid; q < 64; q += kFishThreads) F[q] = v;
        return;
    }
    const int W = (jhi - jlo + 1) * NT;
    double* D = a.D + (size_t)s * 24 * kFishMaxBand * NT;
    double* M = a.M + (size_t)s * 3 * kFishMaxBand * NT;
    for (int q = tid; q < 24 * W; q += kFishThreads) D[q] = 0.0;
    const int base = jlo * NT;
    for (int i = 0; i < 8; i++)
    {
        const int ep = 16 * s + 2 * i, em = ep + 1;
        for (int q = tid; q < 3 * W; q += kFishThreads) M[q] = 0.0;
        __syncthreads();
        {
            const int nw = a.nwave[em];
            const int* L = a.list + (size_t)em * cap;
            const double* V = a.values + (size_t)em * 3 * cap;
            for (int m = tid; m < nw; m += kFishThreads)
            {
                const int q = L[m] + g.kmin - base;
                for (int ch = 0; ch < 3; ch++) M[ch * W + q] = V[ch * cap + m];
            }
        }
        __syncthreads();
        {
            const int nw = a.nwave[ep];
            const int* L = a.list + (size_t)ep * cap;
            const double* V = a.values + (size_t)ep * 3 * cap;
            for (int m = tid; m < nw; m += kFishThreads)
            {
                const int k = L[m];
                const int it = (k + g.kmin) % NT;
                if (it > g.imin && it < g.imax && k >= 0 && k < a.npix)
                {
                    const int q = k + g.kmin - base;
                    for (int ch = 0; ch < 3; ch++)
                        D[(i * 3 + ch) * W + q] = (V[ch * cap + m] - M[ch * W + q]) * invstep;
                }
            }
        }
        __syncthreads();
    }
    double acc[36];
#pragma unroll
    for (int p = 0; p < 36; p++) acc[p] = 0.0;
    bool miss = false;
    for (int q = tid; q < W; q += kFishThreads)
    {
        const int k = base + q - g.kmin;
        if (k < 0 || k >= a.npix) continue;
        double d[8][3];
        bool any = false;
#pragma unroll
        for (int i = 0; i < 8; i++)
#pragma unroll
            for (int ch = 0; ch < 3; ch++)
            {
                d[i][ch] = D[(i * 3 + ch) * W + q];
                any |= d[i][ch] != 0.0;
            }
        if (!any) continue;
        const int ki = k - a.koff;
        if (ki < 0 || ki >= a.klen)
        {
            miss = true;
            continue;
        }
        double C[9];
#pragma unroll
        for (int p = 0; p < 9; p++) C[p] = a.invC[a.pmap[p] * a.pstride + ki];
        int idx = 0;
#pragma unroll
        for (int i = 0; i < 8; i++)
#pragma unroll
            for (int j = i; j < 8; j++) acc[idx++] += fisher_terms(d[i], d[j], C);
    }
    const int lane = tid & 63, wv = tid >> 6;
#pragma unroll
    for (int p = 0; p < 36; p++)
    {
        const double v = wave_sum(acc[p]);
        if (lane == 0) red[p][wv] = v;
    }
    __shared__ int missed;
    if (tid == 0) missed = 0;
    __syncthreads();
    if (miss) atomicOr(&missed, 1);
    __syncthreads();
    if (tid < 36)
    {
        double f = 0.0;
        for (int w = 0; w < kFishThreads / 64; w++) f += red[tid][w];
        if (f != f) f = 10.0;
        if (missed) f = __builtin_nan("");
        // element tid of the upper triangle, row-major
        int i = 0, r = tid;
        while (r >= 8 - i)
        {
            r -= 8 - i;
            i++;
        }
        const int j = i + r;
        F[i * 8 + j] = f;
        F[j * 8 + i] = f;
    }
}

// The 16 perturbed parameter vectors of each of n sources (slot 16 s + 2 i
// and + 1), as ucb_fisher_wavelet forms them (glass_ucb_waveform.c:556-576).
__global__ void fisher_params_kernel(int n, const double* __restrict__ params, double* __restrict__ out)
{
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= 16 * n) return;
    const int s = q / 16, t = q % 16, i = t / 2, sgn = t % 2;
    const double epsilon = 1.0e-6;
    double* o = out + (size_t)q * 8;
    for (int k = 0; k < 8; k++) o[k] = params[(size_t)s * 8 + k];
    if (sgn == 0) o[i] += epsilon / 2.;
    else o[i] -= epsilon / 2.;
    if (i == 1 || i == 4)
    {
        if (sgn == 0 && o[i] > 1.0) o[i] = 1.0;
        if (sgn == 1 && o[i] < -1.0) o[i] = -1.0;
    }
}

// -------------------------------------------------- geometry cache ------

struct GeoKey
{
    std::vector<double> blob;
    bool operator<(const GeoKey& o) const { return blob < o.blob; }
};

static std::mutex g_geo_mu;
static std::map<std::pair<int, GeoKey>, GeoHost*> g_geo;

static int geo_get(const glass_hip_wdm* w, int Norb, const double* ot, const double* ox, const double* oy,
                   const double* oz, double Tobs, double t0, const GeoHost** out, int Lf = 0)
{
    int rc = check_grid(w, Norb);
    if (rc) return rc;
    if (Lf != 0 && !forced_layers_ok(w->NT, Lf))
        return set_error("wavelet templates: forced layer count %d unsupported at NT = %d (L + 1 a power of two "
                         "from 8 to 64 with NT (L + 1) <= %d, NT = 256 or 512)",
                         Lf, w->NT, kMaxForcedSamples),
               GLASS_HIP_EINVAL;
    int dev = 0;
    GH_CHECK(hipGetDevice(&dev));
    GeoKey key;
    key.blob = {(double)w->NF, (double)w->NT, w->dt, w->df, w->A, (double)w->kmin, (double)w->kmax,
                (double)w->imin, (double)w->imax, Tobs, t0, (double)Norb, (double)Lf};
    key.blob.insert(key.blob.end(), ot, ot + Norb);
    // pos rows: spacecraft i coordinate d at 3i+d
    std::vector<double> pos(9 * (size_t)Norb);
    for (int i = 0; i < 3; i++)
    {
        std::memcpy(pos.data() + (3 * i + 0) * (size_t)Norb, ox + i * (size_t)Norb, sizeof(double) * Norb);
        std::memcpy(pos.data() + (3 * i + 1) * (size_t)Norb, oy + i * (size_t)Norb, sizeof(double) * Norb);
        std::memcpy(pos.data() + (3 * i + 2) * (size_t)Norb, oz + i * (size_t)Norb, sizeof(double) * Norb);
    }
    key.blob.insert(key.blob.end(), pos.begin(), pos.end());
    std::lock_guard<std::mutex> lk(g_geo_mu);
    auto it = g_geo.find({dev, key});
    if (it != g_geo.end())
    {
        *out = it->second;
        return GLASS_HIP_OK;
    }
    if ((rc = set_lds_limits())) return rc;
    GeoHost* G = new GeoHost();
    if ((rc = geo_build(*G, *w, Norb, ot, pos.data(), Tobs, t0, Lf)))
    {
        delete G;
        return rc;
    }
    g_geo[{dev, key}] = G;
    *out = G;
    return GLASS_HIP_OK;
}

}  // namespace wdm
}  // namespace glass

using namespace glass;
using namespace glass::wdm;

// ------------------------------------------------------------- drop-ins --

extern "C" int glass_hip_interpolated_analytic_orbit(const glass_hip_orbit* orbit, double Tobs, double t0, int* Norb,
                                                     double* t, double* x, double* y, double* z)
{
#pragma clang fp contract(off)
    if (!orbit || !Norb || Tobs <= 0) return set_error("interpolated_analytic_orbit: bad arguments"), GLASS_HIP_EINVAL;
    // initialize_interpolated_analytic_orbits (utils/src/glass_lisa.c:271-380)
    const double YEAR = 3.15581497632e7;
    int N = (int)(200 * Tobs / YEAR);
    if (N < 20) N = 20;
    *Norb = N;
    if (!t) return GLASS_HIP_OK;
    if (!x || !y || !z) return set_error("interpolated_analytic_orbit: NULL position array"), GLASS_HIP_EINVAL;
    const double buffer = Tobs / (double)(N - 1);
    const double cadence = (Tobs + 2.0 * buffer) / (double)(N - 1);
    for (int n = 0; n < N; n++)
    {
        const double tn = t0 + n * cadence - buffer;
        double p9[9];
        analytic_positions(*orbit, tn, p9);
        t[n] = tn;
        for (int i = 0; i < 3; i++)
        {
            x[i * (size_t)N + n] = p9[i];
            y[i * (size_t)N + n] = p9[3 + i];
            z[i * (size_t)N + n] = p9[6 + i];
        }
    }
    return GLASS_HIP_OK;
}

extern "C" int glass_hip_ucb_waveform_wavelet(const glass_hip_wdm* w, int Norb, const double* orbit_t,
                                              const double* orbit_x, const double* orbit_y,
                                              const double* orbit_z, double Tobs, double t0,
                                              const double* params, int* wavelet_list, int* Nwavelet, double* X,
                                              double* Y, double* Z)
{
    if (!orbit_t || !orbit_x || !orbit_y || !orbit_z || !params || !wavelet_list || !Nwavelet || !X || !Y || !Z)
        return set_error("ucb_waveform_wavelet: NULL argument"), GLASS_HIP_EINVAL;
    ThreadCtx* c;
    int rc = ctx_get(&c);
    if (rc) return rc;
    const GeoHost* G;
    if ((rc = geo_get(w, Norb, orbit_t, orbit_x, orbit_y, orbit_z, Tobs, t0, &G))) return rc;
    const int NT = w->NT;
    // device: params 8 | scratch | list 3NT ints | values 9NT | nwave
    const size_t nscr = scratch_doubles(Norb);
    const size_t bytes = sizeof(double) * (8 + nscr + 9 * NT) + sizeof(int) * (3 * NT + 4);
    if ((rc = c->dbuf.ensure(bytes)) || (rc = c->hbuf.ensure(bytes))) return rc;
    double* dp = (double*)c->dbuf.p;
    double* dscr = dp + 8;
    double* dval = dscr + nscr;
    int* dlist = (int*)(dval + 9 * NT);
    int* dnw = dlist + 3 * NT;
    double* hp = (double*)c->hbuf.p;
    std::memcpy(hp, params, sizeof(double) * 8);
    GH_CHECK(hipMemcpyAsync(dp, hp, sizeof(double) * 8, hipMemcpyHostToDevice, c->stream));
    LayerArgs a{};
    a.nwave = dnw;
    a.list = dlist;
    a.values = dval;
    if ((rc = big_scratch(c, NT, 1, a))) return rc;
    if ((rc = launch_templates(*G, 1, dp, dscr, a, c->stream))) return rc;
    GH_CHECK(hipMemcpyAsync(hp, dval, sizeof(double) * 9 * NT + sizeof(int) * (3 * NT + 1), hipMemcpyDeviceToHost,
                            c->stream));
    GH_CHECK(hipStreamSynchronize(c->stream));
    const double* hv = hp;
    const int* hl = (const int*)(hp + 9 * NT);
    const int nw = hl[3 * NT];
    *Nwavelet = nw;
    // insert the pixels at their list positions (the caller pre-zeroes, as
    // the reference's callers do)
    for (int t = 0; t < nw; t++)
    {
        wavelet_list[t] = hl[t];
        X[hl[t]] = hv[t];
        Y[hl[t]] = hv[3 * NT + t];
        Z[hl[t]] = hv[6 * NT + t];
    }
    return GLASS_HIP_OK;
}

// ---------------------------------------------------------------- batch --

struct glass_hip_wdm_batch
{
    int device = 0;
    const GeoHost* G = nullptr;
    int npix = 0, max_templates = 0;
    double* data = nullptr;   // 3 x npix
    double* invC = nullptr;   // 6 x npix
    double* scratch = nullptr;
    int* list = nullptr;
    double* values = nullptr;
    int* nwave = nullptr;
    // wavelet Fisher: perturbed parameters [max_templates x 8], derivative
    // and minus-template windows [max_templates / 16 sources] (allocated on
    // first use)
    double* fparams = nullptr;
    double* fD = nullptr;
    double* fM = nullptr;
    // long-series scratch of the NT >= 1024 (or forced layer count) layer
    // kernel: nbig slices of bigslice double2
    double2* big = nullptr;
    int nbig = 0;
    size_t bigslice = 0;
    int vcap = 0;  // pixels per template and channel
    int layers = 0;
};

static int wdm_batch_create(glass_hip_wdm_batch** plan, const glass_hip_wdm* w, int Norb, const double* orbit_t,
                            const double* orbit_x, const double* orbit_y, const double* orbit_z, double Tobs,
                            double t0, const double* data, const double* invC, int npix, int max_templates,
                            int layers)
{
    if (!plan || !orbit_t || !orbit_x || !orbit_y || !orbit_z || !data || !invC)
        return set_error("wdm_batch_create: NULL argument"), GLASS_HIP_EINVAL;
    if (npix <= 0 || max_templates <= 0)
        return set_error("wdm_batch_create: npix=%d max_templates=%d", npix, max_templates), GLASS_HIP_EINVAL;
    ThreadCtx* c;
    int rc = ctx_get(&c);
    if (rc) return rc;
    auto* P = new glass_hip_wdm_batch();
    P->device = c->device;
    auto fail = [&](int r) {
        glass_hip_wdm_batch_destroy(P);
        return r;
    };
    if ((rc = geo_get(w, Norb, orbit_t, orbit_x, orbit_y, orbit_z, Tobs, t0, &P->G, layers))) return fail(rc);
    if (w->kmax - w->kmin != npix)
    {
        set_error("wdm_batch_create: npix = %d but kmax - kmin = %d", npix, w->kmax - w->kmin);
        return fail(GLASS_HIP_EINVAL);
    }
    P->npix = npix;
    P->max_templates = max_templates;
    P->layers = layers;
    const int NT = w->NT;
    P->vcap = NT * (layers > kMaxLayers ? layers : kMaxLayers);
    if (hipMalloc(&P->data, sizeof(double) * 3 * (size_t)npix) != hipSuccess ||
        hipMalloc(&P->invC, sizeof(double) * 6 * (size_t)npix) != hipSuccess ||
        hipMalloc(&P->scratch, sizeof(double) * scratch_doubles(Norb) * (size_t)max_templates) != hipSuccess ||
        hipMalloc(&P->list, sizeof(int) * (size_t)P->vcap * max_templates) != hipSuccess ||
        hipMalloc(&P->values, sizeof(double) * 3 * (size_t)P->vcap * max_templates) != hipSuccess ||
        hipMalloc(&P->nwave, sizeof(int) * (size_t)max_templates) != hipSuccess)
    {
        set_error("wdm_batch_create: device allocation failed");
        return fail(GLASS_HIP_ERUNTIME);
    }
    if (NT >= 1024 || layers > 0)
    {
        // long-series slices of as many templates as are in flight at a time
        int ncu = 0;
        GH_CHECK(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, P->device));
        P->nbig = std::min(max_templates, 2 * std::max(ncu, 1));
        P->bigslice = big_layer_slice(NT, layers);
        if (hipMalloc(&P->big, sizeof(double2) * P->bigslice * (size_t)P->nbig) != hipSuccess)
        {
            set_error("wdm_batch_create: device allocation failed");
            return fail(GLASS_HIP_ERUNTIME);
        }
    }
    if (hipMemcpy(P->data, data, sizeof(double) * 3 * (size_t)npix, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(P->invC, invC, sizeof(double) * 6 * (size_t)npix, hipMemcpyHostToDevice) != hipSuccess)
    {
        set_error("wdm_batch_create: upload failed");
        return fail(GLASS_HIP_ERUNTIME);
    }
    *plan = P;
    return GLASS_HIP_OK;
}

extern "C" int glass_hip_wdm_batch_create(glass_hip_wdm_batch** plan, const glass_hip_wdm* w, int Norb,
                                          const double* orbit_t, const double* orbit_x, const double* orbit_y,
                                          const double* orbit_z, double Tobs, double t0, const double* data,
                                          const double* invC, int npix, int max_templates)
{
    return wdm_batch_create(plan, w, Norb, orbit_t, orbit_x, orbit_y, orbit_z, Tobs, t0, data, invC, npix,
                            max_templates, 0);
}

extern "C" int glass_hip_wdm_batch_create_layers(glass_hip_wdm_batch** plan, const glass_hip_wdm* w, int Norb,
                                                 const double* orbit_t, const double* orbit_x,
                                                 const double* orbit_y, const double* orbit_z, double Tobs,
                                                 double t0, const double* data, const double* invC, int npix,
                                                 int max_templates, int layers)
{
    if (layers <= 0)
        return set_error("wdm_batch_create_layers: layer count %d (use glass_hip_wdm_batch_create for the "
                         "reference's own)",
                         layers),
               GLASS_HIP_EINVAL;
    return wdm_batch_create(plan, w, Norb, orbit_t, orbit_x, orbit_y, orbit_z, Tobs, t0, data, invC, npix,
                            max_templates, layers);
}

extern "C" int glass_hip_wdm_batch_capacity(const glass_hip_wdm_batch* P, int* vcap)
{
    if (!P || !vcap) return set_error("wdm_batch_capacity: NULL argument"), GLASS_HIP_EINVAL;
    *vcap = P->vcap;
    return GLASS_HIP_OK;
}

extern "C" int glass_hip_wdm_batch_destroy(glass_hip_wdm_batch* P)
{
    if (!P) return GLASS_HIP_OK;
    (void)hipSetDevice(P->device);
    for (void* p : {(void*)P->data, (void*)P->invC, (void*)P->scratch, (void*)P->list, (void*)P->values,
                    (void*)P->nwave, (void*)P->fparams, (void*)P->fD, (void*)P->fM, (void*)P->big})
        if (p) (void)hipFree(p);
    delete P;
    return GLASS_HIP_OK;
}

extern "C" int glass_hip_wdm_batch_buffers(glass_hip_wdm_batch* P, int** d_nwave, int** d_list,
                                           double** d_values)
{
    if (!P) return set_error("wdm_batch_buffers: NULL plan"), GLASS_HIP_EINVAL;
    if (d_nwave) *d_nwave = P->nwave;
    if (d_list) *d_list = P->list;
    if (d_values) *d_values = P->values;
    return GLASS_HIP_OK;
}

extern "C" int glass_hip_wdm_batch_eval(glass_hip_wdm_batch* P, int n, const double* d_params, double* d_dlogL,
                                        double* d_snr, void* stream)
{
    if (!P || !d_params || !d_dlogL || !d_snr) return set_error("wdm_batch_eval: NULL argument"), GLASS_HIP_EINVAL;
    if (n < 0 || n > P->max_templates)
        return set_error("wdm_batch_eval: n = %d outside 0..%d", n, P->max_templates), GLASS_HIP_EINVAL;
    GH_CHECK(hipSetDevice(P->device));
    LayerArgs a{};
    a.data = P->data;
    a.invC = P->invC;
    a.npix = P->npix;
    a.nwave = P->nwave;
    a.list = P->list;
    a.values = P->values;
    a.dlogL = d_dlogL;
    a.snr = d_snr;
    a.big = P->big;
    a.nbig = P->nbig;
    a.bigslice = P->bigslice;
    a.vcap = P->vcap;
    return launch_templates(*P->G, n, d_params, P->scratch, a, (hipStream_t)stream);
}

extern "C" int glass_hip_wdm_batch_templates(glass_hip_wdm_batch* P, int n, int* nwave, int* list, double* values)
{
    if (!P || !nwave || !list || !values) return set_error("wdm_batch_templates: NULL argument"), GLASS_HIP_EINVAL;
    if (n < 0 || n > P->max_templates)
        return set_error("wdm_batch_templates: n = %d outside 0..%d", n, P->max_templates), GLASS_HIP_EINVAL;
    GH_CHECK(hipSetDevice(P->device));
    GH_CHECK(hipDeviceSynchronize());
    const size_t vcap = P->vcap;
    GH_CHECK(hipMemcpy(nwave, P->nwave, sizeof(int) * n, hipMemcpyDeviceToHost));
    GH_CHECK(hipMemcpy(list, P->list, sizeof(int) * vcap * n, hipMemcpyDeviceToHost));
    GH_CHECK(hipMemcpy(values, P->values, sizeof(double) * 3 * vcap * n, hipMemcpyDeviceToHost));
    return GLASS_HIP_OK;
}

extern "C" int glass_hip_wdm_batch_scratch(glass_hip_wdm_batch* P, int e, double* out, int nout)
{
    if (!P || !out) return set_error("wdm_batch_scratch: NULL argument"), GLASS_HIP_EINVAL;
    const size_t ns = scratch_doubles(P->G->g.Norb);
    if (e < 0 || e >= P->max_templates || nout < (int)ns)
        return set_error("wdm_batch_scratch: template %d / buffer %d (need %zu)", e, nout, ns), GLASS_HIP_EINVAL;
    GH_CHECK(hipSetDevice(P->device));
    GH_CHECK(hipDeviceSynchronize());
    GH_CHECK(hipMemcpy(out, P->scratch + ns * (size_t)e, sizeof(double) * ns, hipMemcpyDeviceToHost));
    return GLASS_HIP_OK;
}

// ------------------------------------------------------ wavelet Fisher --

extern "C" int glass_hip_ucb_fisher_wavelet(const glass_hip_wdm* w, int Norb, const double* orbit_t,
                                            const double* orbit_x, const double* orbit_y, const double* orbit_z,
                                            double Tobs, double t0, const double* params, const double* invC, int N,
                                            double* fisher)
{
    if (!w || !orbit_t || !orbit_x || !orbit_y || !orbit_z || !params || !invC || !fisher)
        return set_error("ucb_fisher_wavelet: NULL argument"), GLASS_HIP_EINVAL;
    if (N != w->kmax - w->kmin)
        return set_error("ucb_fisher_wavelet: N = %d but kmax - kmin = %d", N, w->kmax - w->kmin), GLASS_HIP_EINVAL;
    ThreadCtx* c;
    int rc = ctx_get(&c);
    if (rc) return rc;
    const GeoHost* G;
    if ((rc = geo_get(w, Norb, orbit_t, orbit_x, orbit_y, orbit_z, Tobs, t0, &G))) return rc;
    const int NT = w->NT;
    // the 16 perturbed parameter vectors (glass_ucb_waveform.c:556-576) and
    // the layer band their templates cover (ucb_wavelet_layers, the rule the
    // template kernels apply)
    double p16[16 * 8];
    int jlo = 1 << 30, jhi = -(1 << 30);
    for (int q = 0; q < 16; q++)
    {
        const int i = q / 2, sgn = q % 2;
        const double epsilon = 1.0e-6;
        double* o = p16 + 8 * q;
        std::memcpy(o, params, sizeof(double) * 8);
        if (sgn == 0) o[i] += epsilon / 2.;
        else o[i] -= epsilon / 2.;
        if (i == 1 || i == 4)
        {
            if (sgn == 0 && o[i] > 1.0) o[i] = 1.0;
            if (sgn == 1 && o[i] < -1.0) o[i] = -1.0;
        }
        int js, jw;
        wavelet_layers(o[0], o[7], Tobs, w->df, w->A, &js, &jw);
        jlo = std::min(jlo, js);
        jhi = std::max(jhi, js + jw - 1);
    }
    const int nb = jhi - jlo + 1;
    if (nb < 1 || nb > kFishMaxBand)
        return set_error("ucb_fisher_wavelet: templates span %d layers (at most %d)", nb, kFishMaxBand),
               GLASS_HIP_EINVAL;
    const int klen = nb * NT, koff = jlo * NT - w->kmin;
    // device: params 128 | scratch | values | invC band 9 klen | D | M | fisher 64 | list | nwave
    const size_t nscr = scratch_doubles(Norb);
    const size_t nD = 24 * (size_t)kFishMaxBand * NT, nM = 3 * (size_t)kFishMaxBand * NT;
    const size_t nd = 128 + 16 * nscr + 16 * 9 * (size_t)NT + 9 * (size_t)klen + nD + nM + 64;
    const size_t bytes = sizeof(double) * nd + sizeof(int) * (16 * 3 * (size_t)NT + 16);
    const size_t hbytes = sizeof(double) * (128 + 9 * (size_t)klen + 64);
    if ((rc = c->dbuf.ensure(bytes)) || (rc = c->hbuf.ensure(hbytes))) return rc;
    double* dp = (double*)c->dbuf.p;
    double* dscr = dp + 128;
    double* dval = dscr + 16 * nscr;
    double* dinv = dval + 16 * 9 * (size_t)NT;
    double* dD = dinv + 9 * (size_t)klen;
    double* dM = dD + nD;
    double* dF = dM + nM;
    int* dlist = (int*)(dF + 64);
    int* dnw = dlist + 16 * 3 * NT;
    double* hp = (double*)c->hbuf.p;
    std::memcpy(hp, p16, sizeof(p16));
    double* hinv = hp + 128;
    for (int p = 0; p < 9; p++)
        for (int q = 0; q < klen; q++)
        {
            const long long k = (long long)koff + q;
            hinv[(size_t)p * klen + q] = (k >= 0 && k < N) ? invC[(size_t)p * N + k] : 0.0;
        }
    GH_CHECK(hipMemcpyAsync(dp, hp, sizeof(double) * 128, hipMemcpyHostToDevice, c->stream));
    GH_CHECK(hipMemcpyAsync(dinv, hinv, sizeof(double) * 9 * klen, hipMemcpyHostToDevice, c->stream));
    LayerArgs a{};
    a.nwave = dnw;
    a.list = dlist;
    a.values = dval;
    if ((rc = big_scratch(c, NT, 16, a))) return rc;
    if ((rc = launch_templates(*G, 16, dp, dscr, a, c->stream))) return rc;
    FishArgs fa{};
    fa.nwave = dnw;
    fa.list = dlist;
    fa.values = dval;
    fa.invC = dinv;
    fa.pstride = klen;
    fa.koff = koff;
    fa.klen = klen;
    for (int p = 0; p < 9; p++) fa.pmap[p] = p;
    fa.npix = N;
    fa.D = dD;
    fa.M = dM;
    fa.fisher = dF;
    hipLaunchKernelGGL(fisher_kernel, dim3(1), dim3(kFishThreads), 0, c->stream, G->g, 1, fa);
    GH_CHECK(hipGetLastError());
    double* hF = hinv + 9 * (size_t)klen;
    GH_CHECK(hipMemcpyAsync(hF, dF, sizeof(double) * 64, hipMemcpyDeviceToHost, c->stream));
    GH_CHECK(hipStreamSynchronize(c->stream));
    for (int q = 0; q < 64; q++)
        if (hF[q] != hF[q]) return set_error("ucb_fisher_wavelet: template pixels outside the invC band"),
                                   GLASS_HIP_ERUNTIME;
    std::memcpy(fisher, hF, sizeof(double) * 64);
    return GLASS_HIP_OK;
}

extern "C" int glass_hip_wdm_batch_fisher(glass_hip_wdm_batch* P, int n, const double* d_params, double* d_fisher,
                                          void* stream)
{
    if (!P || !d_params || !d_fisher) return set_error("wdm_batch_fisher: NULL argument"), GLASS_HIP_EINVAL;
    if (n < 0 || 16LL * n > P->max_templates)
        return set_error("wdm_batch_fisher: n = %d sources need %lld template slots of %d", n, 16LL * n,
                         P->max_templates),
               GLASS_HIP_EINVAL;
    if (P->layers > 0)
        return set_error("wdm_batch_fisher: the plan forces %d layers per template; ucb_fisher_wavelet takes the "
                         "reference's own layer count",
                         P->layers),
               GLASS_HIP_EINVAL;
    if (n == 0) return GLASS_HIP_OK;
    GH_CHECK(hipSetDevice(P->device));
    const int NT = P->G->g.NT;
    const size_t nsrc = (size_t)P->max_templates / 16;
    if (!P->fparams)
    {
        GH_CHECK(hipMalloc(&P->fparams, sizeof(double) * 8 * (size_t)P->max_templates));
        GH_CHECK(hipMalloc(&P->fD, sizeof(double) * 24 * (size_t)kFishMaxBand * NT * nsrc));
        GH_CHECK(hipMalloc(&P->fM, sizeof(double) * 3 * (size_t)kFishMaxBand * NT * nsrc));
    }
    hipStream_t s = (hipStream_t)stream;
    hipLaunchKernelGGL(fisher_params_kernel, dim3((16 * n + 255) / 256), dim3(256), 0, s, n, d_params, P->fparams);
    GH_CHECK(hipGetLastError());
    LayerArgs a{};
    a.nwave = P->nwave;
    a.list = P->list;
    a.values = P->values;
    a.big = P->big;
    a.nbig = P->nbig;
    a.bigslice = P->bigslice;
    a.vcap = P->vcap;
    int rc;
    if ((rc = launch_templates(*P->G, 16 * n, P->fparams, P->scratch, a, s))) return rc;
    FishArgs fa{};
    fa.nwave = P->nwave;
    fa.list = P->list;
    fa.values = P->values;
    fa.invC = P->invC;
    fa.pstride = P->npix;
    fa.koff = 0;
    fa.klen = P->npix;
    const int pm[9] = {0, 3, 4, 3, 1, 5, 4, 5, 2};  // XX YY ZZ XY XZ YZ planes, symmetric
    for (int p = 0; p < 9; p++) fa.pmap[p] = pm[p];
    fa.npix = P->npix;
    fa.D = P->fD;
    fa.M = P->fM;
    fa.fisher = d_fisher;
    hipLaunchKernelGGL(fisher_kernel, dim3(n), dim3(kFishThreads), 0, s, P->G->g, n, fa);
    GH_CHECK(hipGetLastError());
    return GLASS_HIP_OK;
}
