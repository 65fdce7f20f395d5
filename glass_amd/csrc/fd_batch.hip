// fd_batch.hip -- batched, device-resident UCB waveform + delta-logL
// (include/glass_hip_batch.h).
//
// One evaluation = one MCMC proposal of the reference's ucb_mcmc step
// (ucb/src/glass_ucb_sampler.c:139-155): regenerate one source's template
// and evaluate the chain's likelihood and the template's snr.  The sweep is
// a fixed launch sequence with no host synchronisation:
//   1. zero the BW-class counters (a kernel, not a memset: graph-safe),
//      where more than one align workgroup adds to them
//   2. align_kernel: ucb_alignment per proposal on the device; each block
//      histograms its proposals into the 8 BW classes (32..4096) in LDS and
//      reserves its slots with one atomic per class
//   3. per BW class, an eval_kernel<N, NTHR, LOOP> over all proposals,
//      launched with the class's tile (threads per workgroup; one
//      workgroup per proposal slot, or a multiple of the resident capacity
//      striding over the class list), chosen by glass_hip_fd_batch_autotune
//      from the compiled candidates: each workgroup takes an entry of its
//      class list, builds the template in LDS (slow series, 5 FFTs, TDI)
//      and reduces (r|dh) - (dh|dh)/2 over the union of the old and new
//      supports only, reading the chain residual, the group's invC and the
//      source's stored template with coalesced loads.  Up to kFewItems
//      proposals run in one launch for all classes instead.
// The full-window likelihood is therefore never re-read per proposal: the
// algorithmic HBM traffic per proposal is ~144 bytes per template bin, and
// proposals of one chain find their window in L2.
#include <cmath>
#include <cstring>
#include <vector>

#include "../../include/glass_hip_batch.h"
#include "fd_batch_hooks.h"
#include "fd_derivs.h"
#include "fd_waveform.h"
#include "reduce.h"
#include "runtime.h"

namespace glass {

int parse_format(const char* format);

constexpr int kMaxSrcDefault = 8;   // source slots per chain of glass_hip_fd_batch_create
constexpr int kMaxSrcLimit = 64;    // largest max_src of glass_hip_fd_batch_create_ex
constexpr int kNClass = 8;     // BW = 32 << k, k = 0..7 (32..4096)
constexpr int kPosN = 4096;    // positions table samples (largest BW)
constexpr int kAlignOne = 256; // items of one align_kernel workgroup

// Where an item's template meets its chain: written once per item by
// align_kernel, read by scalar loads where the class kernels need it.  A class
// kernel that followed item -> chain -> window -> offsets itself waited for
// five dependent loads before its first sample, and held every pointer in
// scalar registers (spilled to vector lanes) until its last bin.
struct EvalRec
{
    double2* tmpl;      // the source's stored template, 3 rows of cap
    double2* R;         // the chain's residual, 3 rows of W
    const double* iC;   // the window's invC, 6 rows of W
    double logl;        // the chain's logL
    int W, cap;
    int imin;           // first window bin of the new template
    int imin_o, bw_o;   // ... and of the stored one, with its bins
    int cls;            // BW class; kNClass: none holds it, -1: left out
};

struct BatchDev
{
    // groups
    const int* g_qmin;
    const int* g_W;
    const long long* g_off;  // bins before group g
    const double2* data;     // [3][W_g] per group
    const double* invC;      // [6][W_g] per group
    // chains
    const int* c_group;
    const int* c_nsrc;
    const long long* c_roff;  // bins before chain c's residual
    double2* resid;           // [3][W] per chain
    double* logl;             // [C]
    double* sparams;          // [C][8][8]
    int* s_bw;                // [C*8]
    int* s_imin;              // [C*8]
    // templates: chain c's live sources s < c_nsrc[c] hold [3][cap] complex
    // at tmpl + c_toff[c] + 3 s cap, cap = g_cap[group] (the largest BW the
    // window allows: the largest power of two <= W)
    double2* tmpl;
    const int* g_cap;
    const long long* c_toff;
    int bwcap;                // largest g_cap
    int maxsrc;               // source slots per chain in sparams / s_bw / s_imin
    UcbConst* pc;             // per-item template constants, written by align_kernel
    struct EvalRec* rec;      // per-item places, written by align_kernel
    // constants
    double T, t0, L, fstar;
    OrbitReach reach;
    const double* pos;      // positions table, kPosN samples
    const double* pos_soa;  // structure-of-arrays position blocks per series length
    const double2* tw;
    int fmt;
};

// What the class kernels read: kernel arguments, few enough to stay in
// scalar registers.
struct EvalArgs
{
    const UcbConst* pc;
    const EvalRec* rec;
    const double* pos;  // the class's structure-of-arrays positions (coalesced loads)
    const double2* tw;
    double2* stg;       // optional staging of the templates (Items)
    double* logl;
    double* snr;
    int bwcap, fmt;
};

// A scalar load of memory no kernel in flight writes; p uniform.
__device__ __forceinline__ int scalar_load(const int* p)
{
    return *(const __attribute__((address_space(4))) int*)p;
}

// One item's EvalRec by scalar loads (LoadedConst's way).
__device__ __forceinline__ EvalRec load_rec(const EvalRec* p)
{
    static_assert(sizeof(EvalRec) % 8 == 0, "read as 64-bit words");
    auto g = (const __attribute__((address_space(4))) unsigned long long*)uniform_ptr(p);
    asm volatile("" : "+s"(g));
    unsigned long long w[sizeof(EvalRec) / 8];
#pragma unroll
    for (int i = 0; i < (int)(sizeof(EvalRec) / 8); i++) w[i] = g[i];
    EvalRec r;
    __builtin_memcpy(&r, w, sizeof r);
    return r;
}

// Work items: item e refers to entry q = sel ? sel[e] : e of the
// (chain, src, params[8]) arrays.
struct Items
{
    const int* chain;
    const int* src;
    const double* params;
    const int* sel;
    // optional device-side item count (items e >= *dn are left out); lets
    // graph-captured callers size a pass on the device
    const int* dn = nullptr;
    // optional template staging of an eval: item e's X, Y, Z bins go to
    // stg[e * 3 bwcap + ch * N + m] (N its template bins)
    double2* stg = nullptr;
};

__device__ inline int item_q(const Items& it, int e) { return it.sel ? it.sel[e] : e; }
__device__ inline const double* item_params(const Items& it, int e) { return it.params + (size_t)item_q(it, e) * 8; }
__device__ inline int item_chain(const Items& it, int e) { return it.chain[item_q(it, e)]; }
__device__ inline int item_src(const Items& it, int e) { return it.src[item_q(it, e)]; }

__device__ inline int chain_cap(const BatchDev& B, int c) { return B.g_cap[B.c_group[c]]; }
__device__ inline double2* src_tmpl(const BatchDev& B, int c, int s)
{
    return B.tmpl + B.c_toff[c] + (size_t)s * 3 * chain_cap(B, c);
}

__global__ void zero_int_kernel(int* p, int n)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

// ucb_alignment on the device (ucb/src/glass_ucb_waveform.c:727-736) and
// bucketing by BW class.  Class slots are reserved per block (an LDS
// histogram, then one global atomic per class per block) so the class
// counters are not hammered by every item.  Items whose BW falls outside
// the classes are counted in *err (cls_count[kNClass]) and left out.  One
// workgroup alone writes the counts; more add to counts cleared before.
__global__ __launch_bounds__(kAlignOne) void align_kernel(int n, Items it, BatchDev B, int* __restrict__ bw_out,
                                                          int* __restrict__ imin_out, int* __restrict__ cls_count,
                                                          int* __restrict__ cls_list, int cls_stride,
                                                          double* __restrict__ logl_out,
                                                          double* __restrict__ snr_out)
{
    __shared__ int hist[kNClass + 1], base[kNClass + 1];
    if (threadIdx.x <= kNClass) hist[threadIdx.x] = 0;
    __syncthreads();
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    int k = -1, slot = 0;
    // items past the device count, or with a negative source index (a
    // proposal already rejected), are left out of every class list
    if (e < n && (!it.dn || e < *it.dn) && item_src(it, e) >= 0)
    {
        const double* p = item_params(it, e);
        int c = item_chain(it, e);
        int g = B.c_group[c];
        int W = B.g_W[g];
        double f0 = p[0] / B.T;
        double costh = p[1], amp = exp(p[3]);
        double dfdt = p[7] / (B.T * B.T);
        int BW = 2 * ucb_bandwidth(B.L, B.fstar, f0, dfdt, costh, amp, B.T, W);
        int qmin = (int)(f0 * B.T) - BW / 2;
        bw_out[e] = BW;
        imin_out[e] = qmin - B.g_qmin[g];
        // the template constants and places of the class kernels, once per item
        ucb_setup(p, 8, B.T, B.t0, B.L, B.fstar, B.reach, B.pc[e]);
        const int s = item_src(it, e), so = c * B.maxsrc + s;
        EvalRec r;
        r.tmpl = src_tmpl(B, c, s);
        r.R = B.resid + (size_t)B.c_roff[c] * 3;
        r.iC = B.invC + (size_t)B.g_off[g] * 6;
        r.logl = B.logl[c];
        r.W = W;
        r.cap = B.g_cap[g];
        r.imin = qmin - B.g_qmin[g];
        r.imin_o = B.s_imin[so];
        r.bw_o = B.s_bw[so];
        k = 31 - __clz(BW) - 5;  // log2(BW) - 5
        if (BW > B.g_cap[g] || k < 0 || k >= kNClass || (BW & (BW - 1)))
        {
            k = kNClass;
            // no class kernel evaluates this item: a likelihood of -inf
            // (and snr 0) keeps a sampler from ever accepting it
            if (logl_out) logl_out[e] = -INFINITY;
            if (snr_out) snr_out[e] = 0.0;
        }
        r.cls = k;
        B.rec[e] = r;
        slot = atomicAdd(&hist[k], 1);
    }
    else if (e < n)
        B.rec[e].cls = -1;
    __syncthreads();
    if (threadIdx.x <= kNClass)
    {
        const int h = hist[threadIdx.x];
        base[threadIdx.x] = 0;
        if (gridDim.x == 1)
            cls_count[threadIdx.x] = h;
        else if (h)
            base[threadIdx.x] = atomicAdd(&cls_count[threadIdx.x], h);
    }
    __syncthreads();
    if (k >= 0 && k < kNClass) cls_list[k * cls_stride + base[k] + slot] = e;
}

// half of bform(u, u, w): the cross terms once
__device__ inline double qform(const double2* u, const double* w)
{
    auto re = [](double2 a, double2 b) { return a.x * b.x + a.y * b.y; };
    const double d = w[0] * re(u[0], u[0]) + w[1] * re(u[1], u[1]) + w[2] * re(u[2], u[2]);
    const double o = w[3] * re(u[0], u[1]) + w[4] * re(u[0], u[2]) + w[5] * re(u[1], u[2]);
    return d + 2.0 * o;
}

// symmetric 3x3 weighted bilinear form of complex 3-vectors:
// 2 * sum_ab Re(u_a conj v_b) w_ab, w planes XX,YY,ZZ,XY,XZ,YZ
__device__ inline double bform(const double2* u, const double2* v, const double* w)
{
    auto re = [](double2 a, double2 b) { return a.x * b.x + a.y * b.y; };
    double d = w[0] * re(u[0], v[0]) + w[1] * re(u[1], v[1]) + w[2] * re(u[2], v[2]);
    double o = w[3] * (re(u[0], v[1]) + re(u[1], v[0])) + w[4] * (re(u[0], v[2]) + re(u[2], v[0])) +
               w[5] * (re(u[1], v[2]) + re(u[2], v[1]));
    return 2.0 * (d + o);
}

__device__ inline void load_w(const double* __restrict__ iC, int W, int j, double* w)
{
#pragma unroll
    for (int q = 0; q < 6; q++) w[q] = gload(iC + (size_t)q * W + j);
}

// Fused waveform + delta-logL + snr of item e.
template <int N>
__device__ __forceinline__ void eval_item(int e, double2* lds, const EvalArgs& A)
{
    constexpr int NTHR = fd_threads(N);
    // the constants and places by scalar loads where they are used: no LDS
    // copy and no barriers around it, and the slow series reads them as
    // scalar operands
    const LoadedConst k{A.pc + e};
    const EvalRec* rec = A.rec + e;
    // the record's cache line is fetched beside the constants'; held whole
    // from here it would push vector values out of 79 registers
    const int warm = scalar_load(&rec->W);
    double acc = 0.0, s2 = 0.0;
    // the old template's values at bin m, loaded before the bin's transform
    // (their latency, an HBM read per source, overlaps the FFT) where no
    // other series wait in registers meanwhile, else with the bin
    constexpr bool EARLY = fd_series(N) == 1;
    double2 hpre[3];
    auto old_bin = [&](const EvalRec& r, int m) {
        const int j = r.imin + m, mo = j - r.imin_o;
        const bool inold = j >= 0 && j < r.W && mo >= 0 && mo < r.bw_o;
#pragma unroll
        for (int ch = 0; ch < 3; ch++) hpre[ch] = inold ? gload(r.tmpl + ch * r.cap + mo) : make_double2(0.0, 0.0);
    };
    auto pre = [&](int m) {
        asm volatile("" ::"s"(warm));
        if constexpr (EARLY) old_bin(load_rec(rec), m);
    };
    // new-template bins (and the old template where they overlap)
    // no tail barrier: the reduction's barrier below separates this
    // item's last LDS reads from the next item's writes
    fd_link_bins<N, true>(
        k, lds, opaque(A.pos), 0, opaque(A.tw), kTwN / N, pre, [&](int, int m, const double2* dl) {
            double2 v[5];
            fd_tdi<N>(k(), m, A.fmt, dl, v);
            if (A.stg)
#pragma unroll
                for (int ch = 0; ch < 3; ch++) A.stg[(size_t)e * 3 * A.bwcap + ch * N + m] = v[ch];
            const EvalRec r = load_rec(rec);
            if constexpr (!EARLY) old_bin(r, m);
            double wq[6];
            load_w(r.iC, r.W, m, wq);  // snr: template bin m against window bin m
            s2 += qform(v, wq);
            const int j = r.imin + m;
            if (j >= 0 && j < r.W)
            {
                double2 d[3], x[3];
#pragma unroll
                for (int ch = 0; ch < 3; ch++)
                {
                    const double2 h0 = hpre[ch];  // zero outside the old template
                    d[ch] = make_double2(v[ch].x - h0.x, v[ch].y - h0.y);
                    // (r|d) - (d|d)/2 = (r - d/2|d)
                    x[ch] = gload(r.R + (size_t)ch * r.W + j);
                    x[ch].x = fma(-0.5, d[ch].x, x[ch].x);
                    x[ch].y = fma(-0.5, d[ch].y, x[ch].y);
                }
                load_w(r.iC, r.W, j, wq);
                acc += bform(x, d, wq);
            }
        });
    // old-template bins outside the new support: dh = -h_old
    const EvalRec r = load_rec(rec);
    for (int mo = threadIdx.x; mo < r.bw_o; mo += NTHR)
    {
        const int j = r.imin_o + mo;
        if (j < 0 || j >= r.W || (j >= r.imin && j < r.imin + N)) continue;
        double2 d[3], x[3];
        double wq[6];
#pragma unroll
        for (int ch = 0; ch < 3; ch++)
        {
            const double2 h0 = gload(r.tmpl + ch * r.cap + mo);
            d[ch] = make_double2(-h0.x, -h0.y);
            x[ch] = gload(r.R + (size_t)ch * r.W + j);
            x[ch].x = fma(0.5, h0.x, x[ch].x);
            x[ch].y = fma(0.5, h0.y, x[ch].y);
        }
        load_w(r.iC, r.W, j, wq);
        acc += bform(x, d, wq);
    }
    // both sums over the workgroup behind one barrier (block_sum's
    // order: wave sums, then the waves' partials in turn); thread 0
    // writes the logL, thread 1 the snr.  The partials are next written
    // by the following item's reduction, many barriers later.
    constexpr int NW = NTHR / 64;
    __shared__ double part[NW][2];
    const double wa = wave_sum(acc), ws = wave_sum(s2);
    if ((threadIdx.x & 63) == 0)
    {
        part[threadIdx.x >> 6][0] = wa;
        part[threadIdx.x >> 6][1] = ws;
    }
    __syncthreads();
    if (threadIdx.x < 2)
    {
        double q = 0.0;
        for (int i = 0; i < NW; i++) q += part[i][threadIdx.x];
        if (threadIdx.x == 0)
            A.logl[e] = r.logl + q;
        else
            A.snr[e] = sqrt(2.0 * q);
    }
}

// The proposals of one BW class.  LOOP = false: one workgroup per proposal
// slot (grid = proposal count; workgroups past the class count exit at
// once), so the body has no loop and nothing is hoisted across templates.
// LOOP = true: any grid, each workgroup strides over the class list.
// MINW: waves per SIMD the register allocation must allow (1: the
// compiler's choice; more trades register spills for resident waves).
template <int N, int NTHR, bool LOOP, int MINW>
__global__ __launch_bounds__(NTHR) __attribute__((amdgpu_waves_per_eu(MINW, 8))) void eval_kernel(
    const int* __restrict__ list, const int* __restrict__ count, EvalArgs A)
{
    __shared__ double2 lds[FdShape<N>::LDS];
    const int cnt = scalar_load(count);
    if constexpr (LOOP)
    {
        for (int w = blockIdx.x; w < cnt; w += gridDim.x) eval_item<N>(scalar_load(list + w), lds, A);
    }
    else
    {
        if ((int)blockIdx.x < cnt) eval_item<N>(scalar_load(list + blockIdx.x), lds, A);
    }
}

// Compiled launch shapes of the class kernels (tile candidates), default
// first: (class k, template bins N, workgroup threads, waves per SIMD).
#ifndef GH_EVAL_TILES
#define GH_EVAL_TILES(X)                                                                                      \
    X(0, 32, 64, 1) X(1, 64, 64, 1) X(1, 64, 64, 6) X(2, 128, 128, 1) X(3, 256, 256, 1) X(4, 512, 512, 6)    \
    X(4, 512, 512, 1) X(5, 1024, 512, 4) X(5, 1024, 512, 5) X(6, 2048, 1024, 1) X(7, 4096, 1024, 1)
#endif

// Template of each listed item into its source's slot.  LOOP: the grid
// strides over the class list (large rebuilds, where one workgroup per
// item would mostly launch workgroups that exit at once).  use(rec, m, v):
// called with each bin m's X, Y, Z.
template <int N, typename Use>
__device__ __forceinline__ void tmpl_item(int e, double2* lds, const EvalArgs& A, Use&& use)
{
    const LoadedConst k{A.pc + e};
    const EvalRec* rec = A.rec + e;
    fd_link_bins<N, true>(
        k, lds, opaque(A.pos), 0, opaque(A.tw), kTwN / N, [](int) {}, [&](int, int m, const double2* dl) {
            double2 v[5];
            fd_tdi<N>(k(), m, A.fmt, dl, v);
            const EvalRec r = load_rec(rec);
#pragma unroll
            for (int ch = 0; ch < 3; ch++) gstore(r.tmpl + ch * r.cap + m, v[ch]);
            use(r, m, v);
        });
}
constexpr auto kNoUse = [](const EvalRec&, int, const double2*) {};

template <int N, bool LOOP>
__global__ __launch_bounds__(fd_threads(N)) void tmpl_kernel(const int* __restrict__ list, const int* __restrict__ count,
                                                    EvalArgs A)
{
    __shared__ double2 lds[FdShape<N>::LDS];
    const int cnt = scalar_load(count);
    if constexpr (LOOP)
    {
        for (int w = blockIdx.x; w < cnt; w += gridDim.x)
        {
            tmpl_item<N>(scalar_load(list + w), lds, A, kNoUse);
            __syncthreads();  // its last LDS reads before the next item's writes
        }
    }
    else
    {
        if ((int)blockIdx.x < cnt) tmpl_item<N>(scalar_load(list + blockIdx.x), lds, A, kNoUse);
    }
}

// residual += h_old over the stored template's support
__device__ __forceinline__ void accept_add_old(double2* R, int W, const double2* ho, int cap, int io, int bo)
{
    for (int j = max(0, io) + threadIdx.x; j < min(W, io + bo); j += blockDim.x)
        for (int ch = 0; ch < 3; ch++)
        {
            double2 v = R[(size_t)ch * W + j];
            v.x += ho[ch * cap + j - io].x;
            v.y += ho[ch * cap + j - io].y;
            R[(size_t)ch * W + j] = v;
        }
}

// The source of accepted item a takes its parameters and alignment.
__device__ __forceinline__ void accept_source(const Items& it, int a, const BatchDev& B, int bw, int imin,
                                              const double* __restrict__ logl_new)
{
    const int c = item_chain(it, a), so = c * B.maxsrc + item_src(it, a);
    if (threadIdx.x < 8) B.sparams[(size_t)so * 8 + threadIdx.x] = item_params(it, a)[threadIdx.x];
    if (threadIdx.x == 0)
    {
        B.s_bw[so] = bw;
        B.s_imin[so] = imin;
        B.logl[c] = logl_new[item_q(it, a)];
    }
}

// f(integral constant N) of class k's template bins, the classes of at most
// NTHR threads a workgroup; the waves past a class's own threads end, and its
// barriers wait for the others.
template <int NTHR, typename F>
__device__ __forceinline__ void with_class(int k, F&& f)
{
#define GH_K(kk, N)                                                                 \
    case kk:                                                                        \
        if constexpr (fd_threads(N) <= NTHR)                                        \
            if ((int)threadIdx.x < fd_threads(N)) f(std::integral_constant<int, N>()); \
        break;
    switch (k)
    {
        GH_K(0, 32) GH_K(1, 64) GH_K(2, 128) GH_K(3, 256) GH_K(4, 512) GH_K(5, 1024) GH_K(6, 2048) GH_K(7, 4096)
    }
#undef GH_K
}

// A few proposals (one sampler step of some chains): all classes in one
// launch, workgroup e evaluates item e.  The launches bound it: eight over
// four streams with their fork and join took 90 us of host and queue time for
// 20 us of work (evaluate and accept 12 proposals: 309 -> 148 us).  NTHR: the
// largest class's threads.  A.pos: the whole table.
template <int NTHR>
__global__ __launch_bounds__(NTHR) void eval_few_kernel(EvalArgs A)
{
    __shared__ double2 lds[FdShape<NTHR == 512 ? 1024 : 4096>::LDS];
    const int e = blockIdx.x;
    with_class<NTHR>(scalar_load(&A.rec[e].cls), [&](auto n) {
        constexpr int N = decltype(n)::value;
        EvalArgs a = A;
        a.pos += pos_soa_offset(N);
        eval_item<N>(e, lds, a);
    });
}

// ... and accepted: the three passes of the accept kernels below with the
// template between them, workgroup e for item e.  Per bin r + h_old - h_new.
template <int NTHR>
__global__ __launch_bounds__(NTHR) void accept_few_kernel(Items it, BatchDev B, EvalArgs A,
                                                          const double* __restrict__ logl_new)
{
    __shared__ double2 lds[FdShape<NTHR == 512 ? 1024 : 4096>::LDS];
    const int e = blockIdx.x;
    const EvalRec* rec = A.rec + e;
    const int cls = scalar_load(&rec->cls);
    if (cls < 0 || cls >= kNClass) return;  // no class holds it: the source stays
    {
        const EvalRec r = load_rec(rec);
        accept_add_old(r.R, r.W, r.tmpl, r.cap, r.imin_o, r.bw_o);
    }
    __syncthreads();  // before the old template's slot and the residual are written again
    with_class<NTHR>(cls, [&](auto n) {
        constexpr int N = decltype(n)::value;
        EvalArgs a = A;
        a.pos += pos_soa_offset(N);
        tmpl_item<N>(e, lds, a, [&](const EvalRec& r, int m, const double2* v) {
            const int j = r.imin + m;
            if (j < 0 || j >= r.W) return;
#pragma unroll
            for (int ch = 0; ch < 3; ch++)
            {
                double2* R = r.R + (size_t)ch * r.W + j;
                const double2 x = gload(R);
                gstore(R, make_double2(x.x - v[ch].x, x.y - v[ch].y));
            }
        });
        accept_source(it, e, B, N, load_rec(rec).imin, logl_new);
    });
}

// r_c = d_g - sum_s h_cs (add_ucb_model, ucb/src/glass_ucb_model.c:192-232)
// One workgroup per chain (grid = chain count), striding over its window.
__global__ __launch_bounds__(256) void resid_kernel(BatchDev B)
{
    const int c = blockIdx.x;
    const int g = B.c_group[c], W = B.g_W[g], cap = B.g_cap[g];
    const double2* D = B.data + (size_t)B.g_off[g] * 3;
    double2* R = B.resid + (size_t)B.c_roff[c] * 3;
    for (int j = threadIdx.x; j < W; j += blockDim.x)
        for (int ch = 0; ch < 3; ch++)
        {
            double2 v = D[(size_t)ch * W + j];
            for (int s = 0; s < B.c_nsrc[c]; s++)
            {
                const int so = c * B.maxsrc + s;
                const int m = j - B.s_imin[so];
                if (m >= 0 && m < B.s_bw[so])
                {
                    const double2 h = src_tmpl(B, c, s)[ch * cap + m];
                    v.x -= h.x;
                    v.y -= h.y;
                }
            }
            R[(size_t)ch * W + j] = v;
        }
}

// logL_c = -1/2 (r_c | r_c) over the whole window
__global__ __launch_bounds__(256) void chain_logl_kernel(BatchDev B)
{
    const int c = blockIdx.x;
    const int g = B.c_group[c], W = B.g_W[g];
    const double2* R = B.resid + (size_t)B.c_roff[c] * 3;
    const double* iC = B.invC + (size_t)B.g_off[g] * 6;
    double acc = 0.0;
    for (int j = threadIdx.x; j < W; j += 256)
    {
        double2 r[3];
        double w[6];
        for (int ch = 0; ch < 3; ch++) r[ch] = R[(size_t)ch * W + j];
        load_w(iC, W, j, w);
        acc += bform(r, r, w);
    }
    acc = block_sum<256>(acc);
    if (threadIdx.x == 0) B.logl[c] = -0.5 * acc;
}

// Accept, in place: (1) residual += h_old over the old support, (2) the new
// template overwrites the source's slot, (3) residual -= h_new over the new
// support and the source takes its new parameters.  Per bin the residual
// sees r + h_old - h_new in that order.  One workgroup per accepted
// proposal (grid = nacc).
__global__ __launch_bounds__(256) void accept_add_old_kernel(int nacc, Items it, BatchDev B)
{
    const int a = blockIdx.x;
    if (a >= nacc || (it.dn && a >= *it.dn)) return;
    const int c = item_chain(it, a), s = item_src(it, a), so = c * B.maxsrc + s;
    if (s < 0) return;  // left out, as accept_few_kernel and the template kernels do
    const int g = B.c_group[c], W = B.g_W[g], cap = B.g_cap[g];
    accept_add_old(B.resid + (size_t)B.c_roff[c] * 3, W, src_tmpl(B, c, s), cap, B.s_imin[so], B.s_bw[so]);
}

__global__ __launch_bounds__(256) void accept_sub_new_kernel(int nacc, Items it, BatchDev B,
                                                             const int* __restrict__ bw_new,
                                                             const int* __restrict__ imin_new,
                                                             const double* __restrict__ logl_new)
{
    const int a = blockIdx.x;
    if (a >= nacc || (it.dn && a >= *it.dn)) return;
    const int c = item_chain(it, a), s = item_src(it, a);
    if (s < 0) return;
    const int g = B.c_group[c], W = B.g_W[g], cap = B.g_cap[g];
    const int in = imin_new[a], bn = bw_new[a];
    double2* R = B.resid + (size_t)B.c_roff[c] * 3;
    const double2* hn = src_tmpl(B, c, s);
    for (int j = max(0, in) + threadIdx.x; j < min(W, in + bn); j += blockDim.x)
        for (int ch = 0; ch < 3; ch++)
        {
            double2 v = R[(size_t)ch * W + j];
            v.x -= hn[ch * cap + j - in].x;
            v.y -= hn[ch * cap + j - in].y;
            R[(size_t)ch * W + j] = v;
        }
    accept_source(it, a, B, bn, in, logl_new);
}

}  // namespace glass

using namespace glass;

// Exact derivatives of chain sources at their current parameters: per-item
// arguments of the derivative kernels (fd_derivs.h) and BW-class lists
// (BW 32..4096, classes 0..7).  Items outside those (another BW, a chain or
// source index out of range) get NaN outputs.
constexpr int kNDClass = 8;

struct DerivItems
{
    int *pidx, *imin, *W, *tcap;
    long long *roff, *ioff, *toff;
    int* cnt;   // [kNDClass]
    int* list;  // [kNDClass][cap]
};

__global__ __launch_bounds__(256) void derivs_prep_kernel(int n, const int* __restrict__ chain,
                                                          const int* __restrict__ src, int nchain, BatchDev B,
                                                          DerivItems D, int cap, double* __restrict__ outL,
                                                          double* __restrict__ grad, double* __restrict__ fisher)
{
    __shared__ int hist[kNDClass + 1], base[kNDClass + 1];
    if (threadIdx.x <= kNDClass) hist[threadIdx.x] = 0;
    __syncthreads();
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    int k = -1, slot = 0;
    if (e < n)
    {
        const int c = chain[e], s = src[e];
        k = kNDClass;
        if (c >= 0 && c < nchain && s >= 0 && s < B.c_nsrc[c])
        {
            const int so = c * B.maxsrc + s, g = B.c_group[c];
            D.pidx[e] = so;
            D.imin[e] = B.s_imin[so];
            D.W[e] = B.g_W[g];
            D.roff[e] = B.c_roff[c] * 3;
            D.ioff[e] = B.g_off[g] * 6;
            D.toff[e] = B.c_toff[c] + (long long)s * 3 * B.g_cap[g];
            D.tcap[e] = B.g_cap[g];
            const int bw = B.s_bw[so];
            if (bw >= 32 && bw <= 4096 && (bw & (bw - 1)) == 0) k = 31 - __clz(bw) - 5;
        }
        slot = atomicAdd(&hist[k], 1);
    }
    __syncthreads();
    if (threadIdx.x < kNDClass && hist[threadIdx.x]) base[threadIdx.x] = atomicAdd(&D.cnt[threadIdx.x], hist[threadIdx.x]);
    __syncthreads();
    if (k >= 0 && k < kNDClass) D.list[k * cap + base[k] + slot] = e;
    if (k == kNDClass)
    {
        const double nan = __builtin_nan("");
        outL[e] = nan;
        for (int q = 0; q < 8; q++) grad[(size_t)e * 8 + q] = nan;
        for (int q = 0; q < 64; q++) fisher[(size_t)e * 64 + q] = nan;
    }
}

struct glass_hip_fd_batch
{
    int device = 0;
    glass_hip_orbit orbit{};
    int fmt = TDI_SANGRIA;
    double T = 0, t0 = 0;
    int G = 0, C = 0, maxprop = 0, ninit = 0;
    int Wmax = 0;
    std::vector<void*> allocs;
    BatchDev B{};
    // proposal buffers
    int *p_chain = nullptr, *p_src = nullptr;
    double *p_params = nullptr, *p_logl = nullptr, *p_snr = nullptr;
    int *p_bw = nullptr, *p_imin = nullptr;
    int* cls = nullptr;       // [kNClass] counts + [1] error
    int* cls_list = nullptr;  // [kNClass][cap]
    int cls_cap = 0;
    // init items: (chain, src) of every live source, its params gathered
    int *i_chain = nullptr, *i_src = nullptr, *i_slot = nullptr;
    double* i_params = nullptr;
    size_t tmpl_bytes = 0;    // template slots
    int maxsrc = kMaxSrcDefault;
    size_t alloc_bytes = 0;   // device memory the plan holds
    double2* d2048 = nullptr; // BW-2048 derivative scratch, one slice per CU
    double2* d4096 = nullptr; // BW-4096 derivative scratch, one slice per CU
    DerivItems D{};
    int ncu = 0;
    int tgrid[kNClass] = {0};
    glass_hip_tile tile[kNClass] = {};  // launch shape of each class's eval kernel
    bool own_tiles = false;             // the caller chose them (not the default, nor an autotuner's)
    // graph cache
    hipGraph_t graph = nullptr;
    hipGraphExec_t gexec = nullptr;
    int g_nprop = -1;
    // class kernels run concurrently: classes k with k % 4 = 1, 2, 3 go to
    // side streams forked from and joined back into the caller's stream
    // (so graph capture records them as parallel branches)
    hipStream_t side[3] = {};
    hipEvent_t evf = nullptr, evj[3] = {};
    bool concurrent = true;
    // profiling (eager evals only): events around each class kernel
    bool prof = false;
    hipEvent_t ev[kNClass][2] = {};
    double prof_ms[kNClass] = {0};
    int prof_launches[kNClass] = {0};
    int prof_count[kNClass] = {0};
    const void* g_key[5] = {nullptr, nullptr, nullptr, nullptr, nullptr};
    // sweep graph (eval + derivatives)
    hipGraph_t sgraph = nullptr;
    hipGraphExec_t sgexec = nullptr;
    long long s_key[12] = {};
};

template <typename T>
static int dalloc(glass_hip_fd_batch* P, T** p, size_t n)
{
    void* q = nullptr;
    GH_CHECK(hipMalloc(&q, sizeof(T) * (n ? n : 1)));
    P->allocs.push_back(q);
    P->alloc_bytes += sizeof(T) * (n ? n : 1);
    *p = (T*)q;
    return GLASS_HIP_OK;
}

// Workgroups of a class kernel resident per CU, as bounded by LDS (160 KB)
// and by the waves per SIMD the register allocation allows (4 by default,
// `waves` when forced higher).
static int resident_per_cu(int N, int nthr, int waves)
{
    const int lds = (int)sizeof(double2) * kNLink * wave_fft_stride(N < 512 ? N : 512) + 512;
    int per = (160 * 1024) / lds;
    const int wv = 4 * (waves > 4 ? waves : 4) / ((nthr + 63) / 64);
    if (wv < per) per = wv;
    return per < 1 ? 1 : per;
}

// Waves per SIMD of the default tiles (the first candidate of each class):
// 6 at 512 bins, where the compiler's choice of 81 vector registers is one
// above what three workgroups per CU allow (130,042 evaluations 2.60 -> 2.28
// ms), and 4 at 1024, two workgroups per CU (41,400 in 1.77 ms, 2.47 before
// the series were cut to 512 points; with 5 the spills make it 2.36).
constexpr int batch_default_waves(int N) { return N == 512 ? 6 : (N == 1024 ? 4 : 1); }

static bool default_tile(int k, glass_hip_tile t)
{
    const int N = 32 << k;
    return t.nthr == fd_threads(N) && t.gmul == 0 && t.waves == batch_default_waves(N);
}

static int setup_grids(glass_hip_fd_batch* P)
{
    GH_CHECK(hipDeviceGetAttribute(&P->ncu, hipDeviceAttributeMultiprocessorCount, P->device));
    for (int k = 0; k < kNClass; k++)
    {
        const int N = 32 << k;
        P->tgrid[k] = P->ncu * resident_per_cu(N, fd_threads(N), batch_default_waves(N));
        P->tile[k] = glass_hip_tile{fd_threads(N), 0, batch_default_waves(N)};
    }
    return GLASS_HIP_OK;
}

// Grid multipliers of the tile candidates: 0 = one workgroup per proposal
// slot (striding 4 x the resident ones where eval_strides), m > 0 = m x (resident workgroups per CU) x CUs, striding.
constexpr int kGmul[] = {0, 1, 2, 4};
constexpr int kNGmul = sizeof(kGmul) / sizeof(kGmul[0]);

static bool tile_compiled(int k, int nthr, int waves)
{
#define GH_X(kk, N, T, MW) \
    if (k == kk && nthr == T && waves == MW) return true;
    GH_EVAL_TILES(GH_X)
#undef GH_X
    return false;
}

// Shapes of class k that earlier builds compiled (other thread counts of the
// same kernels, and waves that the compiler did not grant or that the default
// has: 128 bins with 6, 256 with 6 and 8, 512 with 8): a caller's saved choice of
// one runs as the default shape with its grid multiplier.
static bool tile_retired(int k, int nthr, int waves)
{
    static constexpr int shape[][3] = {{2, 64, 1},  {2, 128, 6},  {3, 128, 1}, {3, 128, 4}, {3, 256, 5},
                                       {3, 256, 6}, {3, 256, 8},  {4, 256, 1}, {4, 512, 8}, {5, 512, 1},
                                       {5, 1024, 1}, {5, 256, 1}, {6, 512, 1}, {7, 512, 1}};
    for (const auto& x : shape)
        if (x[0] == k && x[1] == nthr && x[2] == waves) return true;
    return false;
}

// Classes whose default grid strides.  The grid cannot know how many of the n
// proposals are in a class; a slot that is not costs the launch of an empty
// workgroup, 0.2 ns of 64 threads and 0.7 ns of 1024 (0.07 and 0.22 ms of
// 327,680), while the striding loop holds more vector registers.  A workgroup a
// slot against striding, of 327,680 mixed proposals: 74 of 32 bins 0.080 / 0.012
// ms, 20,188 of 64 bins 0.108 / 0.049, 23,671 of 2048 bins 3.1 / 2.8, 379 of 4096
// bins 0.46 / 0.17; and where all proposals are of one length: 20,000 of 64 bins 96
// / 99 us, of 2048 2.51 / 2.53 ms, of 4096 5.65 / 5.72.  In between one workgroup a
// slot: of 60,000 of one length 128 bins 266 / 303 us, 256 bins 0.51 / 0.62 ms, 512
// bins 1.04 / 1.19, 1024 bins 2.36 / 2.96; of the mixed proposals 37,679 of 128 bins
// 0.19 / 0.17, 74,247 of 256 bins 0.59 / 0.66, 130,042 of 512 bins 2.33 / 2.53,
// 41,400 of 1024 bins 1.80 / 1.75.
constexpr int kStrideGmul = 4;  // their grid multiplier for gmul 0
constexpr bool eval_strides(int k) { return k < 2 || k > 5; }

static int tile_grid(const glass_hip_fd_batch* P, int k, glass_hip_tile t, int n)
{
    if (t.gmul <= 0 && !eval_strides(k)) return n;
    const long long g = (long long)(t.gmul > 0 ? t.gmul : kStrideGmul) * P->ncu * resident_per_cu(32 << k, t.nthr, t.waves);
    return (int)(g < n ? g : n);
}

static EvalArgs eval_args(const glass_hip_fd_batch* P, int N, const Items& it, double* logl_out, double* snr_out)
{
    const BatchDev& B = P->B;
    return EvalArgs{B.pc, B.rec, B.pos_soa + pos_soa_offset(N), B.tw, it.stg, logl_out, snr_out, B.bwcap, B.fmt};
}

// The class-k eval kernel under tile t over the n proposal slots.
static int launch_eval(glass_hip_fd_batch* P, int k, glass_hip_tile t, int n, const int* list, const int* cnt,
                       const Items& it, double* logl_out, double* snr_out, hipStream_t s)
{
    const int g = tile_grid(P, k, t, n);
#define GH_X(kk, N, T, MW)                                                                                       \
    if (k == kk && t.nthr == T && t.waves == MW)                                                                 \
    {                                                                                                            \
        const EvalArgs A = eval_args(P, N, it, logl_out, snr_out);                                               \
        if (t.gmul > 0 || eval_strides(k))                                                                       \
            eval_kernel<N, T, true, MW><<<g, T, 0, s>>>(list, cnt, A);                                           \
        else                                                                                                     \
            eval_kernel<N, T, eval_strides(kk), MW><<<g, T, 0, s>>>(list, cnt, A);                               \
        return GLASS_HIP_OK;                                                                                     \
    }
    GH_EVAL_TILES(GH_X)
#undef GH_X
    set_error("batch: no compiled tile for class %d with %d threads, %d waves", k, t.nthr, t.waves);
    return GLASS_HIP_EINVAL;
}

// alignment and class lists of the items
static void launch_align(glass_hip_fd_batch* P, int n, const Items& it, double* logl_out, double* snr_out,
                         hipStream_t s)
{
    if (n > kAlignOne) zero_int_kernel<<<1, 64, 0, s>>>(P->cls, kNClass + 1);
    align_kernel<<<(n + kAlignOne - 1) / kAlignOne, kAlignOne, 0, s>>>(n, it, P->B, P->p_bw, P->p_imin, P->cls,
                                                                       P->cls_list, P->cls_cap, logl_out, snr_out);
}

// Items that one launch of all classes takes: four per CU.  Evaluating in one
// launch against eight launches of the classes, eager and replayed as a graph, us:
// 2-year windows of 512 to 4096 bins, 12 proposals 21, 38 / 105, 91; 252 in 40, 44 /
// 114, 100; 1020 in 71, 78 / 119, 127; 2040 in 117, 124 / 145, 127; 1-year windows of
// 96 to 256 bins, 12 in 21, 33 / 72, 62; 1020 in 26, 34 / 78, 67; 2040 in 35, 42 / 77,
// 66.  Templates of 2048 and 4096 bins alone take the same time either way from
// about 1000 on (0.19 and 0.36 us each), where the launches no longer count and the
// class kernels need fewer registers: the line is there.  The class kernels run for
// a caller's own tiles, and evaluate in the profiling mode, which times them; tiles
// that an autotuner chose are for the class kernels of more items and leave the line
// where it is.
constexpr int kFewItems = 1024;
static bool few_items(const glass_hip_fd_batch* P, int n) { return n <= kFewItems && !P->own_tiles; }
static bool few_evals(const glass_hip_fd_batch* P, int n) { return few_items(P, n) && !P->prof; }

// alignment + per-class launches for items; mode 0: eval, 1: templates
static int launch_items(glass_hip_fd_batch* P, int n, const Items& it, int mode, double* logl_out, double* snr_out,
                        hipStream_t s)
{
    if (n <= 0) return GLASS_HIP_OK;
    if (n > P->cls_cap)
    {
        set_error("batch: %d items exceed capacity %d", n, P->cls_cap);
        return GLASS_HIP_EINVAL;
    }
    launch_align(P, n, it, mode == 0 ? logl_out : nullptr, mode == 0 ? snr_out : nullptr, s);
    if (mode == 0 && few_evals(P, n))
    {
        EvalArgs A = eval_args(P, 32, it, logl_out, snr_out);
        A.pos = P->B.pos_soa;
        if (P->B.bwcap <= 1024)
            eval_few_kernel<512><<<n, 512, 0, s>>>(A);
        else
            eval_few_kernel<1024><<<n, 1024, 0, s>>>(A);
        GH_CHECK(hipGetLastError());
        return GLASS_HIP_OK;
    }
    // the per-class timings of the profiling mode need the classes in turn
    const bool par = P->concurrent && !(P->prof && mode == 0);
    if (par)
    {
        GH_CHECK(hipEventRecord(P->evf, s));
        for (int j = 0; j < 3; j++) GH_CHECK(hipStreamWaitEvent(P->side[j], P->evf, 0));
    }
    int lrc = GLASS_HIP_OK;
    for (int k = kNClass - 1; k >= 0; k--)
    {
        const int* list = P->cls_list + (size_t)k * P->cls_cap;
        const int* cnt = P->cls + k;
        const bool pr = P->prof && mode == 0;
        const hipStream_t sk = par && (k & 3) ? P->side[(k & 3) - 1] : s;
        if (pr) GH_CHECK(hipEventRecord(P->ev[k][0], sk));
        if ((32 << k) > P->B.bwcap)
        {
            // align_kernel routes BW above every window's cap to the error
            // count, so this class is empty; its one-workgroup-per-item grid
            // would only launch empty workgroups
        }
        else if (mode == 0)
        {
            if ((lrc = launch_eval(P, k, P->tile[k], n, list, cnt, it, logl_out, snr_out, sk))) break;
        }
        else
        {
            // one workgroup per item, or a striding grid of 4x the resident
            // capacity when the items are many more
            const bool loop = n > 4 * P->tgrid[k];
            const int g = loop ? 4 * P->tgrid[k] : n;
#define GH_L(kk, N)                                                                               \
    case kk:                                                                                      \
        if (loop)                                                                                 \
            tmpl_kernel<N, true><<<g, fd_threads(N), 0, sk>>>(                                    \
                list, cnt, eval_args(P, N, it, nullptr, nullptr));                                \
        else                                                                                      \
            tmpl_kernel<N, false><<<g, fd_threads(N), 0, sk>>>(                                   \
                list, cnt, eval_args(P, N, it, nullptr, nullptr));                                \
        break;
            switch (k)
            {
                GH_L(0, 32) GH_L(1, 64) GH_L(2, 128) GH_L(3, 256) GH_L(4, 512) GH_L(5, 1024) GH_L(6, 2048)
                GH_L(7, 4096)
            }
#undef GH_L
        }
        if (pr) GH_CHECK(hipEventRecord(P->ev[k][1], sk));
    }
    // joined also after a failed launch, so a capture is never left open
    if (par)
        for (int j = 0; j < 3; j++)
        {
            GH_CHECK(hipEventRecord(P->evj[j], P->side[j]));
            GH_CHECK(hipStreamWaitEvent(s, P->evj[j], 0));
        }
    if (lrc) return lrc;
    GH_CHECK(hipGetLastError());
    if (P->prof && mode == 0)
    {
        // synchronous in profiling mode: accumulate the class kernels' times
        int cnt[kNClass + 1];
        GH_CHECK(hipMemcpyAsync(cnt, P->cls, sizeof(int) * (kNClass + 1), hipMemcpyDeviceToHost, s));
        GH_CHECK(hipStreamSynchronize(s));
        for (int k = 0; k < kNClass; k++)
        {
            float ms = 0.f;
            GH_CHECK(hipEventElapsedTime(&ms, P->ev[k][0], P->ev[k][1]));
            P->prof_ms[k] += ms;
            P->prof_launches[k] += 1;
            P->prof_count[k] = cnt[k];
        }
    }
    return GLASS_HIP_OK;
}

// slot alignment from an alignment pass over the init items
__global__ void slot_align_kernel(int n, const int* __restrict__ slot, const int* __restrict__ bw,
                                  const int* __restrict__ imin, int* __restrict__ s_bw, int* __restrict__ s_imin)
{
    int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n) return;
    s_bw[slot[e]] = bw[e];
    s_imin[slot[e]] = imin[e];
}

__global__ void gather_params_kernel(int n, const int* __restrict__ slot, const double* __restrict__ sparams,
                                     double* __restrict__ out)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n * 8) return;
    out[i] = sparams[(size_t)slot[i / 8] * 8 + (i % 8)];
}

static int rebuild(glass_hip_fd_batch* P, hipStream_t s)
{
    const int n = P->ninit;
    gather_params_kernel<<<(n * 8 + 255) / 256, 256, 0, s>>>(n, P->i_slot, P->B.sparams, P->i_params);
    Items it{P->i_chain, P->i_src, P->i_params, nullptr};
    int rc;
    if ((rc = launch_items(P, n, it, 1, nullptr, nullptr, s))) return rc;
    slot_align_kernel<<<(n + 255) / 256, 256, 0, s>>>(n, P->i_slot, P->p_bw, P->p_imin, P->B.s_bw, P->B.s_imin);
    resid_kernel<<<P->C, 256, 0, s>>>(P->B);
    chain_logl_kernel<<<P->C, 256, 0, s>>>(P->B);
    GH_CHECK(hipGetLastError());
    return GLASS_HIP_OK;
}

static int check_err(glass_hip_fd_batch* P, hipStream_t s)
{
    int h = 0;
    GH_CHECK(hipMemcpyAsync(&h, P->cls + kNClass, sizeof(int), hipMemcpyDeviceToHost, s));
    GH_CHECK(hipStreamSynchronize(s));
    if (h)
    {
        set_error("batch: %d items with BW outside 32..%d", h, P->B.bwcap);
        return GLASS_HIP_EINVAL;
    }
    return GLASS_HIP_OK;
}

static int drop_graph(glass_hip_fd_batch* P);

extern "C" int glass_hip_fd_batch_create_ex(glass_hip_fd_batch** plan, const glass_hip_orbit* orbit,
                                            const char* format, double T, double t0, int ngroup,
                                            const int* group_qmin, const int* group_W, const double* data,
                                            const double* invC, int nchain, const int* chain_group,
                                            const int* chain_nsrc, int max_src, const double* src_params,
                                            int max_prop);

extern "C" int glass_hip_fd_batch_create(glass_hip_fd_batch** plan, const glass_hip_orbit* orbit, const char* format,
                                         double T, double t0, int ngroup, const int* group_qmin, const int* group_W,
                                         const double* data, const double* invC, int nchain, const int* chain_group,
                                         const int* chain_nsrc, const double* src_params, int max_prop)
{
    return glass_hip_fd_batch_create_ex(plan, orbit, format, T, t0, ngroup, group_qmin, group_W, data, invC, nchain,
                                        chain_group, chain_nsrc, kMaxSrcDefault, src_params, max_prop);
}

extern "C" int glass_hip_fd_batch_create_ex(glass_hip_fd_batch** plan, const glass_hip_orbit* orbit,
                                            const char* format, double T, double t0, int ngroup,
                                            const int* group_qmin, const int* group_W, const double* data,
                                            const double* invC, int nchain, const int* chain_group,
                                            const int* chain_nsrc, int max_src, const double* src_params,
                                            int max_prop)
{
    if (!plan || !orbit || ngroup <= 0 || nchain <= 0 || max_prop < 0 || !group_qmin || !group_W || !data ||
        !invC || !chain_group || !chain_nsrc || !src_params || max_src < 1 || max_src > kMaxSrcLimit)
    {
        set_error("fd_batch_create: bad arguments (max_src %d: 1..%d)", max_src, kMaxSrcLimit);
        return GLASS_HIP_EINVAL;
    }
    int fmt = parse_format(format);
    if (fmt < 0)
    {
        set_error("Unsupported data format %s", format ? format : "(null)");
        return GLASS_HIP_EINVAL;
    }
    std::vector<long long> goff(ngroup + 1, 0), roff(nchain + 1, 0);
    int Wmax = 0;
    for (int g = 0; g < ngroup; g++)
    {
        // ucb_bandwidth allows 2 * 2^floor(log2(W/2)) bins: at most the
        // 4096-bin template slots (and positions table) for W < 8192
        if (group_W[g] < 32 || group_W[g] >= 2 * kPosN)
        {
            set_error("fd_batch_create: window %d has W=%d outside 32..%d", g, group_W[g], 2 * kPosN - 1);
            return GLASS_HIP_EINVAL;
        }
        goff[g + 1] = goff[g] + group_W[g];
        if (group_W[g] > Wmax) Wmax = group_W[g];
    }
    std::vector<int> ic, is, islot;
    for (int c = 0; c < nchain; c++)
    {
        int g = chain_group[c];
        if (g < 0 || g >= ngroup || chain_nsrc[c] < 0 || chain_nsrc[c] > max_src)
        {
            set_error("fd_batch_create: chain %d has group %d / nsrc %d", c, g, chain_nsrc[c]);
            return GLASS_HIP_EINVAL;
        }
        roff[c + 1] = roff[c] + group_W[g];
        for (int s = 0; s < chain_nsrc[c]; s++)
        {
            ic.push_back(c);
            is.push_back(s);
            islot.push_back(c * max_src + s);
        }
    }
    ThreadCtx* cx;
    int rc;
    if ((rc = ctx_get(&cx))) return rc;
    glass_hip_fd_batch* P = new glass_hip_fd_batch();
    P->orbit = *orbit;
    P->fmt = fmt;
    P->T = T;
    P->t0 = t0;
    P->G = ngroup;
    P->C = nchain;
    P->maxprop = max_prop;
    P->ninit = (int)ic.size();
    P->Wmax = Wmax;
    P->cls_cap = std::max(max_prop, std::max(P->ninit, nchain));
    GH_CHECK(hipGetDevice(&P->device));
    // template slot capacity per window: the largest BW the window allows,
    // 2 * 2^floor(log2(W/2)) <= W (ucb_bandwidth clamps to it), at most 4096
    std::vector<int> gcap(ngroup);
    P->B.bwcap = 32;
    for (int g = 0; g < ngroup; g++)
    {
        int cp = 32;
        while (cp * 2 <= group_W[g] && cp < kPosN) cp *= 2;
        gcap[g] = cp;
        P->B.bwcap = std::max(P->B.bwcap, cp);
    }
    std::vector<long long> toff(nchain + 1, 0);
    for (int c = 0; c < nchain; c++)
        toff[c + 1] = toff[c] + (long long)chain_nsrc[c] * 3 * gcap[chain_group[c]];
    P->tmpl_bytes = sizeof(double2) * (size_t)toff[nchain];
    P->maxsrc = max_src;
    P->B.maxsrc = max_src;
    auto fail = [&](int r) {
        glass_hip_fd_batch_destroy(P);
        return r;
    };
    int *g_qmin, *g_W, *c_group, *c_nsrc, *g_cap;
    long long *g_off, *c_roff, *c_toff;
    double2 *ddata, *resid, *tmpl;
    double *dinvC, *logl, *sparams;
    int *s_bw, *s_imin;
    const size_t nslot = (size_t)nchain * max_src;
    if ((rc = dalloc(P, &g_qmin, ngroup)) || (rc = dalloc(P, &g_W, ngroup)) || (rc = dalloc(P, &g_off, ngroup)) ||
        (rc = dalloc(P, &ddata, 3 * (size_t)goff[ngroup])) || (rc = dalloc(P, &dinvC, 6 * (size_t)goff[ngroup])) ||
        (rc = dalloc(P, &c_group, nchain)) || (rc = dalloc(P, &c_nsrc, nchain)) || (rc = dalloc(P, &c_roff, nchain)) ||
        (rc = dalloc(P, &resid, 3 * (size_t)roff[nchain])) || (rc = dalloc(P, &logl, nchain)) ||
        (rc = dalloc(P, &sparams, nslot * 8)) || (rc = dalloc(P, &s_bw, nslot)) || (rc = dalloc(P, &s_imin, nslot)) ||
        (rc = dalloc(P, &tmpl, (size_t)toff[nchain])) || (rc = dalloc(P, &g_cap, ngroup)) ||
        (rc = dalloc(P, &c_toff, nchain)) ||
        (rc = dalloc(P, &P->p_chain, P->cls_cap)) ||
        (rc = dalloc(P, &P->p_src, P->cls_cap)) || (rc = dalloc(P, &P->p_params, (size_t)P->cls_cap * 8)) ||
        (rc = dalloc(P, &P->p_logl, P->cls_cap)) || (rc = dalloc(P, &P->p_snr, P->cls_cap)) ||
        (rc = dalloc(P, &P->p_bw, P->cls_cap)) || (rc = dalloc(P, &P->p_imin, P->cls_cap)) ||
        (rc = dalloc(P, &P->cls, kNClass + 1)) || (rc = dalloc(P, &P->cls_list, (size_t)kNClass * P->cls_cap)) ||
        (rc = dalloc(P, &P->B.pc, P->cls_cap)) || (rc = dalloc(P, &P->B.rec, P->cls_cap)) ||
        (rc = dalloc(P, &P->i_chain, P->ninit)) || (rc = dalloc(P, &P->i_src, P->ninit)) ||
        (rc = dalloc(P, &P->i_slot, P->ninit)) || (rc = dalloc(P, &P->i_params, (size_t)P->ninit * 8)) ||
        (rc = dalloc(P, &P->D.pidx, P->cls_cap)) || (rc = dalloc(P, &P->D.imin, P->cls_cap)) ||
        (rc = dalloc(P, &P->D.W, P->cls_cap)) || (rc = dalloc(P, &P->D.tcap, P->cls_cap)) ||
        (rc = dalloc(P, &P->D.roff, P->cls_cap)) || (rc = dalloc(P, &P->D.ioff, P->cls_cap)) ||
        (rc = dalloc(P, &P->D.toff, P->cls_cap)) || (rc = dalloc(P, &P->D.cnt, kNDClass)) ||
        (rc = dalloc(P, &P->D.list, (size_t)kNDClass * P->cls_cap)))
        return fail(rc);
    auto up = [&](void* d, const void* h, size_t b) { return hipMemcpy(d, h, b, hipMemcpyHostToDevice); };
    if (up(g_qmin, group_qmin, sizeof(int) * ngroup) || up(g_W, group_W, sizeof(int) * ngroup) ||
        up(g_off, goff.data(), sizeof(long long) * ngroup) || up(ddata, data, 48 * (size_t)goff[ngroup]) ||
        up(dinvC, invC, 48 * (size_t)goff[ngroup]) || up(c_group, chain_group, sizeof(int) * nchain) ||
        up(c_nsrc, chain_nsrc, sizeof(int) * nchain) || up(c_roff, roff.data(), sizeof(long long) * nchain) ||
        up(sparams, src_params, sizeof(double) * nslot * 8) || up(g_cap, gcap.data(), sizeof(int) * ngroup) ||
        up(c_toff, toff.data(), sizeof(long long) * nchain) ||
        (P->ninit && (up(P->i_chain, ic.data(), sizeof(int) * P->ninit) ||
                      up(P->i_src, is.data(), sizeof(int) * P->ninit) ||
                      up(P->i_slot, islot.data(), sizeof(int) * P->ninit))))
    {
        set_error("fd_batch_create: upload failed");
        return fail(GLASS_HIP_ERUNTIME);
    }
    const double *pos, *pos_soa;
    const double2* tw;
    static_assert(kPosN == kPosSoaMax, "one position grid for both tables");
    if ((rc = positions(*orbit, T, t0, kPosN, &pos)) || (rc = positions_soa(*orbit, T, t0, &pos_soa)) ||
        (rc = twiddles(&tw)))
        return fail(rc);
    BatchDev& B = P->B;
    B.g_qmin = g_qmin;
    B.g_W = g_W;
    B.g_off = g_off;
    B.data = ddata;
    B.invC = dinvC;
    B.c_group = c_group;
    B.c_nsrc = c_nsrc;
    B.c_roff = c_roff;
    B.resid = resid;
    B.logl = logl;
    B.sparams = sparams;
    B.s_bw = s_bw;
    B.s_imin = s_imin;
    B.tmpl = tmpl;
    B.g_cap = g_cap;
    B.c_toff = c_toff;
    B.T = T;
    B.t0 = t0;
    B.L = orbit->L;
    B.fstar = orbit->fstar;
    B.reach = analytic_reach(orbit->L, orbit->fstar, orbit->R, T, t0);
    B.pos = pos;
    B.pos_soa = pos_soa;
    B.tw = tw;
    B.fmt = fmt;
    if ((rc = setup_grids(P))) return fail(rc);
    for (int j = 0; j < 3; j++)
        if (hipStreamCreateWithFlags(&P->side[j], hipStreamNonBlocking) != hipSuccess ||
            hipEventCreateWithFlags(&P->evj[j], hipEventDisableTiming) != hipSuccess)
        {
            set_error("fd_batch_create: side streams");
            return fail(GLASS_HIP_ERUNTIME);
        }
    if (hipEventCreateWithFlags(&P->evf, hipEventDisableTiming) != hipSuccess)
    {
        set_error("fd_batch_create: fork event");
        return fail(GLASS_HIP_ERUNTIME);
    }
    if (P->B.bwcap >= 2048 && (rc = dalloc(P, &P->d2048, (size_t)P->ncu * kDeriv2048Scratch))) return fail(rc);
    if (P->B.bwcap >= 4096 && (rc = dalloc(P, &P->d4096, (size_t)P->ncu * kDeriv4096Scratch))) return fail(rc);
    if ((rc = rebuild(P, cx->stream)) || (rc = check_err(P, cx->stream))) return fail(rc);
    *plan = P;
    return GLASS_HIP_OK;
}

extern "C" int glass_hip_fd_batch_destroy(glass_hip_fd_batch* P)
{
    if (!P) return GLASS_HIP_OK;
    (void)hipSetDevice(P->device);
    if (P->gexec) (void)hipGraphExecDestroy(P->gexec);
    for (int k = 0; k < kNClass; k++)
        for (int j = 0; j < 2; j++)
            if (P->ev[k][j]) (void)hipEventDestroy(P->ev[k][j]);
    if (P->graph) (void)hipGraphDestroy(P->graph);
    if (P->sgexec) (void)hipGraphExecDestroy(P->sgexec);
    if (P->sgraph) (void)hipGraphDestroy(P->sgraph);
    (void)hipDeviceSynchronize();
    for (int j = 0; j < 3; j++)
    {
        if (P->side[j]) (void)hipStreamDestroy(P->side[j]);
        if (P->evj[j]) (void)hipEventDestroy(P->evj[j]);
    }
    if (P->evf) (void)hipEventDestroy(P->evf);
    for (void* p : P->allocs) (void)hipFree(p);
    delete P;
    return GLASS_HIP_OK;
}

extern "C" int glass_hip_fd_batch_buffers(glass_hip_fd_batch* P, int** d_chain, int** d_src, double** d_params,
                                          double** d_logL, double** d_snr)
{
    if (!P)
    {
        set_error("fd_batch_buffers: null plan");
        return GLASS_HIP_EINVAL;
    }
    if (d_chain) *d_chain = P->p_chain;
    if (d_src) *d_src = P->p_src;
    if (d_params) *d_params = P->p_params;
    if (d_logL) *d_logL = P->p_logl;
    if (d_snr) *d_snr = P->p_snr;
    return GLASS_HIP_OK;
}

extern "C" int glass_hip_fd_batch_eval(glass_hip_fd_batch* P, int nprop, const int* d_chain, const int* d_src,
                                       const double* d_params, double* d_logL, double* d_snr, void* stream)
{
    if (!P || nprop < 0 || nprop > P->maxprop || (nprop && (!d_chain || !d_src || !d_params || !d_logL || !d_snr)))
    {
        set_error("fd_batch_eval: bad arguments (nprop %d, max %d)", nprop, P ? P->maxprop : 0);
        return GLASS_HIP_EINVAL;
    }
    GH_CHECK(hipSetDevice(P->device));
    Items it{d_chain, d_src, d_params, nullptr};
    return launch_items(P, nprop, it, 0, d_logL, d_snr, (hipStream_t)stream);
}

extern "C" int glass_hip_fd_batch_eval_graph(glass_hip_fd_batch* P, int nprop, const int* d_chain, const int* d_src,
                                             const double* d_params, double* d_logL, double* d_snr, void* stream)
{
    if (!P)
    {
        set_error("fd_batch_eval_graph: null plan");
        return GLASS_HIP_EINVAL;
    }
    GH_CHECK(hipSetDevice(P->device));
    hipStream_t s = (hipStream_t)stream;
    const void* key[5] = {d_chain, d_src, d_params, d_logL, d_snr};
    bool same = P->gexec && P->g_nprop == nprop;
    for (int i = 0; i < 5 && same; i++) same = key[i] == P->g_key[i];
    if (!same)
    {
        if (int rc = drop_graph(P)) return rc;
        // capture on a private stream so the caller's stream may be the
        // legacy default stream
        hipStream_t cs;
        GH_CHECK(hipStreamCreateWithFlags(&cs, hipStreamNonBlocking));
        GH_CHECK(hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal));
        int rc = glass_hip_fd_batch_eval(P, nprop, d_chain, d_src, d_params, d_logL, d_snr, cs);
        hipGraph_t g = nullptr;
        hipError_t ec = hipStreamEndCapture(cs, &g);
        (void)hipStreamDestroy(cs);
        if (rc) return rc;
        if (ec != hipSuccess)
        {
            set_error("graph capture failed: %s", hipGetErrorString(ec));
            return GLASS_HIP_ERUNTIME;
        }
        P->graph = g;
        GH_CHECK(hipGraphInstantiate(&P->gexec, g, nullptr, nullptr, 0));
        P->g_nprop = nprop;
        for (int i = 0; i < 5; i++) P->g_key[i] = key[i];
    }
    GH_CHECK(hipGraphLaunch(P->gexec, s));
    return GLASS_HIP_OK;
}

extern "C" int glass_hip_fd_batch_accept(glass_hip_fd_batch* P, int nacc, const int* d_idx, const int* d_chain,
                                         const int* d_src, const double* d_params, const double* d_logL, void* stream)
{
    if (!P || nacc < 0 || nacc > P->C || (nacc && (!d_idx || !d_chain || !d_src || !d_params || !d_logL)))
    {
        set_error("fd_batch_accept: bad arguments");
        return GLASS_HIP_EINVAL;
    }
    if (nacc == 0) return GLASS_HIP_OK;
    GH_CHECK(hipSetDevice(P->device));
    hipStream_t s = (hipStream_t)stream;
    Items it{d_chain, d_src, d_params, d_idx};
    int rc;
    if (few_items(P, nacc))
    {
        launch_align(P, nacc, it, nullptr, nullptr, s);
        EvalArgs A = eval_args(P, 32, it, nullptr, nullptr);
        A.pos = P->B.pos_soa;
        if (P->B.bwcap <= 1024)
            accept_few_kernel<512><<<nacc, 512, 0, s>>>(it, P->B, A, d_logL);
        else
            accept_few_kernel<1024><<<nacc, 1024, 0, s>>>(it, P->B, A, d_logL);
        GH_CHECK(hipGetLastError());
        return GLASS_HIP_OK;
    }
    accept_add_old_kernel<<<nacc, 256, 0, s>>>(nacc, it, P->B);
    if ((rc = launch_items(P, nacc, it, 1, nullptr, nullptr, s))) return rc;
    accept_sub_new_kernel<<<nacc, 256, 0, s>>>(nacc, it, P->B, P->p_bw, P->p_imin, d_logL);
    GH_CHECK(hipGetLastError());
    return GLASS_HIP_OK;
}

// Accept with templates staged by the eval (Items::stg of that eval): per
// accepted item, residual += h_old over the old support, the staged
// template into the source's slot, residual -= h_new over the new support
// (per bin r + h_old - h_new, as the three-pass accept), new parameters.
// bw_e / imin_e / logl_new are indexed by the eval's item (item_q).  At most
// one accepted item per chain.  One workgroup per accepted item.
__global__ __launch_bounds__(256) void accept_staged_kernel(int nacc, Items it, BatchDev B,
                                                            const double2* __restrict__ stg,
                                                            const int* __restrict__ bw_e,
                                                            const int* __restrict__ imin_e,
                                                            const double* __restrict__ logl_new)
{
    const int a = blockIdx.x;
    if (a >= nacc || (it.dn && a >= *it.dn)) return;
    const int q = item_q(it, a);
    const int c = it.chain[q], s = it.src[q], so = c * B.maxsrc + s;
    const int g = B.c_group[c], W = B.g_W[g], cap = B.g_cap[g];
    const int io = B.s_imin[so], bo = B.s_bw[so];
    const int in = imin_e[q], bn = bw_e[q];
    // an item the alignment left out of every class (BW above the window's
    // slot) has no staged template: never written into the slot
    if (bn > cap || bn > B.bwcap) return;
    double2* R = B.resid + (size_t)B.c_roff[c] * 3;
    double2* h = src_tmpl(B, c, s);
    const double2* hs = stg + (size_t)q * 3 * B.bwcap;
    // one pass over the union of both supports: (r + h_old) - h_new per bin
    const int j0 = max(0, min(io, in)), j1 = min(W, max(io + bo, in + bn));
    for (int j = j0 + threadIdx.x; j < j1; j += blockDim.x)
    {
        const bool o = j >= io && j < io + bo, nw = j >= in && j < in + bn;
        if (!o && !nw) continue;
#pragma unroll
        for (int ch = 0; ch < 3; ch++)
        {
            double2 v = R[(size_t)ch * W + j];
            if (o)
            {
                v.x += h[ch * cap + j - io].x;
                v.y += h[ch * cap + j - io].y;
            }
            if (nw)
            {
                v.x -= hs[ch * bn + j - in].x;
                v.y -= hs[ch * bn + j - in].y;
            }
            R[(size_t)ch * W + j] = v;
        }
    }
    __syncthreads();  // the old template is read before its slot is overwritten
    for (int m = threadIdx.x; m < bn; m += blockDim.x)
#pragma unroll
        for (int ch = 0; ch < 3; ch++) h[ch * cap + m] = hs[ch * bn + m];
    if (threadIdx.x < 8) B.sparams[(size_t)so * 8 + threadIdx.x] = it.params[(size_t)q * 8 + threadIdx.x];
    if (threadIdx.x == 0)
    {
        B.s_bw[so] = bn;
        B.s_imin[so] = in;
        B.logl[c] = logl_new[q];
    }
}

// ------------------------------------------- hooks for the device sampler ---

namespace glass {

FdBatchView fd_batch_view(glass_hip_fd_batch* P)
{
    FdBatchView v{};
    v.device = P->device;
    v.C = P->C;
    v.G = P->G;
    v.maxsrc = P->maxsrc;
    v.ninit = P->ninit;
    v.cap = P->cls_cap;
    v.T = P->T;
    v.c_group = P->B.c_group;
    v.c_nsrc = P->B.c_nsrc;
    v.sparams = P->B.sparams;
    v.logl = P->B.logl;
    v.i_chain = P->i_chain;
    v.i_src = P->i_src;
    return v;
}

int fd_batch_eval_dev(glass_hip_fd_batch* P, int n, const int* chain, const int* src, const double* params,
                      double* logl, double* snr, hipStream_t s, double2* stage)
{
    Items it{chain, src, params, nullptr};
    it.stg = stage;
    return launch_items(P, n, it, 0, logl, snr, s);
}

size_t fd_batch_stage_bytes(glass_hip_fd_batch* P, int n) { return sizeof(double2) * (size_t)n * 3 * P->B.bwcap; }

int fd_batch_accept_staged_dev(glass_hip_fd_batch* P, int nmax, const int* d_n, const int* d_idx, const int* chain,
                               const int* src, const double* params, const double* logl, const double2* stage,
                               hipStream_t s)
{
    if (nmax <= 0) return GLASS_HIP_OK;
    if (nmax > P->C || nmax > P->cls_cap || !stage)
    {
        set_error("batch accept: %d items exceed the plan (%d chains, capacity %d) or no staged templates", nmax,
                  P->C, P->cls_cap);
        return GLASS_HIP_EINVAL;
    }
    Items it{chain, src, params, d_idx, d_n};
    accept_staged_kernel<<<nmax, 256, 0, s>>>(nmax, it, P->B, stage, P->p_bw, P->p_imin, logl);
    GH_CHECK(hipGetLastError());
    return GLASS_HIP_OK;
}

}  // namespace glass

extern "C" int glass_hip_fd_batch_refresh(glass_hip_fd_batch* P, void* stream)
{
    if (!P)
    {
        set_error("fd_batch_refresh: null plan");
        return GLASS_HIP_EINVAL;
    }
    GH_CHECK(hipSetDevice(P->device));
    return rebuild(P, (hipStream_t)stream);
}

extern "C" int glass_hip_fd_batch_set_concurrent(glass_hip_fd_batch* P, int on)
{
    if (!P)
    {
        set_error("fd_batch_set_concurrent: null plan");
        return GLASS_HIP_EINVAL;
    }
    if (int rc = drop_graph(P)) return rc;
    P->concurrent = on != 0;
    return GLASS_HIP_OK;
}

extern "C" int glass_hip_fd_batch_profile(glass_hip_fd_batch* P, int on)
{
    if (!P)
    {
        set_error("fd_batch_profile: null plan");
        return GLASS_HIP_EINVAL;
    }
    GH_CHECK(hipSetDevice(P->device));
    if (on && !P->ev[0][0])
        for (int k = 0; k < kNClass; k++)
            for (int j = 0; j < 2; j++) GH_CHECK(hipEventCreate(&P->ev[k][j]));
    P->prof = on != 0;
    for (int k = 0; k < kNClass; k++)
    {
        P->prof_ms[k] = 0;
        P->prof_launches[k] = 0;
        P->prof_count[k] = 0;
    }
    return GLASS_HIP_OK;
}

extern "C" int glass_hip_fd_batch_profile_read(glass_hip_fd_batch* P, double* ms, int* launches, int* count)
{
    if (!P || !ms || !launches || !count)
    {
        set_error("fd_batch_profile_read: bad arguments");
        return GLASS_HIP_EINVAL;
    }
    for (int k = 0; k < kNClass; k++)
    {
        ms[k] = P->prof_ms[k];
        launches[k] = P->prof_launches[k];
        count[k] = P->prof_count[k];
    }
    return GLASS_HIP_OK;
}

extern "C" int glass_hip_fd_batch_state(glass_hip_fd_batch* P, double* logL, double* src_params)
{
    if (!P || !logL)
    {
        set_error("fd_batch_state: bad arguments");
        return GLASS_HIP_EINVAL;
    }
    GH_CHECK(hipSetDevice(P->device));
    GH_CHECK(hipDeviceSynchronize());
    int rc;
    if ((rc = check_err(P, nullptr))) return rc;
    GH_CHECK(hipMemcpy(logL, P->B.logl, sizeof(double) * P->C, hipMemcpyDeviceToHost));
    if (src_params)
        GH_CHECK(hipMemcpy(src_params, P->B.sparams, sizeof(double) * P->C * P->maxsrc * 8, hipMemcpyDeviceToHost));
    return GLASS_HIP_OK;
}

// ------------------------------------------------------------- tiles ---

static int drop_graph(glass_hip_fd_batch* P)
{
    if (P->gexec) GH_CHECK(hipGraphExecDestroy(P->gexec));
    if (P->graph) GH_CHECK(hipGraphDestroy(P->graph));
    if (P->sgexec) GH_CHECK(hipGraphExecDestroy(P->sgexec));
    if (P->sgraph) GH_CHECK(hipGraphDestroy(P->sgraph));
    P->gexec = nullptr;
    P->graph = nullptr;
    P->sgexec = nullptr;
    P->sgraph = nullptr;
    P->g_nprop = -1;
    return GLASS_HIP_OK;
}

extern "C" int glass_hip_fd_batch_tile_candidates(int k, glass_hip_tile* out, int max, int* n)
{
    if (k < 0 || k >= kNClass || !n || (max > 0 && !out))
    {
        set_error("fd_batch_tile_candidates: bad arguments");
        return GLASS_HIP_EINVAL;
    }
    int c = 0;
#define GH_X(kk, N, T, MW)                                          \
    if (k == kk)                                                    \
        for (int m = 0; m < kNGmul; m++, c++)                       \
            if (c < max) out[c] = glass_hip_tile{T, kGmul[m], MW};
    GH_EVAL_TILES(GH_X)
#undef GH_X
    *n = c;
    return GLASS_HIP_OK;
}

extern "C" int glass_hip_fd_batch_get_tiles(glass_hip_fd_batch* P, glass_hip_tile* tiles)
{
    if (!P || !tiles)
    {
        set_error("fd_batch_get_tiles: bad arguments");
        return GLASS_HIP_EINVAL;
    }
    for (int k = 0; k < kNClass; k++) tiles[k] = P->tile[k];
    return GLASS_HIP_OK;
}

static int set_tiles(glass_hip_fd_batch* P, const glass_hip_tile* tiles, bool tuned)
{
    if (!P || !tiles)
    {
        set_error("fd_batch_set_tiles: bad arguments");
        return GLASS_HIP_EINVAL;
    }
    glass_hip_tile use[kNClass];
    bool own = false;
    for (int k = 0; k < kNClass; k++)
    {
        use[k] = tiles[k];
        if (tile_retired(k, use[k].nthr, use[k].waves))
            use[k] = glass_hip_tile{fd_threads(32 << k), tiles[k].gmul, batch_default_waves(32 << k)};
        if (!tile_compiled(k, use[k].nthr, use[k].waves) || use[k].gmul < 0 || use[k].gmul > 64)
        {
            set_error("fd_batch_set_tiles: class %d (BW %d): no compiled tile with %d threads, %d waves, grid x%d",
                      k, 32 << k, tiles[k].nthr, tiles[k].waves, tiles[k].gmul);
            return GLASS_HIP_EINVAL;
        }
    }
    GH_CHECK(hipSetDevice(P->device));
    if (int rc = drop_graph(P)) return rc;
    for (int k = 0; k < kNClass; k++)
    {
        P->tile[k] = use[k];
        own = own || !default_tile(k, use[k]);
    }
    P->own_tiles = own && !tuned;
    return GLASS_HIP_OK;
}

extern "C" int glass_hip_fd_batch_set_tiles(glass_hip_fd_batch* P, const glass_hip_tile* tiles)
{
    return set_tiles(P, tiles, false);
}

extern "C" int glass_hip_fd_batch_set_tuned_tiles(glass_hip_fd_batch* P, const glass_hip_tile* tiles)
{
    return set_tiles(P, tiles, true);
}

extern "C" int glass_hip_fd_batch_one_launch(const glass_hip_fd_batch* P, int n)
{
    return P && n > 0 && few_evals(P, n);
}

extern "C" int glass_hip_fd_batch_autotune(glass_hip_fd_batch* P, int nprop, const int* d_chain, const int* d_src,
                                           const double* d_params, int reps, glass_hip_tile* best,
                                           double* best_ms, void* stream)
{
    if (!P || nprop <= 0 || nprop > P->maxprop || !d_chain || !d_src || !d_params || reps < 1)
    {
        set_error("fd_batch_autotune: bad arguments (nprop %d, max %d, reps %d)", nprop, P ? P->maxprop : 0, reps);
        return GLASS_HIP_EINVAL;
    }
    GH_CHECK(hipSetDevice(P->device));
    hipStream_t s = (hipStream_t)stream;
    Items it{d_chain, d_src, d_params, nullptr};
    // class lists of these proposals, as an eval builds them
    launch_align(P, nprop, it, nullptr, nullptr, s);
    GH_CHECK(hipGetLastError());
    int cnt[kNClass + 1];
    GH_CHECK(hipMemcpyAsync(cnt, P->cls, sizeof(cnt), hipMemcpyDeviceToHost, s));
    GH_CHECK(hipStreamSynchronize(s));
    if (cnt[kNClass])
    {
        set_error("fd_batch_autotune: %d proposals with BW outside 32..%d", cnt[kNClass], P->B.bwcap);
        return GLASS_HIP_EINVAL;
    }
    if (int rc = drop_graph(P)) return rc;
    P->own_tiles = false;
    hipEvent_t e0, e1;
    GH_CHECK(hipEventCreate(&e0));
    GH_CHECK(hipEventCreate(&e1));
    int rc = GLASS_HIP_OK;
    for (int k = 0; k < kNClass && !rc; k++)
    {
        double bms = 0.0;
        if (cnt[k] > 0)
        {
            glass_hip_tile cand[64];
            int nc = 0;
            glass_hip_fd_batch_tile_candidates(k, cand, 64, &nc);
            const int* list = P->cls_list + (size_t)k * P->cls_cap;
            const int* cntp = P->cls + k;
            bms = 1e300;
            for (int c = 0; c < nc && c < 64 && !rc; c++)
            {
                // the same launch as gmul 0
                if (eval_strides(k) && cand[c].gmul == kStrideGmul) continue;
                // one untimed launch, then reps timed ones; results go to
                // the plan's own logL/snr buffers
                if ((rc = launch_eval(P, k, cand[c], nprop, list, cntp, it, P->p_logl, P->p_snr, s))) break;
                if (hipEventRecord(e0, s) != hipSuccess) rc = GLASS_HIP_ERUNTIME;
                for (int r = 0; r < reps && !rc; r++)
                    rc = launch_eval(P, k, cand[c], nprop, list, cntp, it, P->p_logl, P->p_snr, s);
                float ms = 0.f;
                if (!rc && (hipEventRecord(e1, s) != hipSuccess || hipEventSynchronize(e1) != hipSuccess ||
                            hipEventElapsedTime(&ms, e0, e1) != hipSuccess))
                {
                    set_error("fd_batch_autotune: timing failed");
                    rc = GLASS_HIP_ERUNTIME;
                }
                if (!rc && ms / reps < bms)
                {
                    bms = ms / reps;
                    P->tile[k] = cand[c];
                }
            }
        }
        if (best) best[k] = P->tile[k];
        if (best_ms) best_ms[k] = bms;
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (!rc && hipGetLastError() != hipSuccess) rc = GLASS_HIP_ERUNTIME;
    return rc;
}

// ------------------------------------------------------- derivatives ---

extern "C" int glass_hip_fd_batch_derivs(glass_hip_fd_batch* P, int n, const int* d_chain, const int* d_src,
                                         double* d_logL, double* d_grad, double* d_fisher, void* stream)
{
    if (!P || n < 0 || n > P->cls_cap || (n && (!d_chain || !d_src || !d_logL || !d_grad || !d_fisher)))
    {
        set_error("fd_batch_derivs: bad arguments (n %d, capacity %d)", n, P ? P->cls_cap : 0);
        return GLASS_HIP_EINVAL;
    }
    if (n == 0) return GLASS_HIP_OK;
    GH_CHECK(hipSetDevice(P->device));
    hipStream_t s = (hipStream_t)stream;
    zero_int_kernel<<<1, 64, 0, s>>>(P->D.cnt, kNDClass);
    derivs_prep_kernel<<<(n + 255) / 256, 256, 0, s>>>(n, d_chain, d_src, P->C, P->B, P->D, P->cls_cap, d_logL,
                                                       d_grad, d_fisher);
    GH_CHECK(hipGetLastError());
    const BatchDev& B = P->B;
    DerivArgs A{};
    A.params = B.sparams;
    A.pidx = P->D.pidx;
    A.imin = P->D.imin;
    A.iW = P->D.W;
    A.resid = B.resid;
    A.iroff = P->D.roff;
    A.invC = B.invC;
    A.iioff = P->D.ioff;
    A.tadd = B.tmpl;
    A.taddoff = P->D.toff;
    A.taddcap = P->D.tcap;
    A.mode = 0;
    A.T = B.T;
    A.t0 = B.t0;
    A.L = B.L;
    A.fstar = B.fstar;
    A.reach = B.reach;
    A.pos = B.pos;
    A.tw = B.tw;
    A.fmt = B.fmt;
    A.outL = d_logL;
    A.grad = d_grad;
    A.fisher = d_fisher;
    // the classes on the plan's side streams as in launch_items (k % 4)
    const bool par = P->concurrent;
    if (par)
    {
        GH_CHECK(hipEventRecord(P->evf, s));
        for (int j = 0; j < 3; j++) GH_CHECK(hipStreamWaitEvent(P->side[j], P->evf, 0));
    }
    int lrc = GLASS_HIP_OK;
    for (int k = kNDClass - 1; k >= 0 && !lrc; k--)
    {
        const hipStream_t sk = par && (k & 3) ? P->side[(k & 3) - 1] : s;
        A.list = P->D.list + (size_t)k * P->cls_cap;
        A.count = P->D.cnt + k;
        if (32 << k == 2048)
        {
            // BW 2048 only occurs when some window allows it (then d2048 exists)
            if (P->d2048) lrc = launch_derivs_2048(A, std::min(n, P->ncu), P->d2048, sk);
        }
        else if (32 << k == 4096)
        {
            if (P->d4096) lrc = launch_derivs_4096(A, std::min(n, P->ncu), P->d4096, sk);
        }
        else
            lrc = launch_derivs(32 << k, A, n, sk);
    }
    if (par)
        for (int j = 0; j < 3; j++)
        {
            GH_CHECK(hipEventRecord(P->evj[j], P->side[j]));
            GH_CHECK(hipStreamWaitEvent(s, P->evj[j], 0));
        }
    return lrc;
}

extern "C" int glass_hip_fd_batch_sweep_graph(glass_hip_fd_batch* P, int nprop, const int* d_chain, const int* d_src,
                                              const double* d_params, double* d_logL, double* d_snr, int nder,
                                              const int* d_dchain, const int* d_dsrc, double* d_dlogL,
                                              double* d_grad, double* d_fisher, void* stream)
{
    if (!P)
    {
        set_error("fd_batch_sweep_graph: null plan");
        return GLASS_HIP_EINVAL;
    }
    GH_CHECK(hipSetDevice(P->device));
    const long long key[12] = {nprop, (long long)d_chain, (long long)d_src, (long long)d_params,
                               (long long)d_logL, (long long)d_snr, nder, (long long)d_dchain,
                               (long long)d_dsrc, (long long)d_dlogL, (long long)d_grad, (long long)d_fisher};
    bool same = P->sgexec != nullptr;
    for (int i = 0; i < 12 && same; i++) same = key[i] == P->s_key[i];
    if (!same)
    {
        if (P->sgexec) GH_CHECK(hipGraphExecDestroy(P->sgexec));
        if (P->sgraph) GH_CHECK(hipGraphDestroy(P->sgraph));
        P->sgexec = nullptr;
        P->sgraph = nullptr;
        hipStream_t cs;
        GH_CHECK(hipStreamCreateWithFlags(&cs, hipStreamNonBlocking));
        GH_CHECK(hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal));
        int rc = glass_hip_fd_batch_eval(P, nprop, d_chain, d_src, d_params, d_logL, d_snr, cs);
        if (!rc) rc = glass_hip_fd_batch_derivs(P, nder, d_dchain, d_dsrc, d_dlogL, d_grad, d_fisher, cs);
        hipGraph_t g = nullptr;
        hipError_t ec = hipStreamEndCapture(cs, &g);
        (void)hipStreamDestroy(cs);
        if (rc)
        {
            if (g) (void)hipGraphDestroy(g);
            return rc;
        }
        if (ec != hipSuccess)
        {
            set_error("sweep graph capture failed: %s", hipGetErrorString(ec));
            return GLASS_HIP_ERUNTIME;
        }
        P->sgraph = g;
        GH_CHECK(hipGraphInstantiate(&P->sgexec, g, nullptr, nullptr, 0));
        for (int i = 0; i < 12; i++) P->s_key[i] = key[i];
    }
    GH_CHECK(hipGraphLaunch(P->sgexec, (hipStream_t)stream));
    return GLASS_HIP_OK;
}

extern "C" int glass_hip_fd_batch_memory(glass_hip_fd_batch* P, long long* template_bytes, long long* total_bytes)
{
    if (!P)
    {
        set_error("fd_batch_memory: null plan");
        return GLASS_HIP_EINVAL;
    }
    if (template_bytes) *template_bytes = (long long)P->tmpl_bytes;
    if (total_bytes) *total_bytes = (long long)P->alloc_bytes;
    return GLASS_HIP_OK;
}
