// reduce.h -- deterministic FP64 block reductions (DPP within a wave, then LDS).
#pragma once
#include <hip/hip_runtime.h>

namespace glass {

// v + (v of the lane a DPP control names, 0 where it names none).
template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ double dpp_add(double v)
{
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWS, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWS, 0xf, false);
    return v + __hiloint2double(hi, lo);
}

// Sum over the wave, the same in every lane: shifts within the rows of 16
// lanes, then the rows' sums handed on (18 vector instructions, no LDS; the
// six exchanges through LDS they replace waited for each other).
__device__ inline double wave_sum(double v)
{
    v = dpp_add<0x111>(v);       // row_shr:1
    v = dpp_add<0x112>(v);       // row_shr:2
    v = dpp_add<0x114>(v);       // row_shr:4
    v = dpp_add<0x118>(v);       // row_shr:8: lane 15 of each row has its sum
    v = dpp_add<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
    v = dpp_add<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
    const int lo = __builtin_amdgcn_readlane(__double2loint(v), 63);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(v), 63);
    return __hiloint2double(hi, lo);
}

// K sums over the block at once: each wave's tree sum of each value, one
// barrier, then thread k adds the waves' partials of value k in order into
// out[k] (LDS or global); ends with a barrier.  The per-value order is
// block_sum's, so the results are the same as K separate block_sum calls.
template <int NTHR, int K>
__device__ inline void block_sum_many(const double (&v)[K], double* out)
{
    static_assert(NTHR % 64 == 0 && K <= NTHR, "wave64 workgroups, K <= threads");
    __shared__ double part[NTHR / 64][K];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < K; k++)
    {
        const double x = wave_sum(v[k]);
        if (lane == 0) part[w][k] = x;
    }
    __syncthreads();
    if (threadIdx.x < K)
    {
        double r = 0.0;
        for (int i = 0; i < NTHR / 64; i++) r += part[i][threadIdx.x];
        out[threadIdx.x] = r;
    }
    __syncthreads();
}

// K sums over the block through LDS: CH values at a time are laid out one row
// per value (rows a double apart in banks), each thread adds CH entries of one
// row, the lanes of a row add up by exchanges and the waves' partials in order
// into out[K].  170 instructions a thread for 48 values, where wave_sum takes
// 960.  Fixed order.  buf: CH (NTHR + 1) doubles, whose readers have passed a
// barrier; ends with one.
template <int NTHR, int CH, int K, int KV>
__device__ __forceinline__ void block_sum_rows(const double (&v)[KV], double* buf, double* out)
{
    static_assert(NTHR % 64 == 0 && 64 % CH == 0 && K <= KV, "whole chunks of a wave");
    constexpr int NW = NTHR / 64, ROW = NTHR + 1, KP = (K + CH - 1) / CH * CH;
    __shared__ double part[KP][NW];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
#pragma unroll
    for (int k0 = 0; k0 < K; k0 += CH)
    {
        if (k0) __syncthreads();
#pragma unroll
        for (int i = 0; i < CH; i++)
            if (k0 + i < K) buf[i * ROW + t] = v[k0 + i];
        __syncthreads();
        const int i = t % CH;  // a row past K holds a former chunk's, and is not read below
        const double* row = buf + i * ROW + (t / CH) * CH;
        double s = 0.0;
#pragma unroll
        for (int j = 0; j < CH; j++) s += row[j];
#pragma unroll
        for (int d = CH; d < 64; d *= 2) s += __shfl_xor(s, d, 64);
        if (lane < CH) part[k0 + i][wave] = s;
    }
    __syncthreads();
    for (int k = t; k < K; k += NTHR)
    {
        double s = 0.0;
        for (int i = 0; i < NW; i++) s += part[k][i];
        out[k] = s;
    }
    __syncthreads();
}

// Sum over the block; the result is valid in thread 0.  Fixed order, so
// results are reproducible run to run.
template <int NTHR>
__device__ inline double block_sum(double v)
{
    static_assert(NTHR % 64 == 0, "wave64");
    __shared__ double part[NTHR / 64];
    v = wave_sum(v);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) part[w] = v;
    __syncthreads();
    double r = 0.0;
    if (threadIdx.x == 0)
        for (int i = 0; i < NTHR / 64; i++) r += part[i];
    __syncthreads();
    return r;
}

}  // namespace glass
