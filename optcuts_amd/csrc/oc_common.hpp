// Shared device helpers for the gfx950 geometry-step kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace oc {

constexpr int kWave = 64;     // CDNA wavefront width
constexpr int kBlock = 256;   // threads per workgroup for 1-D kernels (4 waves)

// ---------------------------------------------------------------------------
// Exact-rounding helpers: a*b and a+b each rounded once, never contracted
// into an FMA, so expressions that the reference evaluates as two IEEE
// operations round the same way here.
__device__ __forceinline__ double mul_rn(double a, double b) { return __dmul_rn(a, b); }
__device__ __forceinline__ double add_rn(double a, double b) { return __dadd_rn(a, b); }

// ---------------------------------------------------------------------------
// Compensated (TwoSum) accumulation: value + running error, combined
// pairwise in a fixed tree order so every reduction is deterministic.
struct CSum {
    double s, c;
};

__device__ __forceinline__ CSum csum_add(CSum a, CSum b)
{
    const double s = add_rn(a.s, b.s);
    const double bp = __dsub_rn(s, a.s);
    const double err = add_rn(__dsub_rn(a.s, __dsub_rn(s, bp)), __dsub_rn(b.s, bp));
    return CSum{s, a.c + b.c + err};
}

// x of lane i (the same i in every lane)
__device__ __forceinline__ double read_lane(double x, int i)
{
    const long long b = __double_as_longlong(x);
    const unsigned int lo = __builtin_amdgcn_readlane((int)b, i), hi = __builtin_amdgcn_readlane((int)(b >> 32), i);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ __forceinline__ float read_lane(float x, int i)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), i));
}

// x of another lane of the same 16-lane row, chosen by a DPP control: a move inside the vector unit (30 clocks with
// the FP64 addition that follows, against 90 for a shuffle through LDS).
template <int CTRL>
__device__ __forceinline__ float lane_swap(float x)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ double lane_swap(double x)
{
    const long long b = __double_as_longlong(x);
    const unsigned int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, true);
    const unsigned int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
template <int CTRL>
__device__ __forceinline__ CSum lane_swap(CSum x)
{
    return CSum{lane_swap<CTRL>(x.s), lane_swap<CTRL>(x.c)};
}
__device__ __forceinline__ CSum read_lane(CSum x, int i) { return CSum{read_lane(x.s, i), read_lane(x.c, i)}; }

// All-reduce of a commutative operation over aligned groups of LANES (up to 16) lanes; every lane of the group takes
// part and ends with the same value: lanes 1 apart, 2 apart (quad permutes), then the mirror images within 8 and 16
// lanes, whose partners hold the other half's value.
template <int LANES, typename X, typename Op>
__device__ __forceinline__ X row_reduce(X x, Op op)
{
    static_assert(LANES >= 1 && LANES <= 16, "within a row of 16 lanes");
    if (LANES >= 2) x = op(x, lane_swap<0xB1>(x));
    if (LANES >= 4) x = op(x, lane_swap<0x4E>(x));
    if (LANES >= 8) x = op(x, lane_swap<0x141>(x));
    if (LANES >= 16) x = op(x, lane_swap<0x140>(x));
    return x;
}
// The same over a whole wave (every lane active): the four rows' values are read as scalars.
template <typename X, typename Op>
__device__ __forceinline__ X wave_reduce(X x, Op op)
{
    x = row_reduce<16>(x, op);
    return op(op(read_lane(x, 0), read_lane(x, 16)), op(read_lane(x, 32), read_lane(x, 48)));
}

__device__ __forceinline__ CSum wave_csum(CSum v)
{
    return wave_reduce(v, [](CSum a, CSum b) { return csum_add(a, b); });
}
__device__ __forceinline__ double wave_sum(double v)
{
    return wave_reduce(v, [](double a, double b) { return a + b; });
}
__device__ __forceinline__ float wave_sumf(float v)
{
    return wave_reduce(v, [](float a, float b) { return a + b; });
}
__device__ __forceinline__ double wave_max(double v)
{
    return wave_reduce(v, [](double a, double b) { return fmax(a, b); });
}
__device__ __forceinline__ double wave_min(double v)
{
    return wave_reduce(v, [](double a, double b) { return fmin(a, b); });
}

// Sums over aligned groups of LANES lanes, in every lane of the group (all of them active).
template <int LANES, int NV>
__device__ __forceinline__ void group_sum(double (&v)[NV])
{
#pragma unroll
    for (int i = 0; i < NV; ++i) v[i] = row_reduce<(LANES < 16 ? LANES : 16)>(v[i], [](double a, double b) { return a + b; });
#pragma unroll
    for (int off = 16; off < LANES; off <<= 1)
#pragma unroll
        for (int i = 0; i < NV; ++i) v[i] += __shfl_xor(v[i], off, LANES);
}

// This thread's share of the sum of n records' NV values (value k of record b at part[b * stride + k]), for workgroups
// of kBlock threads: four records in flight per thread (a loop that adds each record as it arrives pays a memory
// round trip for every kBlock of them).
template <int NV>
__device__ __forceinline__ void sum_records(const double* __restrict__ part, int n, int stride, double (&acc)[NV])
{
#pragma unroll
    for (int k = 0; k < NV; ++k) acc[k] = 0.0;
    for (int base = threadIdx.x; base < n; base += 4 * kBlock) {
        double v[4][NV];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int b = base + q * kBlock;
#pragma unroll
            for (int k = 0; k < NV; ++k) v[q][k] = b < n ? part[(size_t)b * stride + k] : 0.0;
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int k = 0; k < NV; ++k) acc[k] += v[q][k];
    }
}

// Block reduction of NV independent compensated sums; result valid in thread 0.
template <int NV>
__device__ __forceinline__ void block_csum(CSum (&v)[NV])
{
    __shared__ CSum sh[kBlock / kWave][NV];
    const int lane = threadIdx.x % kWave, wid = threadIdx.x / kWave;
#pragma unroll
    for (int k = 0; k < NV; ++k) v[k] = wave_csum(v[k]);
    if (lane == 0)
#pragma unroll
        for (int k = 0; k < NV; ++k) sh[wid][k] = v[k];
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            CSum a = sh[0][k];
            for (int w = 1; w < (int)(blockDim.x / kWave); ++w) a = csum_add(a, sh[w][k]);
            v[k] = a;
        }
    }
    __syncthreads();
}

// Block reduction of NV plain sums; result valid in thread 0.
template <int NV>
__device__ __forceinline__ void block_sum(double (&v)[NV])
{
    __shared__ double sh[kBlock / kWave][NV];
    const int lane = threadIdx.x % kWave, wid = threadIdx.x / kWave;
#pragma unroll
    for (int k = 0; k < NV; ++k) v[k] = wave_sum(v[k]);
    if (lane == 0)
#pragma unroll
        for (int k = 0; k < NV; ++k) sh[wid][k] = v[k];
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            double a = sh[0][k];
            for (int w = 1; w < (int)(blockDim.x / kWave); ++w) a += sh[w][k];
            v[k] = a;
        }
    }
    __syncthreads();
}

// Workgroup sums of every thread's values, identical in every thread of every workgroup that sums the same values.
template <int NV>
__device__ __forceinline__ void all_sum(double (&acc)[NV])
{
    __shared__ double sh[kBlock / kWave][NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) acc[k] = wave_sum(acc[k]);
    if (threadIdx.x % kWave == 0)
#pragma unroll
        for (int k = 0; k < NV; ++k) sh[threadIdx.x / kWave][k] = acc[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        acc[k] = sh[0][k];
#pragma unroll
        for (int w = 1; w < kBlock / kWave; ++w) acc[k] += sh[w][k];
    }
}

// Order-preserving map of a double to uint64 (for atomicMin over doubles of
// either sign); NaN inputs are filtered by the caller.
__device__ __forceinline__ unsigned long long dbl_to_ordered(double x)
{
    unsigned long long u = (unsigned long long)__double_as_longlong(x);
    return (u & 0x8000000000000000ull) ? ~u : (u | 0x8000000000000000ull);
}

__device__ __forceinline__ double ordered_to_dbl(unsigned long long u)
{
    u = (u & 0x8000000000000000ull) ? (u & 0x7fffffffffffffffull) : ~u;
    return __longlong_as_double((long long)u);
}

inline double ordered_to_dbl_host(unsigned long long u)
{
    u = (u & 0x8000000000000000ull) ? (u & 0x7fffffffffffffffull) : ~u;
    double d;
    __builtin_memcpy(&d, &u, sizeof(d));
    return d;
}

inline unsigned long long dbl_to_ordered_host(double x)
{
    unsigned long long u;
    __builtin_memcpy(&u, &x, sizeof(u));
    return (u & 0x8000000000000000ull) ? ~u : (u | 0x8000000000000000ull);
}

inline int grid_for(long n, int block = kBlock)
{
    long g = (n + block - 1) / block;
    return (int)(g < 1 ? 1 : g);
}

}  // namespace oc
