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
// the FP64 addition that follows, against 90 for a shuffle through LDS). BANKS: the groups of four lanes that take it,
// the others keep `old`.
template <int CTRL, int BANKS>
__device__ __forceinline__ float lane_move(float old, float x)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(old), __float_as_int(x), CTRL, 0xf, BANKS, true));
}
template <int CTRL, int BANKS>
__device__ __forceinline__ double lane_move(double old, double x)
{
    const long long o = __double_as_longlong(old), b = __double_as_longlong(x);
    const unsigned int lo = __builtin_amdgcn_update_dpp((int)o, (int)b, CTRL, 0xf, BANKS, true);
    const unsigned int hi = __builtin_amdgcn_update_dpp((int)(o >> 32), (int)(b >> 32), CTRL, 0xf, BANKS, true);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
template <int CTRL, int BANKS>
__device__ __forceinline__ CSum lane_move(CSum old, CSum x)
{
    return CSum{lane_move<CTRL, BANKS>(old.s, x.s), lane_move<CTRL, BANKS>(old.c, x.c)};
}

// x of the lane whose number differs in bit OFF (1, 2, 4 or 8). PERIODIC (OFF 4): x repeats every eight lanes of a
// row, where a rotation does it in one move.
template <int OFF, bool PERIODIC, typename X>
__device__ __forceinline__ X lane_xor(X x)
{
    static_assert(OFF == 1 || OFF == 2 || OFF == 4 || OFF == 8, "within a row of 16 lanes");
    if constexpr (OFF == 1) return lane_move<0xB1, 0xf>(x, x);            // quad permute 1, 0, 3, 2
    else if constexpr (OFF == 2) return lane_move<0x4E, 0xf>(x, x);       // quad permute 2, 3, 0, 1
    else if constexpr (OFF == 8) return lane_move<0x128, 0xf>(x, x);      // rotation by 8
    else if constexpr (PERIODIC) return lane_move<0x124, 0xf>(x, x);      // rotation by 4
    else return lane_move<0x114, 0xA>(lane_move<0x104, 0x5>(x, x), x);    // shifts by 4, each for half of the quads
}

// x of the lane 16 or 32 apart, as a pair {the even rows', the odd rows'} (or lower, upper half's) value, the same for
// both lanes of the pair.
template <int OFF>
__device__ __forceinline__ void half_pair(unsigned int x, unsigned int& a, unsigned int& b)
{
    if constexpr (OFF == 32) {
        const auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
        a = r[0], b = r[1];
    } else {
        const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
        a = r[0], b = r[1];
    }
}
template <int OFF>
__device__ __forceinline__ void half_pair(float x, float& a, float& b)
{
    unsigned int u, v;
    half_pair<OFF>((unsigned int)__float_as_int(x), u, v);
    a = __int_as_float((int)u), b = __int_as_float((int)v);
}
template <int OFF>
__device__ __forceinline__ void half_pair(double x, double& a, double& b)
{
    const unsigned long long q = (unsigned long long)__double_as_longlong(x);
    unsigned int al, bl, ah, bh;
    half_pair<OFF>((unsigned int)q, al, bl);
    half_pair<OFF>((unsigned int)(q >> 32), ah, bh);
    a = __longlong_as_double((long long)(((unsigned long long)ah << 32) | al));
    b = __longlong_as_double((long long)(((unsigned long long)bh << 32) | bl));
}
template <int OFF>
__device__ __forceinline__ void half_pair(CSum x, CSum& a, CSum& b)
{
    half_pair<OFF>(x.s, a.s, b.s);
    half_pair<OFF>(x.c, a.c, b.c);
}

// All-reduce of a commutative operation over aligned groups of LANES lanes (a power of two); every lane of the group
// takes part and ends with the same value: the butterfly that starts with the lanes LANES / 2 apart and ends with
// neighbours, so that the order of a sum is that of the same loop over __shfl_xor.
template <int LANES, typename X, typename Op>
__device__ __forceinline__ X group_reduce(X x, Op op)
{
    static_assert(LANES >= 1 && LANES <= 64 && (LANES & (LANES - 1)) == 0, "a part of a wave");
    X a, b;
    if constexpr (LANES >= 64) {
        half_pair<32>(x, a, b);
        x = op(a, b);
    }
    if constexpr (LANES >= 32) {
        half_pair<16>(x, a, b);
        x = op(a, b);
    }
    if constexpr (LANES >= 16) x = op(x, lane_xor<8, false>(x));
    if constexpr (LANES >= 8) x = op(x, lane_xor<4, (LANES >= 16)>(x));
    if constexpr (LANES >= 4) x = op(x, lane_xor<2, false>(x));
    if constexpr (LANES >= 2) x = op(x, lane_xor<1, false>(x));
    return x;
}

__device__ __forceinline__ CSum wave_csum(CSum v)
{
    return group_reduce<kWave>(v, [](CSum a, CSum b) { return csum_add(a, b); });
}
__device__ __forceinline__ double wave_sum(double v)
{
    return group_reduce<kWave>(v, [](double a, double b) { return a + b; });
}
__device__ __forceinline__ float wave_sumf(float v)
{
    return group_reduce<kWave>(v, [](float a, float b) { return a + b; });
}
__device__ __forceinline__ double wave_max(double v)
{
    return group_reduce<kWave>(v, [](double a, double b) { return fmax(a, b); });
}
__device__ __forceinline__ double wave_min(double v)
{
    return group_reduce<kWave>(v, [](double a, double b) { return fmin(a, b); });
}

// Sums over aligned groups of LANES lanes, in every lane of the group (all of them active).
template <int LANES, int NV>
__device__ __forceinline__ void group_sum(double (&v)[NV])
{
#pragma unroll
    for (int i = 0; i < NV; ++i) v[i] = group_reduce<LANES>(v[i], [](double a, double b) { return a + b; });
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

// Whether a kernel is to return: `stop` (its flag's value) is set. first is the first value the kernel loads (a row
// pointer, never negative), so that its load, and not only the flag's, comes before the branch: a kernel of a few
// dependent round trips would otherwise spend one on the flag alone.
__device__ __forceinline__ bool stopped(int stop, int first) { return (stop | (first & 0x80000000)) != 0; }

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

// Sums of the first kBlock threads' values, in every thread of the workgroup and identical in every workgroup that sums
// the same values.
template <int NV>
__device__ __forceinline__ void all_sum(double (&acc)[NV])
{
    __shared__ double sh[kBlock / kWave][NV];
    if (threadIdx.x < kBlock) {
#pragma unroll
        for (int k = 0; k < NV; ++k) acc[k] = wave_sum(acc[k]);
        if (threadIdx.x % kWave == 0)
#pragma unroll
            for (int k = 0; k < NV; ++k) sh[threadIdx.x / kWave][k] = acc[k];
    }
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
