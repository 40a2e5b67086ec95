// Sums over the 64 lanes of a wave in the VALU (gfx950).
#pragma once

#include <hip/hip_runtime.h>

namespace tad {

template <int CTRL>
__device__ __forceinline__ double dpp_move(double v)
{
    int2 u = __builtin_bit_cast(int2, v);
    u.x = __builtin_amdgcn_update_dpp(0, u.x, CTRL, 0xf, 0xf, true);
    u.y = __builtin_amdgcn_update_dpp(0, u.y, CTRL, 0xf, 0xf, true);
    return __builtin_bit_cast(double, u);
}

// a + b with the 16-lane rows (W = 16) or 32-lane halves (W = 32) exchanged:
// every lane gets its own row's (half's) value plus its neighbour's.
template <int W>
__device__ __forceinline__ double lane_swap_add(double v)
{
    const uint2 u = __builtin_bit_cast(uint2, v);
    uint2 a, b;
    if constexpr (W == 16)
    {
        const auto x = __builtin_amdgcn_permlane16_swap(u.x, u.x, false, false);
        const auto y = __builtin_amdgcn_permlane16_swap(u.y, u.y, false, false);
        a = make_uint2(x[0], y[0]);
        b = make_uint2(x[1], y[1]);
    }
    else
    {
        const auto x = __builtin_amdgcn_permlane32_swap(u.x, u.x, false, false);
        const auto y = __builtin_amdgcn_permlane32_swap(u.y, u.y, false, false);
        a = make_uint2(x[0], y[0]);
        b = make_uint2(x[1], y[1]);
    }
    return __builtin_bit_cast(double, a) + __builtin_bit_cast(double, b);
}

// Sum over the wave, the same bits in every lane: quads, 8 lanes, 16-lane
// rows (DPP), then rows and halves by lane swaps.  Six dependent VALU steps;
// the xor shuffles it replaces go through the LDS unit twice per step (about
// 0.3 us per FP64 sum on an otherwise idle CU, and the CG kernels of small
// systems are chains of such sums).  Every lane must be active.
__device__ __forceinline__ double wave_total(double v)
{
    v += dpp_move<0xB1>(v);   // quad_perm 1 0 3 2
    v += dpp_move<0x4E>(v);   // quad_perm 2 3 0 1
    v += dpp_move<0x141>(v);  // row_half_mirror
    v += dpp_move<0x140>(v);  // row_mirror
    v = lane_swap_add<16>(v);
    return lane_swap_add<32>(v);
}

// Sums of NV values over a block of NT threads: wave totals, then the waves
// in order; every thread gets the same bits.  sh: NT / 64 x NV doubles that
// no thread still reads.  One barrier.
template <int NT, int NV>
__device__ __forceinline__ void block_totals(double v[NV], double (*sh)[NV])
{
    const int wave = threadIdx.x >> 6;
#pragma unroll
    for (int i = 0; i < NV; ++i) v[i] = wave_total(v[i]);
    if constexpr (NT == 64) return;
    if ((threadIdx.x & 63) == 0)
    {
#pragma unroll
        for (int i = 0; i < NV; ++i) sh[wave][i] = v[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NV; ++i)
    {
        double t = sh[0][i];
#pragma unroll
        for (int w = 1; w < NT / 64; ++w) t += sh[w][i];
        v[i] = t;
    }
}

// Thread t's share p[t], p[t + NT], ... of n partials: the first NV are
// fetched together (0 past the end), strided_rest adds them and any further
// ones in order.  Split in two so that a kernel can have the loads of several
// arrays in flight before it adds any.
template <int NT, int NV>
__device__ __forceinline__ void strided_fetch(const double* __restrict__ p, int64_t n, double v[NV])
{
#pragma unroll
    for (int m = 0; m < NV; ++m)
    {
        const int64_t i = threadIdx.x + (int64_t)m * NT;
        v[m] = i < n ? p[i] : 0.0;
    }
}

template <int NT, int NV>
__device__ __forceinline__ double strided_rest(const double* __restrict__ p, int64_t n, const double v[NV])
{
    double acc = v[0];
#pragma unroll
    for (int m = 1; m < NV; ++m) acc += v[m];
    for (int64_t i = threadIdx.x + (int64_t)NV * NT; i < n; i += NT) acc += p[i];
    return acc;
}

} // namespace tad
