// HIP kernels of the sparse second-order path for gfx950 (linear algebra part)
// and their launchers.
//
//   k_sum_*, k_dot_*   deterministic FP64 sums (fixed tree, no atomics)
//   k_assemble_*       element-order gather of gradient and CSR values
//                      through the precomputed maps (replaces the serial
//                      triplet loop ScalarObjectiveTerm.hh:257-277 and
//                      setFromTriplets, ScalarFunctionImpl.hh:398)
//   k_pcg_*, k_spmv_sym  block-Jacobi PCG on the block-structured CSR
//                      (replaces SimplicialLDLT, NewtonDirection.hh:25-48)
#include <hip/hip_runtime.h>
#include <cstdint>
#include <algorithm>
#include "tad_internal.hpp"
#include "tad_wave.hpp"
#include "tad_energies.hpp"
#include "tad_elements.hpp"

namespace tad {

// ---------------------------------------------------------------------------
// Deterministic reductions
// ---------------------------------------------------------------------------
// Fixed-order block reduction: butterfly inside each 64-lane wave, then the
// four wave totals in order.  Same bits for the same inputs on every run.
__device__ __forceinline__ double block_sum(double v, double* sh)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    const int wave = threadIdx.x >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) sh[wave] = v;
    __syncthreads();
    double r = sh[0];
#pragma unroll
    for (int w = 1; w < kBlock / 64; ++w) r += sh[w];
    return r;
}

// acc over v[i], v[i + S], v[i + 2S], ... < hi in that order, four loads in flight
template <int S>
__device__ __forceinline__ double strided_sum(const double* __restrict__ v, int64_t i, int64_t hi)
{
    double acc = 0.0;
    for (; i + 3 * S < hi; i += 4 * S)
    {
        const double a0 = v[i], a1 = v[i + S], a2 = v[i + 2 * S], a3 = v[i + 3 * S];
        acc += a0;
        acc += a1;
        acc += a2;
        acc += a3;
    }
    for (; i < hi; i += S) acc += v[i];
    return acc;
}

// the b-th of kReduceBlocks chunks of in[0 .. n), summed by one block
__device__ __forceinline__ double sum_chunk(const double* __restrict__ in, int64_t n, int64_t b, double* sh)
{
    const int64_t chunk = (n + kReduceBlocks - 1) / kReduceBlocks;
    const int64_t lo = b * chunk;
    const int64_t hi = lo + chunk < n ? lo + chunk : n;
    return block_sum(strided_sum<kBlock>(in, lo + threadIdx.x, hi), sh);
}

// block b of row c sums the contiguous chunk [b*chunk, (b+1)*chunk)
__global__ __launch_bounds__(kBlock) void k_sum_stage1(const double* __restrict__ in, int64_t n, int64_t stride,
                                                       double* __restrict__ partials)
{
    __shared__ double sh[kBlock];
    const int c = blockIdx.y;
    const double s = sum_chunk(in + c * stride, n, blockIdx.x, sh);
    if (threadIdx.x == 0) partials[c * kReduceBlocks + blockIdx.x] = s;
}

// out[c] = the sum of row c's partials; err (optional): its value into
// err_out and cleared for the next evaluation.  out and err_out may be pinned
// host memory: a store instead of a copy per result.
__global__ __launch_bounds__(kBlock) void k_sum_stage2(const double* __restrict__ partials, double* __restrict__ out,
                                                       int* __restrict__ err, int* __restrict__ err_out)
{
    __shared__ double sh[kBlock];
    const int c = blockIdx.x;
    double acc = 0.0;
    for (int i = threadIdx.x; i < kReduceBlocks; i += kBlock) acc += partials[c * kReduceBlocks + i];
    const double s = block_sum(acc, sh);
    if (threadIdx.x == 0)
    {
        out[c] = s;
        if (err)
        {
            *err_out = *err;
            *err = 0;
        }
    }
}

hipError_t launch_sum(const double* in, int64_t n, int ncand, int64_t stride, double* partials, double* out,
                      hipStream_t s)
{
    k_sum_stage1<<<dim3(kReduceBlocks, ncand), kBlock, 0, s>>>(in, n, stride, partials);
    k_sum_stage2<<<ncand, kBlock, 0, s>>>(partials, out, nullptr, nullptr);
    return hipGetLastError();
}

__global__ __launch_bounds__(kBlock) void k_dot_stage1(const double* __restrict__ a, const double* __restrict__ b,
                                                       int64_t n, double* __restrict__ partials)
{
    __shared__ double sh[kBlock];
    const int64_t chunk = (n + kReduceBlocks - 1) / kReduceBlocks;
    const int64_t lo = (int64_t)blockIdx.x * chunk;
    const int64_t hi = lo + chunk < n ? lo + chunk : n;
    double acc = 0.0;
    for (int64_t i = lo + threadIdx.x; i < hi; i += kBlock) acc += a[i] * b[i];
    const double s = block_sum(acc, sh);
    if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

hipError_t launch_dot(const double* a, const double* b, int64_t n, double* partials, double* out, hipStream_t s)
{
    k_dot_stage1<<<kReduceBlocks, kBlock, 0, s>>>(a, b, n, partials);
    k_sum_stage2<<<1, kBlock, 0, s>>>(partials, out, nullptr, nullptr);
    return hipGetLastError();
}

__global__ void k_fill(double* p, int64_t n, double v)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

hipError_t launch_fill(double* p, int64_t n, double v, hipStream_t s)
{
    if (n == 0) return hipSuccess;
    k_fill<<<(unsigned)((n + kBlock - 1) / kBlock), kBlock, 0, s>>>(p, n, v);
    return hipGetLastError();
}

// xo = x0 + step[0] * dir where a step was accepted (accepted[0] >= 0)
__global__ void k_axpy_point(const double* __restrict__ x0, const double* __restrict__ dir,
                             const double* __restrict__ step, const int* __restrict__ accepted, int64_t n,
                             double* __restrict__ xo)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (accepted[0] < 0) return;
    if (i < n) xo[i] = fma(step[0], dir[i], x0[i]);
}

// first-stage sums of two dot products (row blockIdx.y), as k_dot_stage1
__global__ __launch_bounds__(kBlock) void k_dot2_stage1(const double* __restrict__ a1, const double* __restrict__ b1,
                                                        const double* __restrict__ a2, const double* __restrict__ b2,
                                                        int64_t n, double* __restrict__ partials)
{
    __shared__ double sh[kBlock];
    const double* __restrict__ a = blockIdx.y ? a2 : a1;
    const double* __restrict__ b = blockIdx.y ? b2 : b1;
    const int64_t chunk = (n + kReduceBlocks - 1) / kReduceBlocks;
    const int64_t lo = (int64_t)blockIdx.x * chunk;
    const int64_t hi = lo + chunk < n ? lo + chunk : n;
    double acc = 0.0;
    for (int64_t i = lo + threadIdx.x; i < hi; i += kBlock) acc += a[i] * b[i];
    const double s = block_sum(acc, sh);
    if (threadIdx.x == 0) partials[blockIdx.y * kReduceBlocks + blockIdx.x] = s;
}

// The end of one batch of line-search trials, one block: the candidates'
// energies and (use_dots) the two dot products from their partials, one wave
// per row with the sums of k_sum_stage2 bit for bit, then the first candidate
// in order that satisfies the Armijo condition (LineSearch.hh:49-58), or -1,
// or -2 at a NaN energy before one is accepted.  Its step goes to the device
// for k_axpy_point, everything to pinned memory for the host.
__global__ __launch_bounds__(kBlock) void k_ls_finish(LineSearchBatch a)
{
    static_assert(kReduceBlocks == kBlock && kBlock == 256, "four partials per lane");
    __shared__ double tot[kMaxTrials + 2];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int rows = a.ncand + (a.use_dots ? 2 : 0);
    for (int r = wv; r < rows; r += kBlock / 64)
    {
        const double* __restrict__ p = r < a.ncand ? a.partials + r * kReduceBlocks
                                                   : a.dot_partials + (r - a.ncand) * kReduceBlocks;
        double v[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = 0.0 + p[lane + 64 * q];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1)
#pragma unroll
            for (int q = 0; q < 4; ++q) v[q] += __shfl_xor(v[q], off, 64);
        if (lane == 0) tot[r] = ((v[0] + v[1]) + v[2]) + v[3];
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    const double dg = a.use_dots ? a.dir_scale * tot[a.ncand] : a.dir_dot_g;
    int acc = -1;
    for (int c = 0; c < a.ncand && acc == -1; ++c)
    {
        // products and sum rounded one by one, as the host computes them
#pragma clang fp contract(off)
        const double bound = a.f + a.armijo * a.sval[c] * dg;
        if (tot[c] != tot[c]) acc = -2;
        else if (tot[c] <= bound) acc = c;
    }
    a.step_out[0] = acc >= 0 ? a.step[acc] : 0.0;
    a.accepted_out[0] = acc;
    for (int c = 0; c < a.ncand; ++c) a.host->f[c] = tot[c];
    if (a.use_dots)
    {
        a.host->dir_dot = tot[a.ncand];
        a.host->dot2 = tot[a.ncand + 1];
    }
    a.host->accepted = acc;
}

hipError_t launch_ls_finish(const LineSearchBatch& b, const double* ls_f, int64_t n_elem, int64_t stride,
                            double* partials, const double* a1, const double* b1, const double* a2, const double* b2,
                            int64_t n, const double* x0, const double* dir, double* x_out, hipStream_t s)
{
    LineSearchBatch a = b;
    a.partials = partials;
    a.dot_partials = partials + kMaxTrials * kReduceBlocks;
    k_sum_stage1<<<dim3(kReduceBlocks, a.ncand), kBlock, 0, s>>>(ls_f, n_elem, stride, partials);
    if (a.use_dots)
        k_dot2_stage1<<<dim3(kReduceBlocks, 2), kBlock, 0, s>>>(a1, b1, a2, b2, n,
                                                                partials + kMaxTrials * kReduceBlocks);
    k_ls_finish<<<1, kBlock, 0, s>>>(a);
    if (n > 0)
        k_axpy_point<<<(unsigned)((n + kBlock - 1) / kBlock), kBlock, 0, s>>>(x0, dir, a.step_out, a.accepted_out, n,
                                                                              x_out);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Assembly: contiguous sums over destination-sorted contributions
// ---------------------------------------------------------------------------
// The element kernels scatter every d x d block (and every per-vertex gradient
// part) to its slot; the slots of one destination are contiguous and in
// element order, so each output entry is a fixed-order sum over one run.
// acc + src[c * S] for c in [c0, c1), in order
template <int S, class T>
__device__ __forceinline__ double run_tail(double acc, const T* __restrict__ src, int64_t c0, int64_t c1)
{
    int64_t c = c0;
    for (; c + 4 <= c1; c += 4)
    {
        const double a0 = (double)src[c * S], a1 = (double)src[(c + 1) * S];
        const double a2 = (double)src[(c + 2) * S], a3 = (double)src[(c + 3) * S];
        acc += a0;
        acc += a1;
        acc += a2;
        acc += a3;
    }
    for (; c < c1; ++c) acc += (double)src[c * S];
    return acc;
}

// sum_{c in [c0, c1)} src[c * S] in index order, four loads in flight
template <int S, class T>
__device__ __forceinline__ double run_sum(const T* __restrict__ src, int64_t c0, int64_t c1)
{
    return run_tail<S>(0.0, src, c0, c1);
}

// Runs exist for the upper blocks; a lower block (u, v), u > v, sums the run
// of (v, u) transposed.
// One thread per block (all D*D entries of a contribution per thread, two
// contributions in flight).  Which shape is faster depends on d, the precision
// and the run lengths (the autotuner times them).
template <class T, int D>
__global__ __launch_bounds__(kBlock) void k_assemble_hessian_tpb(int64_t b_begin, int64_t nb,
                                                                 const int32_t* __restrict__ block_row,
                                                                 const int32_t* __restrict__ brow_ptr,
                                                                 const int64_t* __restrict__ hslot_ptr,
                                                                 const int32_t* __restrict__ mirror,
                                                                 const T* __restrict__ Hc,
                                                                 const int32_t* __restrict__ row_ptr,
                                                                 double* __restrict__ H)
{
    constexpr int DD = D * D;
    const int64_t b = b_begin + (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nb) return;
    const int u = block_row[b];
    const int b0 = brow_ptr[u];
    const int k = (int)(b - b0);
    const int nbu = brow_ptr[u + 1] - b0;
    const int64_t mb = mirror[b];
    double acc[DD];
#pragma unroll
    for (int m = 0; m < DD; ++m) acc[m] = 0.0;
    int64_t c = hslot_ptr[mb];
    const int64_t c1 = hslot_ptr[mb + 1];
    for (; c + 2 <= c1; c += 2)
    {
        double v0[DD], v1[DD];
#pragma unroll
        for (int m = 0; m < DD; ++m)
        {
            v0[m] = (double)Hc[c * DD + m];
            v1[m] = (double)Hc[(c + 1) * DD + m];
        }
#pragma unroll
        for (int m = 0; m < DD; ++m)
        {
            acc[m] += v0[m];
            acc[m] += v1[m];
        }
    }
    for (; c < c1; ++c)
    {
#pragma unroll
        for (int m = 0; m < DD; ++m) acc[m] += (double)Hc[c * DD + m];
    }
    const bool tr = mb != b;
    const int64_t base = row_ptr[D * u];
#pragma unroll
    for (int i = 0; i < D; ++i)
#pragma unroll
        for (int j = 0; j < D; ++j)
            H[base + (int64_t)i * D * nbu + D * k + j] = tr ? acc[j * D + i] : acc[i * D + j];
}

// Upper-run shapes: each run is summed once and written to its upper block
// and, transposed, to the mirrored lower block, so every contribution is read
// once (shapes 0 / 1 read the off-diagonal runs twice).  D*D lanes per upper
// block, lane m = (i, j) writes H_upper(i, j) and H_lower(j, i).
template <class T, int D>
__global__ __launch_bounds__(kBlock) void k_assemble_hessian_upper(int64_t b_begin, int64_t nu,
                                                                   const int64_t* __restrict__ uslot_ptr,
                                                                   const int4* __restrict__ uplace,
                                                                   const T* __restrict__ Hc, double* __restrict__ H)
{
    constexpr int DD = D * D;
    constexpr int BPW = 64 / DD;
    const int lane = threadIdx.x & 63;
    const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    if (lane >= BPW * DD) return;
    const int64_t b = b_begin + wave * BPW + lane / DD;
    if (b >= nu) return;
    const int m = lane % DD;
    const int i = m / D, j = m % D;
    const double acc = run_sum<DD>(Hc + m, uslot_ptr[b], uslot_ptr[b + 1]);
    const int4 pl = uplace[b];
    H[(int64_t)pl.x + (int64_t)i * pl.y + j] = acc;
    if (pl.z >= 0) H[(int64_t)pl.z + (int64_t)j * pl.w + i] = acc;
}

// One thread per upper block, two contributions in flight.
template <class T, int D>
__global__ __launch_bounds__(kBlock) void k_assemble_hessian_upper_tpb(int64_t b_begin, int64_t nu,
                                                                       const int64_t* __restrict__ uslot_ptr,
                                                                       const int4* __restrict__ uplace,
                                                                       const T* __restrict__ Hc,
                                                                       double* __restrict__ H)
{
    constexpr int DD = D * D;
    const int64_t b = b_begin + (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nu) return;
    double acc[DD];
#pragma unroll
    for (int m = 0; m < DD; ++m) acc[m] = 0.0;
    int64_t c = uslot_ptr[b];
    const int64_t c1 = uslot_ptr[b + 1];
    for (; c + 2 <= c1; c += 2)
    {
        double v0[DD], v1[DD];
#pragma unroll
        for (int m = 0; m < DD; ++m)
        {
            v0[m] = (double)Hc[c * DD + m];
            v1[m] = (double)Hc[(c + 1) * DD + m];
        }
#pragma unroll
        for (int m = 0; m < DD; ++m)
        {
            acc[m] += v0[m];
            acc[m] += v1[m];
        }
    }
    for (; c < c1; ++c)
    {
#pragma unroll
        for (int m = 0; m < DD; ++m) acc[m] += (double)Hc[c * DD + m];
    }
    const int4 pl = uplace[b];
#pragma unroll
    for (int i = 0; i < D; ++i)
#pragma unroll
        for (int j = 0; j < D; ++j) H[(int64_t)pl.x + (int64_t)i * pl.y + j] = acc[i * D + j];
    if (pl.z >= 0)
    {
#pragma unroll
        for (int i = 0; i < D; ++i)
#pragma unroll
            for (int j = 0; j < D; ++j) H[(int64_t)pl.z + (int64_t)j * pl.w + i] = acc[i * D + j];
    }
}

// D lanes per handle, floor(64 / D) handles per wave; wave index `wave`.
template <class T, int D>
__device__ __forceinline__ void gradient_rows(int64_t wave, int64_t v_begin, int64_t nh,
                                              const int64_t* __restrict__ gslot_ptr, const T* __restrict__ G,
                                              double* __restrict__ g)
{
    constexpr int HPW = 64 / D;
    const int lane = threadIdx.x & 63;
    if (lane >= HPW * D) return;
    const int64_t v = v_begin + wave * HPW + lane / D;
    if (v >= nh) return;
    const int i = lane % D;
    g[v * D + i] = run_sum<D>(G + i, gslot_ptr[v], gslot_ptr[v + 1]);
}

template <class T, int D>
__global__ __launch_bounds__(kBlock) void k_assemble_gradient(int64_t v_begin, int64_t nh,
                                                              const int64_t* __restrict__ gslot_ptr,
                                                              const T* __restrict__ G, double* __restrict__ g)
{
    gradient_rows<T, D>(((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6, v_begin, nh, gslot_ptr, G, g);
}

// A segment's energy: terms in order, fixed thread stride within each range,
// fixed block tree.
__device__ __forceinline__ double segment_total(const double* __restrict__ elem_f, const int64_t* __restrict__ ranges,
                                                int n_terms, int64_t n_seg, int64_t sgm, double* sh)
{
    double acc = 0.0;
    for (int t = 0; t < n_terms; ++t)
    {
        const int64_t a = ranges[(t * n_seg + sgm) * 2], b = ranges[(t * n_seg + sgm) * 2 + 1];
        int64_t i = a + threadIdx.x;
        for (; i + 3 * kBlock < b; i += 4 * kBlock)  // four loads in flight, same order
        {
            const double v0 = elem_f[i], v1 = elem_f[i + kBlock], v2 = elem_f[i + 2 * kBlock],
                         v3 = elem_f[i + 3 * kBlock];
            acc += v0;
            acc += v1;
            acc += v2;
            acc += v3;
        }
        for (; i < b; i += kBlock) acc += elem_f[i];
    }
    return block_sum(acc, sh);
}

// Everything an evaluation does after its element kernels, in one launch: the
// work is independent, and at small sizes each launch of its own is 2 .. 4 us
// of mostly idle chip.  Blocks, in this order:
//   tile_blocks   CSR values of H, one tile each: whole block rows holding at
//                 most kAsmTileBlocks blocks.  One thread sums one block's
//                 run (two contributions in flight), the values pass through
//                 LDS and leave as one contiguous run.  The blocks of one XCD
//                 (blockIdx % 8) take a contiguous eighth of the tiles, so a
//                 run's second read, for the mirrored block, can hit in that
//                 XCD's L2.  A row with more blocks is a tile of its own,
//                 written directly.
//   grad_blocks   gradient of kBlock / 64 waves of handles
//   copy_blocks   x kept for the coarse space's lever arms
//   kReduceBlocks first-stage sums of the element energies
//   n_seg         segment energies
// 25 x 25 grid: gradient, H, x copy and two sum launches, two result copies and
// a clear, 13 us of kernels and 75 us per evaluation -> 3.3 + 2.5 us and 45 us.
// 256 disks, mixed (430 MB of values written, 190 MB of runs read): 396 us with
// D*D lanes per block, unstaged -> 180 us (3.4 TB/s).
template <class T, int D>
__global__ __launch_bounds__(kBlock) void k_assemble_all(EvalTail a)
{
    constexpr int DD = D * D;
    __shared__ double sm[kAsmTileBlocks * DD < kBlock ? kBlock : kAsmTileBlocks * DD];
    const int t = threadIdx.x;
    int64_t blk = blockIdx.x;
    if (blk < a.tile_blocks)
    {
        const int64_t per = a.tile_blocks >> 3;
        const int64_t tile = (blk & 7) * per + (blk >> 3);
        if (tile >= a.n_tiles) return;
        const T* __restrict__ Hc = (const T*)a.Hc;
        const int64_t b0 = a.tile_ptr[tile], b1 = a.tile_ptr[tile + 1];
        const int nb = (int)(b1 - b0);
        double* __restrict__ out = a.H + b0 * DD;
        const bool direct = nb > kAsmTileBlocks;
        for (int b = t; b < nb; b += kBlock)
        {
            const uint32_t run = a.arun[b0 + b], len = a.alen[b0 + b], pos = a.apos[b0 + b];
            const T* __restrict__ src = Hc + (int64_t)(run & 0x7fffffffu) * DD;
            double acc[DD];
#pragma unroll
            for (int m = 0; m < DD; ++m) acc[m] = 0.0;
            uint32_t c = 0;
            for (; c + 2 <= len; c += 2)
            {
                T v0[DD], v1[DD];
#pragma unroll
                for (int m = 0; m < DD; ++m)
                {
                    v0[m] = src[c * DD + m];
                    v1[m] = src[(c + 1) * DD + m];
                }
#pragma unroll
                for (int m = 0; m < DD; ++m)
                {
                    acc[m] += (double)v0[m];
                    acc[m] += (double)v1[m];
                }
            }
            if (c < len)
            {
#pragma unroll
                for (int m = 0; m < DD; ++m) acc[m] += (double)src[c * DD + m];
            }
            const bool tr = run >> 31;  // the mirror's run, transposed
            const int base = direct ? D * b : (int)(pos & 0xffffu), stride = direct ? D * nb : (int)(pos >> 16);
#pragma unroll
            for (int i = 0; i < D; ++i)
#pragma unroll
                for (int j = 0; j < D; ++j)
                {
                    const double e = tr ? acc[j * D + i] : acc[i * D + j];
                    if (direct) out[base + (int64_t)i * stride + j] = e;
                    else sm[base + i * stride + j] = e;
                }
        }
        if (direct) return;
        __syncthreads();
        for (int i = t; i < nb * DD; i += kBlock) out[i] = sm[i];
        return;
    }
    blk -= a.tile_blocks;
    if (blk < a.grad_blocks)
    {
        gradient_rows<T, D>((blk * kBlock + t) >> 6, 0, a.n_handles, a.gslot_ptr, (const T*)a.G, a.g);
        return;
    }
    blk -= a.grad_blocks;
    if (blk < a.copy_blocks)
    {
        const int64_t i0 = blk * (4 * kBlock) + t;
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (i0 + q * kBlock < a.n_handles * D) a.x_copy[i0 + q * kBlock] = a.x[i0 + q * kBlock];
        return;
    }
    blk -= a.copy_blocks;
    if (blk < kReduceBlocks)
    {
        const double s = sum_chunk(a.elem_f, a.n_elem, blk, sm);
        if (t == 0) a.partials[blk] = s;
        return;
    }
    blk -= kReduceBlocks;
    const double s = segment_total(a.elem_f, a.seg_ranges, a.n_terms, a.n_seg, blk, sm);
    if (t == 0) a.seg_f[blk] = s;
}

hipError_t launch_eval_tail(int d, int precision, EvalTail a, int* err, double* f_out, int* err_out, hipStream_t s)
{
    a.tile_blocks = a.H ? (a.n_tiles + 7) / 8 * 8 : 0;
    const int64_t waves = a.g ? (a.n_handles + 64 / d - 1) / (64 / d) : 0;
    a.grad_blocks = (waves * 64 + kBlock - 1) / kBlock;
    a.copy_blocks = a.x_copy ? (a.n_handles * d + 4 * kBlock - 1) / (4 * kBlock) : 0;
    const int64_t grid = a.tile_blocks + a.grad_blocks + a.copy_blocks + kReduceBlocks + a.n_seg;
    if (grid > 0x7fffffff) return hipErrorInvalidValue;
#define TAD_TAIL(T, D) k_assemble_all<T, D><<<(unsigned)grid, kBlock, 0, s>>>(a)
    if (precision == 0)
    {
        if (d == 1) TAD_TAIL(double, 1);
        else if (d == 2) TAD_TAIL(double, 2);
        else TAD_TAIL(double, 3);
    }
    else if (d == 1) TAD_TAIL(float, 1);
    else if (d == 2) TAD_TAIL(float, 2);
    else TAD_TAIL(float, 3);
#undef TAD_TAIL
    k_sum_stage2<<<1, kBlock, 0, s>>>(a.partials, f_out, err, err_out);
    return hipGetLastError();
}

// Blocks [b0, b1) of the shape's index space: CSR blocks (shapes 0, 1) or
// upper blocks in CSR order (shapes 2, 3).
template <class T, int D>
static void launch_assemble_hessian_td(int shape, const HessAsm& a, int64_t b0, int64_t b1, const T* Hc, double* H,
                                       hipStream_t s)
{
    constexpr int bpw = 64 / (D * D);
    const int64_t n = b1 - b0;
    if (n <= 0) return;
    const unsigned gt = (unsigned)((n + kBlock - 1) / kBlock);
    const unsigned gl = (unsigned)((((n + bpw - 1) / bpw) * 64 + kBlock - 1) / kBlock);
    if (shape <= 1)  // (a range of rows has no whole tiles: shape 1 for shape 0)
        k_assemble_hessian_tpb<T, D><<<gt, kBlock, 0, s>>>(b0, b1, a.block_row, a.brow_ptr, a.hslot_ptr, a.mirror,
                                                           Hc, a.row_ptr, H);
    else if (shape == 2)
        k_assemble_hessian_upper<T, D><<<gl, kBlock, 0, s>>>(b0, b1, a.uslot_ptr, a.uplace, Hc, H);
    else
        k_assemble_hessian_upper_tpb<T, D><<<gt, kBlock, 0, s>>>(b0, b1, a.uslot_ptr, a.uplace, Hc, H);
}

template <class T>
static hipError_t launch_assemble_hessian_t(int d, int shape, const HessAsm& a, int64_t r0, int64_t r1, const T* Hc,
                                            double* H, hipStream_t s)
{
    if (a.n_blocks == 0) return hipSuccess;
    if (shape < 0 || shape >= kAsmShapes) return hipErrorInvalidValue;
    int64_t b0, b1;
    if (shape >= 2)
    {
        b0 = r0 < 0 ? 0 : a.urow_ptr_h[r0];
        b1 = r0 < 0 ? a.n_upper : a.urow_ptr_h[r1];
    }
    else
    {
        b0 = r0 < 0 ? 0 : a.brow_ptr_h[r0];
        b1 = r0 < 0 ? a.n_blocks : a.brow_ptr_h[r1];
    }
    if (d == 1) launch_assemble_hessian_td<T, 1>(shape, a, b0, b1, Hc, H, s);
    else if (d == 2) launch_assemble_hessian_td<T, 2>(shape, a, b0, b1, Hc, H, s);
    else launch_assemble_hessian_td<T, 3>(shape, a, b0, b1, Hc, H, s);
    return hipGetLastError();
}

hipError_t launch_assemble_hessian(int d, int precision, int shape, const HessAsm& a, const void* Hc, double* H,
                                   hipStream_t s, int64_t r0, int64_t r1)
{
    if (precision == 0) return launch_assemble_hessian_t<double>(d, shape, a, r0, r1, (const double*)Hc, H, s);
    return launch_assemble_hessian_t<float>(d, shape, a, r0, r1, (const float*)Hc, H, s);
}

template <class T>
static hipError_t launch_assemble_gradient_t(int d, int64_t v0, int64_t v1, const int64_t* gslot_ptr, const T* G,
                                             double* g, hipStream_t s)
{
    const int64_t nh = v1 - v0;
    if (nh <= 0) return hipSuccess;
    const int hpw = 64 / d;
    const int64_t waves = (nh + hpw - 1) / hpw;
    const unsigned grid = (unsigned)((waves * 64 + kBlock - 1) / kBlock);
    if (d == 1) k_assemble_gradient<T, 1><<<grid, kBlock, 0, s>>>(v0, v1, gslot_ptr, G, g);
    else if (d == 2) k_assemble_gradient<T, 2><<<grid, kBlock, 0, s>>>(v0, v1, gslot_ptr, G, g);
    else k_assemble_gradient<T, 3><<<grid, kBlock, 0, s>>>(v0, v1, gslot_ptr, G, g);
    return hipGetLastError();
}

hipError_t launch_assemble_gradient(int d, int precision, int64_t nh, const int64_t* gslot_ptr, const void* G,
                                    double* g, hipStream_t s, int64_t v0, int64_t v1)
{
    if (v0 < 0)
    {
        v0 = 0;
        v1 = nh;
    }
    if (precision == 0) return launch_assemble_gradient_t<double>(d, v0, v1, gslot_ptr, (const double*)G, g, s);
    return launch_assemble_gradient_t<float>(d, v0, v1, gslot_ptr, (const float*)G, g, s);
}

// ---------------------------------------------------------------------------
// PCG
// ---------------------------------------------------------------------------
// Reductions without atomics or fences: every kernel writes one partial per
// block; the kernel that consumes a scalar re-sums the producer's partials in
// index order in every block (identical bits everywhere, a few KB from L2).
// Scalars that change per iteration live in double-buffered partial slots
// indexed by the iteration number, so no block of a kernel ever reads a value
// another block of the same kernel writes.  Block 0 records bookkeeping
// (iteration count, residual, termination) for later kernels and the host.
//
// Partial buffer layout (doubles): [pq: Gs][rz: 2 x Gv][rr: 2 x Gv]
//
// The solver's vectors, matrix copy and preconditioner are in solver order
// (PcgSystem::perm): the members of an aggregate are consecutive, so that the
// update kernel, whose blocks own a part of one aggregate each, also sums the
// aggregate's restricted residual, the coarse correction adds to consecutive
// entries, and the rows a block of the product takes share most of the
// entries of z they gather.

// The block-Jacobi inverse keeps the upper triangle of each symmetric D x D
// block, row by row: (0,0) (0,1) .. (0,D-1) (1,1) .. (D-1,D-1).
template <int D>
struct PackedBlock
{
    static constexpr int n = D * (D + 1) / 2;
    __device__ static constexpr int at(int i, int j)
    {
        return i <= j ? i * D - (i * (i - 1)) / 2 + (j - i) : j * D - (j * (j - 1)) / 2 + (i - j);
    }
};

template <int D>
__device__ __forceinline__ void invert_block(const double* B, double* o)
{
    if constexpr (D == 1)
        o[0] = 1.0 / B[0];
    else if constexpr (D == 2)
    {
        const double det = B[0] * B[3] - B[1] * B[2];
        o[0] = B[3] / det; o[1] = -B[1] / det; o[2] = -B[2] / det; o[3] = B[0] / det;
    }
    else
    {
        const double c00 = B[4] * B[8] - B[5] * B[7];
        const double c01 = B[5] * B[6] - B[3] * B[8];
        const double c02 = B[3] * B[7] - B[4] * B[6];
        const double det = B[0] * c00 + B[1] * c01 + B[2] * c02;
        const double id = 1.0 / det;
        o[0] = c00 * id; o[3] = c01 * id; o[6] = c02 * id;
        o[1] = (B[2] * B[7] - B[1] * B[8]) * id;
        o[4] = (B[0] * B[8] - B[2] * B[6]) * id;
        o[7] = (B[1] * B[6] - B[0] * B[7]) * id;
        o[2] = (B[1] * B[5] - B[2] * B[4]) * id;
        o[5] = (B[2] * B[3] - B[0] * B[5]) * id;
        o[8] = (B[0] * B[4] - B[1] * B[3]) * id;
    }
}

// Chronopoulos-Gear form of preconditioned CG (the iterates of standard PCG
// in exact arithmetic, one reduction point per iteration):
//   s_k = A z_k,  delta_k = z_k.s_k,  rho_k = r_k.z_k
//   k = 0: beta = 0, alpha = rho_0 / delta_0,            p = z, q = s
//   k > 0: beta = rho_k / rho_{k-1}, alpha = rho_k / (delta_k - beta rho_k / alpha_{k-1}),
//          p = z + beta p,  q = s + beta q
//   x += alpha p,  r -= alpha q,  z = M^-1 r
// so the SpMV gathers only z, which is complete when it runs.

// The solver's copy of H: its lower triangle's blocks in solver order
// (diagonal included), D*D contiguous row-major values each, one thread per
// value.  place[l] is stored block l's offset in H and 4 * row stride + flags
// (1: take the transpose of the block there; 2: diagonal, take the upper
// entries from the lower ones), so that the copy is the symmetric matrix of
// H's scalar lower triangle.
template <int D>
__global__ __launch_bounds__(kBlock) void k_sym_pack(int64_t n_sym, const int2* __restrict__ place,
                                                     const double* __restrict__ H, double* __restrict__ Hs)
{
    constexpr int DD = D * D;
    const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= n_sym * DD) return;
    const int64_t l = id / DD;
    const int m = (int)(id - l * DD);
    int i = m / D, j = m - i * D;
    const int2 pl = place[l];
    if ((pl.y & 1) || ((pl.y & 2) && i < j))
    {
        const int t = i;
        i = j;
        j = t;
    }
    Hs[id] = H[(int64_t)pl.x + (int64_t)i * (pl.y >> 2) + j];
}

// Progress and result of a solve in pinned host memory: the host launches only
// a few iterations ahead of it and never waits for the stream.  Plain
// system-scope stores, the state after the others have been acknowledged: a
// release would write back the XCD's L2 in every iteration.
__device__ __forceinline__ void report(PcgReport* h, double rr, double bb, int k, int breakdown, bool end)
{
    if (end)
    {
        __hip_atomic_store(&h->rr, rr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        __hip_atomic_store(&h->bb, bb, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        __hip_atomic_store(&h->iters, k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        __hip_atomic_store(&h->breakdown, breakdown, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    __hip_atomic_store(&h->state, end ? -1 : k + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// sol = x in handle order (solver entry i belongs to handle perm[i])
template <int D>
__device__ __forceinline__ void unpermute(int64_t nh, const int32_t* __restrict__ perm, const double* __restrict__ x,
                                          double* __restrict__ sol)
{
    for (int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; id < nh * D;
         id += (int64_t)gridDim.x * blockDim.x)
    {
        const int64_t i = id / D;
        sol[(int64_t)perm[i] * D + (id - i * D)] = x[id];
    }
}

template <int D>
__global__ __launch_bounds__(kBlock) void k_unpermute(int64_t nh, const int32_t* __restrict__ perm,
                                                      const double* __restrict__ x, double* __restrict__ sol)
{
    unpermute<D>(nh, perm, x, sol);
}

// CG iteration k, first half: termination test on rr_k = ||r_k||^2 (k = 0:
// ||b||^2, recorded), then s = (w I + H) z and partial z.s.  On termination
// the launch that finds it writes the solution in handle order instead (every
// block decides alike; done = k + 1 marks that launch, so that a block that
// starts late and already reads the flag still writes its share).  The
// termination flag, the residual partials and the first row group's data are
// all requested before the test, so their memory latencies overlap.  LPB
// lanes per block row, lane k takes blocks k, k + LPB, ... of the row, then a
// fixed tree.  H comes from the solver's copy: a row's columns ascend, so its
// blocks up to the diagonal are the stored blocks of the row in order, and an
// upper block is the transpose of stored block usrc (the lower block (v, u)
// it mirrors); every stored off-diagonal block is read twice per product.  XCD: the workgroups of one XCD (blockIdx % 8, the dispatch order
// across the eight XCDs) take a contiguous eighth of the row groups in
// order, so the block an upper block reads belongs to a row that the same
// XCD streams shortly after, and the second read can hit in that XCD's L2.
// Requires gridDim.x % 8 == 0 for XCD.  60^3 cube: 160 MB in 36 us (4.4 TB/s);
// the upper blocks' 72-byte pieces are separate cache lines for every lane.
template <int D, int LPB, bool XCD>
__global__ __launch_bounds__(kBlock) void k_spmv_sym(PcgSystem a, int Gs, int Gv, int k, const int* __restrict__ kdev)
{
    constexpr int DD = D * D;
    const int64_t nh = a.nh;
    const int32_t* __restrict__ bcol = a.bcol;
    const int32_t* __restrict__ usrc = a.usrc;
    const double* __restrict__ Hs = a.Hs;
    const double* __restrict__ z = a.z;
    PcgScalars* sc = a.sc;
    if (kdev) k = *kdev;
    __shared__ double sh[kBlock / 64][1], sh2[kBlock / 64][1];
    __shared__ int flag;
    const int done_v = threadIdx.x == 0 ? sc->done : 0;
    const double* rparts = a.parts + Gs + 2 * Gv + ((k + 1) & 1) * Gv;
    double rv[4];
    strided_fetch<kBlock, 4>(rparts, Gv, rv);
    const int lane = threadIdx.x % LPB;
    constexpr int rows_per_block = kBlock / LPB;
    const int64_t n_groups = (nh + rows_per_block - 1) / rows_per_block;
    int64_t g0, gstep, gend;
    if constexpr (XCD)
    {
        const int64_t per = (n_groups + 7) / 8;
        const int64_t x = blockIdx.x & 7;
        g0 = x * per + (blockIdx.x >> 3);
        gstep = gridDim.x >> 3;
        gend = min(n_groups, (x + 1) * per);
    }
    else
    {
        g0 = blockIdx.x;
        gstep = gridDim.x;
        gend = n_groups;
    }
    // the row's first two blocks of this lane: everything they need is loaded
    // before anything is used, so 16 blocks per row are in flight at once
    struct Two
    {
        double h[2][DD], z[2][D];
        bool tr[2];
    };
    int b0, nbu, s0, nlow;  // first block of the row, blocks, first stored block, stored blocks
    auto row_head = [&](int64_t u) {
        b0 = a.brow_ptr[u];
        nbu = a.brow_ptr[u + 1] - b0;
        s0 = a.sym_ptr[u];
        nlow = a.sym_ptr[u + 1] - s0;
    };
    auto load_block = [&](int kk, double* h, double* zv, bool& tr) {
        const int64_t v = bcol[b0 + kk];
        tr = kk >= nlow;
        const int us = usrc[max(0, b0 - s0 + kk - nlow)];  // (read by every lane: no branch before the block's loads)
        const int64_t si = tr ? us : s0 + kk;
        const double* __restrict__ hb = Hs + si * DD;
#pragma unroll
        for (int m = 0; m < DD; ++m) h[m] = hb[m];
#pragma unroll
        for (int j = 0; j < D; ++j) zv[j] = z[v * D + j];
    };
    auto add_block = [&](const double* h, const double* zv, bool tr, double* acc) {
#pragma unroll
        for (int i = 0; i < D; ++i)
#pragma unroll
            for (int j = 0; j < D; ++j) acc[i] += (tr ? h[j * D + i] : h[i * D + j]) * zv[j];
    };
    Two t2;
    auto load_two = [&](int64_t u) {
        row_head(u);
#pragma unroll
        for (int m = 0; m < 2; ++m)
            if (lane + m * LPB < nbu) load_block(lane + m * LPB, t2.h[m], t2.z[m], t2.tr[m]);
    };
    {
        const int64_t u = g0 * rows_per_block + threadIdx.x / LPB;
        if (g0 < gend && u < nh) load_two(u);
    }
    if (threadIdx.x == 0) flag = done_v;
    double racc[1] = { strided_rest<kBlock, 4>(rparts, Gv, rv) };
    block_totals<kBlock, 1>(racc, sh);  // its barrier publishes the flag
    if (flag != 0 && flag != k + 1) return;
    const double rr = racc[0];
    const double bb = k == 0 ? rr : sc->bb;
    const bool stop = !(rr > a.tol2 * bb) || k >= a.max_iters;  // (a NaN residual stops too)
    if (blockIdx.x == 0 && threadIdx.x == 0)
    {
        if (k == 0) sc->bb = bb;
        if (stop) sc->done = k + 1;
        report(a.host, rr, bb, k, 0, stop);
    }
    if (stop)
    {
        unpermute<D>(nh, a.perm, a.x, a.sol);
        return;
    }
    double zs[1] = { 0.0 };
    bool first = true;
    for (int64_t g = g0; g < gend; g += gstep)
    {
        const int64_t u = g * rows_per_block + threadIdx.x / LPB;
        double acc[D];
#pragma unroll
        for (int i = 0; i < D; ++i) acc[i] = 0.0;
        if (u < nh)
        {
            if (!first) load_two(u);
#pragma unroll
            for (int m = 0; m < 2; ++m)
                if (lane + m * LPB < nbu) add_block(t2.h[m], t2.z[m], t2.tr[m], acc);
            for (int kk = lane + 2 * LPB; kk < nbu; kk += LPB)
            {
                load_block(kk, t2.h[0], t2.z[0], t2.tr[0]);
                add_block(t2.h[0], t2.z[0], t2.tr[0], acc);
            }
        }
        first = false;
        static_assert(LPB == 8, "the sum over a row's lanes: quads, then 8 lanes");
#pragma unroll
        for (int i = 0; i < D; ++i)
        {
            acc[i] += dpp_move<0xB1>(acc[i]);   // quad_perm 1 0 3 2
            acc[i] += dpp_move<0x4E>(acc[i]);   // quad_perm 2 3 0 1
            acc[i] += dpp_move<0x141>(acc[i]);  // row_half_mirror
        }
        if (u < nh && lane == 0)
        {
#pragma unroll
            for (int i = 0; i < D; ++i)
            {
                const double zi = z[u * D + i];
                const double si = acc[i] + a.w * zi;
                a.s[u * D + i] = si;
                zs[0] += zi * si;
            }
        }
    }
    block_totals<kBlock, 1>(zs, sh2);
    if (threadIdx.x == 0) a.parts[blockIdx.x] = zs[0];
}

// ---------------------------------------------------------------------------
// Two-level preconditioner: additive coarse correction on handle aggregates
// ---------------------------------------------------------------------------
// z = D^-1 r + P A_c^-1 P^T r with A_c = P^T (w I + H) P.  P has KC columns per
// aggregate; its rows for handle v are R_v (D x KC): the identity on the
// translations and, for KC > D, the rotations omega about the aggregate's
// first handle, delta x_v = omega x dv (D = 3) or omega (-dv_1, dv_0) (D = 2).
// Every sum below runs in a fixed order (fixed lane assignment and a fixed
// tree), so the correction is bitwise reproducible.
template <int D, int KC>
__device__ __forceinline__ void coarse_rows(const double* __restrict__ dv, double R[D][KC])
{
#pragma unroll
    for (int i = 0; i < D; ++i)
#pragma unroll
        for (int c = 0; c < KC; ++c) R[i][c] = (c == i) ? 1.0 : 0.0;
    if constexpr (KC > D)
    {
        if constexpr (D == 3)
        {
            R[0][4] = dv[2];
            R[0][5] = -dv[1];
            R[1][3] = -dv[2];
            R[1][5] = dv[0];
            R[2][3] = dv[1];
            R[2][4] = -dv[0];
        }
        else if constexpr (D == 2)
        {
            R[0][2] = -dv[1];
            R[1][2] = dv[0];
        }
    }
}

// CG iteration k, second half: scalars, direction recurrences, x / r / z
// update; partials of rho_{k+1} = r.z and ||r||^2 into slot k & 1.  alpha and
// rho of iteration k are kept (slot k & 1 of sc) for iteration k + 1.
// Block b owns the handles [part_ptr[b], part_ptr[b + 1]) of solver order, a
// part of one aggregate, in chunks of 64: thread t updates variable t of the
// chunk (every vector access is a contiguous run), the D x D preconditioner
// blocks, the new residual and the lever arms pass through LDS for
// z = M^-1 r and (KC > 0) the first wave's sums R_v^T r_v of the restricted
// residual: block b = aggregate * ppa + p writes its KC sums to row p of
// rpart, so r_c is the sum of ppa rows and needs no kernel of its own.  At 10K
// handles the kernel is a chain of memory latencies, so the operands of the
// first chunk and all partials of the three scalars are requested before any
// is used: 100 x 100 grid update 6.5 us + restriction 3.2 -> 4.8 us in all;
// 30^3 tet cube 6.7 + 4.2 -> 6.6; 60^3, bound by 78 MB of vectors, 16.0 + 6.4
// -> 14.6 (5.3 TB/s).
//
// INIT (before iteration 0, k = -1): the block-Jacobi inverse from the
// solver's copy of H, x = 0, r = b, z = M^-1 r and the same partials.
constexpr int kUpdVerts = 64;

template <int D, int KC, bool INIT>
__global__ __launch_bounds__(kUpdVerts * D) void k_pcg_update(PcgSystem a, int Gs, int Gv, int k,
                                                              const int* __restrict__ kdev)
{
    constexpr int NT = kUpdVerts * D;
    constexpr int NW = D;  // waves
    constexpr int PB = PackedBlock<D>::n;
    constexpr int ND = (kUpdVerts * PB + NT - 1) / NT;  // packed block entries per thread and chunk
    constexpr bool ROT = KC > D;
    __shared__ double sh[NW][3], sh2[NW][2];
    __shared__ double sD[ND * NT];
    __shared__ double sR[NT];
    __shared__ double sV[ROT ? NT : 1];
    __shared__ int flag;
    PcgScalars* sc = a.sc;
    const int t = threadIdx.x;
    const int blk = blockIdx.x;
    if (INIT) k = -1;
    else if (kdev) k = *kdev;
    const int64_t lo = a.part_ptr[blk], hi = a.part_ptr[blk + 1];
    // operands of one chunk: this thread's variable and its share of the
    // chunk's packed preconditioner blocks
    double zc = 0.0, pc = 0.0, qc = 0.0, sc_ = 0.0, xc = 0.0, rc = 0.0, vc = 0.0, dc[ND];
    auto load = [&](int64_t c0) {
        const int64_t iv = c0 * D + t;
        if (iv < hi * D)
        {
            if constexpr (INIT)
                rc = a.b[(int64_t)a.perm[iv / D] * D + iv % D];
            else
            {
                zc = a.z[iv];
                pc = a.p[iv];
                qc = a.q[iv];
                sc_ = a.s[iv];
                xc = a.x[iv];
                rc = a.r[iv];
            }
            if constexpr (ROT) vc = a.dvec[iv];
        }
        if constexpr (!INIT)
        {
#pragma unroll
            for (int m = 0; m < ND; ++m)
            {
                const int64_t id = c0 * PB + t + (int64_t)m * NT;
                dc[m] = (t + m * NT < kUpdVerts * PB && id < hi * PB) ? a.Dinv[id] : 0.0;
            }
        }
    };
    double alpha = 0.0, beta = 0.0;
    if constexpr (INIT)
    {
        if (lo < hi) load(lo);
        if (blk == 0 && t == 0)
        {
            sc->done = 0;
            sc->k = 0;
        }
    }
    else
    {
        const int done_v = t == 0 ? sc->done : 0;
        const double rho_prev = k > 0 ? sc->rho_hist[(k + 1) & 1] : 1.0;
        const double alpha_prev = k > 0 ? sc->alpha_hist[(k + 1) & 1] : 1.0;
        // delta, r.(D^-1 r), (P^T r).(A_c^-1 P^T r): thread t adds the
        // partials t, t + NT, ... in order
        const double* __restrict__ pd = a.parts;
        const double* __restrict__ pr = a.parts + Gs + ((k + 1) & 1) * Gv;
        const double* __restrict__ pk = a.cparts + ((k + 1) & 1) * a.n_agg;  // n_agg: 0 without a correction
        double vd[6], vr[6], vk[3];
        strided_fetch<NT, 6>(pd, Gs, vd);
        strided_fetch<NT, 6>(pr, Gv, vr);
        strided_fetch<NT, 3>(pk, a.n_agg, vk);
        if (lo < hi) load(lo);  // in flight during the sums
        if (t == 0) flag = done_v;
        double tot[3] = { strided_rest<NT, 6>(pd, Gs, vd), strided_rest<NT, 6>(pr, Gv, vr),
                          strided_rest<NT, 3>(pk, a.n_agg, vk) };
        if constexpr (NT == 64) __syncthreads();
        block_totals<NT, 3>(tot, sh);
        if (flag) return;
        const double delta = tot[0], rho = tot[1] + tot[2];
        double den = delta;
        if (k > 0)
        {
            beta = rho / rho_prev;
            den = delta - beta * rho / alpha_prev;
            // p.Ap from the recurrence can cancel to <= 0 near convergence even
            // for a positive definite matrix: restart along z (beta = 0, p = z,
            // p.Ap = z.Az) instead of reporting a breakdown
            if (!(den > 0.0))
            {
                beta = 0.0;
                den = delta;
            }
        }
        if (!(den > 0.0))
        {
            // not positive definite along z: the same decision in every block
            if (blk == 0 && t == 0)
            {
                sc->done = -1;
                report(a.host, 0.0, 0.0, k, 1, true);
            }
            return;
        }
        alpha = rho / den;
        if (blk == 0 && t == 0)
        {
            sc->rho_hist[k & 1] = rho;
            sc->alpha_hist[k & 1] = alpha;
        }
    }
    double part[2] = { 0.0, 0.0 };  // r.z, ||r||^2
    double cr[KC > 0 ? KC : 1];
#pragma unroll
    for (int c = 0; c < (KC > 0 ? KC : 1); ++c) cr[c] = 0.0;
    for (int64_t c0 = lo; c0 < hi; c0 += kUpdVerts)
    {
        const int64_t iv = c0 * D + t;
        const bool in = iv < hi * D;
        double rv = 0.0;
        if constexpr (INIT)
        {
            if (c0 > lo) __syncthreads();  // the previous chunk's LDS reads are complete
            // inverse diagonal blocks of this chunk (threads 0 .. 63)
            if (t < kUpdVerts)
            {
                const int64_t v = c0 + t;
                double B[D * D], o[D * D];
                bool fr[D];
#pragma unroll
                for (int i = 0; i < D; ++i) fr[i] = false;
#pragma unroll
                for (int m = 0; m < D * D; ++m) o[m] = 0.0;
                if (v < hi)
                {
                    const int64_t h0 = (int64_t)a.perm[v] * D;
                    const int32_t dg = a.diag[v];
#pragma unroll
                    for (int i = 0; i < D; ++i)
                    {
                        fr[i] = a.free_h ? a.free_h[h0 + i] != 0 : true;
                        if (a.free_h) a.free_s[v * D + i] = fr[i] ? 1 : 0;
                    }
                    // reduced basis: a fixed component takes a unit row /
                    // column here and a zero row / column in the inverse (the
                    // free sub-block's inverse); a handle used by no element
                    // has no block: (w I + H) is w I there
#pragma unroll
                    for (int i = 0; i < D; ++i)
#pragma unroll
                        for (int j = 0; j < D; ++j)
                        {
                            const double hb = dg < 0 ? 0.0 : a.Hs[(int64_t)dg * (D * D) + i * D + j];
                            const double e = hb + (i == j ? (dg < 0 && !(a.w > 0.0) ? 1.0 : a.w) : 0.0);
                            B[i * D + j] = (fr[i] && fr[j]) ? e : (i == j ? 1.0 : 0.0);
                        }
                    invert_block<D>(B, o);
                }
                // the upper triangle: the inverse of a symmetric block is
                // symmetric (the cofactor products commute)
#pragma unroll
                for (int i = 0; i < D; ++i)
#pragma unroll
                    for (int j = i; j < D; ++j)
                    {
                        const double e = (fr[i] && fr[j] && !a.dense) ? o[i * D + j] : 0.0;
                        sD[t * PB + PackedBlock<D>::at(i, j)] = e;
                        if (v < hi) a.Dinv[v * PB + PackedBlock<D>::at(i, j)] = e;
                    }
            }
            if (in)
            {
                rv = (a.free_h && !a.free_h[(int64_t)a.perm[iv / D] * D + iv % D]) ? 0.0 : rc;
                a.x[iv] = 0.0;
                a.r[iv] = rv;
            }
        }
        else if (in)
        {
            const double pi = k > 0 ? fma(beta, pc, zc) : zc;
            const double qi = k > 0 ? fma(beta, qc, sc_) : sc_;
            a.p[iv] = pi;
            a.q[iv] = qi;
            a.x[iv] = xc + alpha * pi;
            rv = rc - alpha * qi;
            if (a.free_h && !a.free_s[iv]) rv = 0.0;  // reduced basis: no residual on fixed variables
            a.r[iv] = rv;
        }
        if (!INIT && c0 > lo) __syncthreads();  // the previous chunk's LDS reads are complete
        sR[t] = rv;
        if constexpr (ROT) sV[t] = vc;
        if constexpr (!INIT)
        {
#pragma unroll
            for (int m = 0; m < ND; ++m) sD[t + m * NT] = dc[m];
        }
        __syncthreads();
        if (c0 + kUpdVerts < hi) load(c0 + kUpdVerts);  // next chunk in flight during this one's z
        if (in)
        {
            const int vl = t / D, i = t - vl * D;
            double zi = 0.0;
#pragma unroll
            for (int j = 0; j < D; ++j) zi += sD[vl * PB + PackedBlock<D>::at(i, j)] * sR[vl * D + j];
            a.z[iv] = zi;
            part[0] += rv * zi;
            part[1] += rv * rv;
        }
        if constexpr (KC > 0)
        {
            if (t < kUpdVerts)  // sR is 0 past the part's end
            {
                double dv[D], R[D][KC];
#pragma unroll
                for (int i = 0; i < D; ++i) dv[i] = ROT ? sV[ROT ? t * D + i : 0] : 0.0;
                if (c0 + t >= hi)
                {
#pragma unroll
                    for (int i = 0; i < D; ++i) dv[i] = 0.0;
                }
                coarse_rows<D, KC>(dv, R);
#pragma unroll
                for (int i = 0; i < D; ++i)
#pragma unroll
                    for (int c = 0; c < KC; ++c) cr[c] += R[i][c] * sR[t * D + i];
            }
        }
    }
    if constexpr (KC > 0)
    {
        if (t < 64)
        {
#pragma unroll
            for (int c = 0; c < KC; ++c) cr[c] = wave_total(cr[c]);
            double v = cr[0];
#pragma unroll
            for (int c = 1; c < KC; ++c) v = t == c ? cr[c] : v;
            const int64_t ag = blk / a.ppa, p = blk - ag * a.ppa;
            if (t < KC) a.rpart[p * a.nc + ag * KC + t] = v;
        }
    }
    block_totals<NT, 2>(part, sh2);
    if (t == 0)
    {
        a.parts[Gs + (k & 1) * Gv + blk] = part[0];
        a.parts[Gs + 2 * Gv + (k & 1) * Gv + blk] = part[1];
    }
}

// sum over the 64 lanes of a wave, fixed xor tree (every lane gets the total)
template <int L>
__device__ __forceinline__ void wave_sum(double* v)
{
#pragma unroll
    for (int m = 0; m < L; ++m) v[m] = wave_total(v[m]);
}

// Lever arms dv_v = x_v - x_(first member of v's aggregate), in handle order
// (Galerkin sums) and in solver order (CG iterations).
template <int D>
__global__ __launch_bounds__(kBlock) void k_coarse_dvec(int64_t nh, const double* __restrict__ x,
                                                        const int32_t* __restrict__ agg_of,
                                                        const int32_t* __restrict__ agg_ptr,
                                                        const int32_t* __restrict__ perm, double* __restrict__ dvec_h,
                                                        double* __restrict__ dvec)
{
    const int64_t i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i0 >= nh) return;
    const int64_t v = perm[i0];
    const int64_t root = perm[agg_ptr[agg_of[v]]];
#pragma unroll
    for (int i = 0; i < D; ++i)
    {
        const double e = x[v * D + i] - x[root * D + i];
        dvec_h[v * D + i] = e;
        dvec[i0 * D + i] = e;
    }
}

// one wave per chunk of a coarse block pair's fine blocks (u, v): sum of
// R_u^T (H_uv + w I [u == v]) R_v over the chunk
template <int D, int KC>
__global__ __launch_bounds__(kBlock) void k_coarse_galerkin_chunk(int64_t n_gchunks,
                                                                  const int64_t* __restrict__ gchunk_ptr,
                                                                  const int32_t* __restrict__ pair_blocks,
                                                                  const int32_t* __restrict__ block_row,
                                                                  const int32_t* __restrict__ brow_ptr,
                                                                  const int32_t* __restrict__ bcol,
                                                                  const int32_t* __restrict__ row_ptr,
                                                                  const double* __restrict__ H, double w,
                                                                  const double* __restrict__ dvec,
                                                                  const unsigned char* __restrict__ free_vars,
                                                                  double* __restrict__ gpart)
{
    const int lane = threadIdx.x & 63;
    const int64_t ch = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    if (ch >= n_gchunks) return;
    double acc[KC * KC];
#pragma unroll
    for (int m = 0; m < KC * KC; ++m) acc[m] = 0.0;
    const int64_t c1 = gchunk_ptr[ch + 1];
    for (int64_t c = gchunk_ptr[ch] + lane; c < c1; c += 64)
    {
        const int32_t b = pair_blocks[c];
        const int u = block_row[b];
        const int v = bcol[b];
        const int b0 = brow_ptr[u];
        const int nbu = brow_ptr[u + 1] - b0;
        const int64_t base = (int64_t)row_ptr[D * u] + (int64_t)D * (b - b0);
        double Hb[D][D];
#pragma unroll
        for (int i = 0; i < D; ++i)
#pragma unroll
            for (int j = 0; j < D; ++j)
                Hb[i][j] = H[base + (int64_t)i * D * nbu + j] + ((u == v && i == j) ? w : 0.0);
        double Ru[D][KC], Rv[D][KC];
        coarse_rows<D, KC>(dvec + (int64_t)u * D, Ru);
        coarse_rows<D, KC>(dvec + (int64_t)v * D, Rv);
        if (free_vars)  // reduced basis: P restricted to the free variables
        {
#pragma unroll
            for (int i = 0; i < D; ++i)
#pragma unroll
                for (int c2 = 0; c2 < KC; ++c2)
                {
                    if (!free_vars[(int64_t)u * D + i]) Ru[i][c2] = 0.0;
                    if (!free_vars[(int64_t)v * D + i]) Rv[i][c2] = 0.0;
                }
        }
        double T[D][KC];
#pragma unroll
        for (int i = 0; i < D; ++i)
#pragma unroll
            for (int c2 = 0; c2 < KC; ++c2)
            {
                double t = 0.0;
#pragma unroll
                for (int j = 0; j < D; ++j) t += Hb[i][j] * Rv[j][c2];
                T[i][c2] = t;
            }
#pragma unroll
        for (int ca = 0; ca < KC; ++ca)
#pragma unroll
            for (int c2 = 0; c2 < KC; ++c2)
            {
                double t = 0.0;
#pragma unroll
                for (int i = 0; i < D; ++i) t += Ru[i][ca] * T[i][c2];
                acc[ca * KC + c2] += t;
            }
    }
    wave_sum<KC * KC>(acc);
#pragma unroll
    for (int m = 0; m < KC * KC; ++m)
        if (lane == m) gpart[ch * (KC * KC) + m] = acc[m];
}

// one thread per (pair, entry): chunk partials in order into A_c's (a, b) block
template <int KC>
__global__ __launch_bounds__(kBlock) void k_coarse_galerkin_pairs(int64_t n_pairs, const int32_t* __restrict__ pair_chunk,
                                                                  const int32_t* __restrict__ pair_ab,
                                                                  const double* __restrict__ gpart, int64_t nc,
                                                                  double* __restrict__ Ac)
{
    const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= n_pairs * KC * KC) return;
    const int64_t pr = id / (KC * KC);
    const int m = (int)(id % (KC * KC));
    double t = 0.0;
    for (int32_t ch = pair_chunk[pr]; ch < pair_chunk[pr + 1]; ++ch) t += gpart[(int64_t)ch * (KC * KC) + m];
    const int64_t a = pair_ab[2 * pr], bb = pair_ab[2 * pr + 1];
    Ac[(a * KC + m / KC) + (bb * KC + m % KC) * nc] = t;
}

// A_jj <- A_jj (1 + rel), and 1 where A_jj = 0: a positive semidefinite
// Galerkin matrix of a reduced basis (coarse directions with no free
// variable) becomes positive definite; the added directions prolong to zero.
__global__ __launch_bounds__(kBlock) void k_shift_diagonal(int64_t n, double* __restrict__ A, double rel)
{
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    const double a = A[j + j * n];
    A[j + j * n] = a == 0.0 ? 1.0 : a * (1.0 + rel);
}

// Coarse product and prolongation in one launch, one workgroup of
// kCoarseBlock threads per aggregate a: r_c = the ppa rows of restriction
// partials, y_a = rows a KC .. a KC + KC - 1 of A_c^-1 r_c (row i of the
// symmetric inverse is its contiguous column i; thread t takes the entries t,
// t + kCoarseBlock, ..., then a fixed wave tree and the waves' partials in
// order), one partial r_c[a] . y_a, then z_v += R_v y_a for every member v of
// the aggregate.  The first loads of every kind are issued before the
// termination flag is looked at (100 x 100 grid 5.7 -> 4.0 us, 60^3 cube 12.8
// -> 10.5 us, of which 30 MB are the FP32 inverse).  60^3 cube, 459
// aggregates, per CG iteration: 512 and 256 lanes alike, 1,024 2 us slower.
constexpr int kCoarseBlock = 512;

template <int D, int KC, class TA>
__device__ __forceinline__ void coarse_apply(const PcgSystem& a, const TA* __restrict__ Ainv, int slot, int done_v)
{
    constexpr int NW = kCoarseBlock / 64;
    __shared__ double wpart[NW][KC];
    __shared__ double y[KC], ry[KC];
    __shared__ int flag;
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const int64_t ag = blockIdx.x, nc = a.nc;
    const TA* __restrict__ col = Ainv + ag * KC * nc;
    const double* __restrict__ rpart = a.rpart;
    const int ppa = a.ppa;
    auto rc = [&](int64_t j) {
        double v[4];
#pragma unroll
        for (int p = 0; p < 4; ++p) v[p] = p < ppa ? rpart[p * nc + j] : 0.0;
        double e = ((v[0] + v[1]) + v[2]) + v[3];
        for (int p = 4; p < ppa; ++p) e += rpart[p * nc + j];
        return e;
    };
    double acc[KC];
#pragma unroll
    for (int c = 0; c < KC; ++c) acc[c] = 0.0;
    int64_t j = t;
    if (j < nc)
    {
        const double rj = rc(j);
#pragma unroll
        for (int c = 0; c < KC; ++c) acc[c] = (double)col[c * nc + j] * rj;
    }
    const double rown = t < KC ? rc(ag * KC + t) : 0.0;
    // this thread's first member
    const int64_t m0 = a.agg_ptr[ag], m1 = a.agg_ptr[ag + 1];
    double zv[D], dv[D];
    auto member = [&](int64_t v) {
#pragma unroll
        for (int i = 0; i < D; ++i)
        {
            zv[i] = a.z[v * D + i];
            dv[i] = KC > D ? a.dvec[v * D + i] : 0.0;
        }
    };
    if (m0 + t < m1) member(m0 + t);
    if (t == 0) flag = done_v;
    __syncthreads();
    if (flag) return;
    for (j += kCoarseBlock; j < nc; j += kCoarseBlock)
    {
        const double rj = rc(j);
#pragma unroll
        for (int c = 0; c < KC; ++c) acc[c] += (double)col[c * nc + j] * rj;
    }
    wave_sum<KC>(acc);
    if (lane == 0)
    {
#pragma unroll
        for (int c = 0; c < KC; ++c) wpart[wv][c] = acc[c];
    }
    __syncthreads();
    if (t < KC)
    {
        double v = 0.0;
#pragma unroll
        for (int w = 0; w < NW; ++w) v += wpart[w][t];
        y[t] = v;
        ry[t] = rown * v;
    }
    __syncthreads();
    if (t == 0)
    {
        double v = 0.0;
#pragma unroll
        for (int c = 0; c < KC; ++c) v += ry[c];
        a.cparts[slot * a.n_agg + ag] = v;
    }
    double ya[KC];
#pragma unroll
    for (int c = 0; c < KC; ++c) ya[c] = y[c];
    for (int64_t v = m0 + t; v < m1; v += kCoarseBlock)
    {
        if (v != m0 + t) member(v);
        double R[D][KC];
        coarse_rows<D, KC>(dv, R);
#pragma unroll
        for (int i = 0; i < D; ++i)
        {
            if (a.free_h && !a.free_s[v * D + i]) continue;
            double e = zv[i];
#pragma unroll
            for (int c = 0; c < KC; ++c) e += R[i][c] * ya[c];
            a.z[v * D + i] = e;
        }
    }
}

hipError_t launch_coarse_dvec(int d, int64_t nh, const double* x, const int32_t* agg_of, const int32_t* agg_ptr,
                              const int32_t* perm, double* dvec_h, double* dvec, hipStream_t s)
{
    if (nh == 0) return hipSuccess;
    const unsigned g = (unsigned)((nh + kBlock - 1) / kBlock);
    if (d == 1) k_coarse_dvec<1><<<g, kBlock, 0, s>>>(nh, x, agg_of, agg_ptr, perm, dvec_h, dvec);
    else if (d == 2) k_coarse_dvec<2><<<g, kBlock, 0, s>>>(nh, x, agg_of, agg_ptr, perm, dvec_h, dvec);
    else k_coarse_dvec<3><<<g, kBlock, 0, s>>>(nh, x, agg_of, agg_ptr, perm, dvec_h, dvec);
    return hipGetLastError();
}

template <int D, int KC>
static void galerkin_t(int64_t n_pairs, int64_t n_gchunks, const int64_t* gchunk_ptr, const int32_t* pair_chunk,
                       const int32_t* pair_blocks, const int32_t* pair_ab, const int32_t* block_row,
                       const int32_t* brow_ptr, const int32_t* bcol, const int32_t* row_ptr, const double* H, double w,
                       const double* dvec_h, const unsigned char* free_vars, int64_t nc, double* gpart, double* Ac,
                       hipStream_t s)
{
    const unsigned g1 = (unsigned)((n_gchunks * 64 + kBlock - 1) / kBlock);
    k_coarse_galerkin_chunk<D, KC><<<g1, kBlock, 0, s>>>(n_gchunks, gchunk_ptr, pair_blocks, block_row, brow_ptr,
                                                          bcol, row_ptr, H, w, dvec_h, free_vars, gpart);
    const unsigned g2 = (unsigned)((n_pairs * KC * KC + kBlock - 1) / kBlock);
    k_coarse_galerkin_pairs<KC><<<g2, kBlock, 0, s>>>(n_pairs, pair_chunk, pair_ab, gpart, nc, Ac);
}

hipError_t launch_coarse_galerkin(int d, int kc, int64_t nc, int64_t n_pairs, int64_t n_gchunks,
                                  const int64_t* gchunk_ptr, const int32_t* pair_chunk, const int32_t* pair_blocks,
                                  const int32_t* pair_ab, const int32_t* block_row, const int32_t* brow_ptr,
                                  const int32_t* bcol, const int32_t* row_ptr, const double* H, double w,
                                  const double* dvec_h, const unsigned char* free_vars, double* gpart, double* Ac,
                                  hipStream_t s)
{
    if (n_pairs == 0) return hipSuccess;
#define TAD_GALERKIN(DD, KK) galerkin_t<DD, KK>(n_pairs, n_gchunks, gchunk_ptr, pair_chunk, pair_blocks, pair_ab, \
                                                 block_row, brow_ptr, bcol, row_ptr, H, w, dvec_h, free_vars, nc, \
                                                 gpart, Ac, s)
    if (d == 3 && kc == 6) TAD_GALERKIN(3, 6);
    else if (d == 3 && kc == 3) TAD_GALERKIN(3, 3);
    else if (d == 2 && kc == 3) TAD_GALERKIN(2, 3);
    else if (d == 2 && kc == 2) TAD_GALERKIN(2, 2);
    else if (d == 1 && kc == 1) TAD_GALERKIN(1, 1);
    else return hipErrorInvalidValue;
#undef TAD_GALERKIN
    return hipGetLastError();
}

hipError_t launch_shift_diagonal(int64_t n, double* A, double rel, hipStream_t s)
{
    if (n == 0) return hipSuccess;
    k_shift_diagonal<<<(unsigned)((n + kBlock - 1) / kBlock), kBlock, 0, s>>>(n, A, rel);
    return hipGetLastError();
}

// |A| row sums, one wave per row: lane-strided partial sums, then a fixed
// wave tree; k_rowmax then takes their maximum (||A||_inf).
__global__ __launch_bounds__(kBlock) void k_abs_rowsum(int64_t n, const double* __restrict__ A,
                                                       double* __restrict__ rowsum)
{
    const int lane = threadIdx.x & 63;
    const int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    if (i >= n) return;
    double t = 0.0;
    for (int64_t j = lane; j < n; j += 64) t += fabs(A[i * n + j]);
    wave_sum<1>(&t);
    if (lane == 0) rowsum[i] = t;
}

// out[0] = max of the row sums.  With `mode` (the second norm, of A^-1): the
// coarse correction the CG iterations apply, decided here so that the host
// need not wait for it: 0 none (the sweeps met a pivot that was not positive:
// A_c is not positive definite at working precision), 2 the FP32 copy, where
// 2^-22 kappa_inf <= `change` bounds the relative change of the correction
// by the copy's diagonal shift (2^-23 ||A^-1||_inf, small against the smallest
// eigenvalue of A^-1, >= 1 / ||A||_inf), 1 the FP64 inverse otherwise.
__global__ __launch_bounds__(kBlock) void k_rowmax(int64_t n, const double* __restrict__ rowsum,
                                                   double* __restrict__ out, const double* __restrict__ norm_a,
                                                   const int* __restrict__ info, double change, int* __restrict__ mode,
                                                   int* __restrict__ mode_host)
{
    __shared__ double sh[kBlock];
    double m = 0.0;
    for (int64_t i = threadIdx.x; i < n; i += kBlock) m = fmax(m, rowsum[i]);
    sh[threadIdx.x] = m;
    __syncthreads();
    for (int off = kBlock / 2; off > 0; off >>= 1)
    {
        if ((int)threadIdx.x < off) sh[threadIdx.x] = fmax(sh[threadIdx.x], sh[threadIdx.x + off]);
        __syncthreads();
    }
    if (threadIdx.x != 0) return;
    out[0] = sh[0];
    if (!mode) return;
    const double kappa = norm_a[0] * sh[0];
    const int v = info[0] != 0 ? 0 : (kappa < 1.0 / 0.0 && ldexp(kappa, -22) <= change) ? 2 : 1;
    mode[0] = v;
    mode_host[0] = v;
}

// A32 = fl32(A + delta I), delta = 2^-23 norm[0], when the iterations read it
__global__ __launch_bounds__(kBlock) void k_coarse_to32(int64_t n, const double* __restrict__ A,
                                                        const double* __restrict__ norm, const int* __restrict__ mode,
                                                        float* __restrict__ A32)
{
    if (mode[0] != 2) return;
    const double delta = ldexp(norm[0], -23);
    const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= n * n) return;
    const int64_t i = id / n, j = id - i * n;
    A32[id] = (float)(A[id] + (i == j ? delta : 0.0));
}

hipError_t launch_abs_rowmax(int64_t n, const double* A, double* rowsum, double* out, hipStream_t s)
{
    if (n == 0) return hipSuccess;
    k_abs_rowsum<<<(unsigned)((n * 64 + kBlock - 1) / kBlock), kBlock, 0, s>>>(n, A, rowsum);
    k_rowmax<<<1, kBlock, 0, s>>>(n, rowsum, out, nullptr, nullptr, 0.0, nullptr, nullptr);
    return hipGetLastError();
}

hipError_t launch_coarse_mode(int64_t n, const double* Ainv, double* rowsum, double* norms, const int* info,
                              double change, int* mode, int* mode_host, float* A32, hipStream_t s)
{
    if (n == 0) return hipSuccess;
    k_abs_rowsum<<<(unsigned)((n * 64 + kBlock - 1) / kBlock), kBlock, 0, s>>>(n, Ainv, rowsum);
    k_rowmax<<<1, kBlock, 0, s>>>(n, rowsum, norms + 1, norms, info, change, mode, mode_host);
    k_coarse_to32<<<(unsigned)((n * n + kBlock - 1) / kBlock), kBlock, 0, s>>>(n, Ainv, norms + 1, mode, A32);
    return hipGetLastError();
}

constexpr int kSpmvLanes = 8;

int pcg_spmv_groups(int64_t nh)
{
    // SpMV: kSpmvLanes lanes per block row, at most 1,024 workgroups (60^3
    // tet cube, 227K block rows: 8 lanes and 1,024 workgroups 40.7 us per
    // product against 42.1 with 768, 49.4 with 512, 43.1 with 1,536 and 44.8
    // with 2,048; 16 lanes with 2,048 workgroups 47.3, 4 lanes with 1,536
    // 50.1), a multiple of 8 (the XCDs) from 8 on
    const int64_t rows_per_block = kBlock / kSpmvLanes;
    const int64_t gs = std::max<int64_t>(1, std::min<int64_t>((nh + rows_per_block - 1) / rows_per_block, 1024));
    return (int)(gs < 8 ? gs : (gs + 7) / 8 * 8);
}

int64_t pcg_parts_size(int64_t Gs, int64_t Gv) { return Gs + 4 * Gv; }

hipError_t launch_sym_pack(int d, int64_t n_sym, const int32_t* place, const double* H, double* sym_H, hipStream_t s)
{
    if (n_sym == 0) return hipSuccess;
    const unsigned grid = (unsigned)((n_sym * d * d + kBlock - 1) / kBlock);
    const int2* pl = reinterpret_cast<const int2*>(place);
    if (d == 1) k_sym_pack<1><<<grid, kBlock, 0, s>>>(n_sym, pl, H, sym_H);
    else if (d == 2) k_sym_pack<2><<<grid, kBlock, 0, s>>>(n_sym, pl, H, sym_H);
    else k_sym_pack<3><<<grid, kBlock, 0, s>>>(n_sym, pl, H, sym_H);
    return hipGetLastError();
}

template <int D>
static void spmv_t(const PcgSystem& a, int k, const int* kdev, hipStream_t s)
{
    if (a.Gs % 8 == 0) k_spmv_sym<D, kSpmvLanes, true><<<a.Gs, kBlock, 0, s>>>(a, a.Gs, a.Gv, k, kdev);
    else k_spmv_sym<D, kSpmvLanes, false><<<a.Gs, kBlock, 0, s>>>(a, a.Gs, a.Gv, k, kdev);
}

template <int D, int KC>
static void update_t(const PcgSystem& a, int k, const int* kdev, bool init, hipStream_t s)
{
    if (init) k_pcg_update<D, KC, true><<<a.Gv, kUpdVerts * D, 0, s>>>(a, a.Gs, a.Gv, k, kdev);
    else k_pcg_update<D, KC, false><<<a.Gv, kUpdVerts * D, 0, s>>>(a, a.Gs, a.Gv, k, kdev);
}

static hipError_t update_any(int d, const PcgSystem& a, int k, const int* kdev, bool init, hipStream_t s)
{
    if (d == 3 && a.kc == 6) update_t<3, 6>(a, k, kdev, init, s);
    else if (d == 3 && a.kc == 3) update_t<3, 3>(a, k, kdev, init, s);
    else if (d == 3 && a.kc == 0) update_t<3, 0>(a, k, kdev, init, s);
    else if (d == 2 && a.kc == 3) update_t<2, 3>(a, k, kdev, init, s);
    else if (d == 2 && a.kc == 2) update_t<2, 2>(a, k, kdev, init, s);
    else if (d == 2 && a.kc == 0) update_t<2, 0>(a, k, kdev, init, s);
    else if (d == 1 && a.kc == 1) update_t<1, 1>(a, k, kdev, init, s);
    else if (d == 1 && a.kc == 0) update_t<1, 0>(a, k, kdev, init, s);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

// a.coarse_mode: 2 the FP32 copy, 1 the FP64 inverse, 0 no correction (z stays
// D^-1 r and r_c . y_c is 0).
template <int D, int KC>
__global__ __launch_bounds__(kCoarseBlock) void k_coarse_apply_prolong(PcgSystem a, int k,
                                                                       const int* __restrict__ kdev)
{
    const int done_v = threadIdx.x == 0 ? a.sc->done : 0;
    const int slot = (kdev ? *kdev : k) & 1;
    const int mode = a.coarse_mode[0];
    if (mode == 2) coarse_apply<D, KC, float>(a, a.Ainv32, slot, done_v);
    else if (mode == 1) coarse_apply<D, KC, double>(a, a.Ainv, slot, done_v);
    else if (threadIdx.x == 0) a.cparts[slot * a.n_agg + blockIdx.x] = 0.0;
}

// A small system's dense preconditioner: A = w I + H in FP64 (column-major
// n x n, lower triangle, zeroed by the caller) from the solver's copy in
// handle order, one thread per row of A; rows and columns of fixed variables
// (and rows no element has, for w = 0) are the identity's.
template <int D>
__global__ __launch_bounds__(kBlock) void k_dense_fill(PcgSystem a, double* __restrict__ A)
{
    const int64_t n = a.nh * D;
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= n) return;
    const int64_t u = r / D;
    const int i = (int)(r - u * D);
    const bool fr = a.free_h ? a.free_h[r] != 0 : true;
    const int32_t s0 = a.sym_ptr[u], s1 = a.sym_ptr[u + 1], b0 = a.brow_ptr[u];
    for (int32_t l = s0; l < s1; ++l)
    {
        const int64_t v = a.bcol[b0 + (l - s0)];
#pragma unroll
        for (int j = 0; j < D; ++j)
        {
            const int64_t c = v * D + j;
            if (c >= r || !fr || (a.free_h && !a.free_h[c])) continue;
            A[r + c * n] = a.Hs[(int64_t)l * (D * D) + i * D + j];
        }
    }
    const int32_t dg = a.diag[u];
    const double h = dg < 0 ? 0.0 : a.Hs[(int64_t)dg * (D * D) + i * D + i];
    A[r + r * n] = !fr ? 1.0 : h + (dg < 0 && !(a.w > 0.0) ? 1.0 : a.w);
}

// z = A^-1 r for the dense preconditioner, one wave per row (four per
// workgroup), with the workgroup's partial of r.z.
__global__ __launch_bounds__(kBlock) void k_dense_apply(PcgSystem a, int64_t n, int k, const int* __restrict__ kdev)
{
    constexpr int NW = kBlock / 64;
    __shared__ double sh[NW];
    __shared__ int flag;
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const int done_v = t == 0 ? a.sc->done : 0;
    const int slot = (kdev ? *kdev : k) & 1;
    const int64_t row = (int64_t)blockIdx.x * NW + wv;
    double acc = 0.0;
    if (row < n)
    {
        const double* __restrict__ m = a.Ainv + row * n;
        const double* __restrict__ r = a.r;
        int64_t j = lane;
        for (; j + 7 * 64 < n; j += 8 * 64)
        {
            double mv[8], rv[8];
#pragma unroll
            for (int q = 0; q < 8; ++q)
            {
                mv[q] = m[j + 64 * q];
                rv[q] = r[j + 64 * q];
            }
#pragma unroll
            for (int q = 0; q < 8; ++q) acc = fma(mv[q], rv[q], acc);
        }
        for (; j < n; j += 64) acc = fma(m[j], r[j], acc);
    }
    if (t == 0) flag = done_v;
    acc = wave_total(acc);
    __syncthreads();
    if (flag) return;
    if (lane == 0)
    {
        if (row < n) a.z[row] = acc;
        sh[wv] = row < n ? acc * a.r[row] : 0.0;
    }
    __syncthreads();
    if (t == 0)
    {
        double v = sh[0];
#pragma unroll
        for (int w = 1; w < NW; ++w) v += sh[w];
        a.cparts[slot * a.n_agg + blockIdx.x] = v;
    }
}

hipError_t launch_dense_fill(int d, const PcgSystem& a, double* A, hipStream_t s)
{
    const int64_t n = a.nh * d;
    hipError_t e = launch_fill(A, n * n, 0.0, s);
    if (e != hipSuccess) return e;
    const unsigned grid = (unsigned)((n + kBlock - 1) / kBlock);
    if (d == 1) k_dense_fill<1><<<grid, kBlock, 0, s>>>(a, A);
    else if (d == 2) k_dense_fill<2><<<grid, kBlock, 0, s>>>(a, A);
    else k_dense_fill<3><<<grid, kBlock, 0, s>>>(a, A);
    return hipGetLastError();
}

int64_t dense_apply_groups(int64_t n) { return (n + kBlock / 64 - 1) / (kBlock / 64); }

template <int D, int KC>
static void coarse_t(const PcgSystem& a, int k, const int* kdev, hipStream_t s)
{
    k_coarse_apply_prolong<D, KC><<<(unsigned)a.n_agg, kCoarseBlock, 0, s>>>(a, k, kdev);
}

// z += P A_c^-1 P^T r with the restricted residual's parts of the last update,
// or z = A^-1 r (dense)
static hipError_t coarse_any(int d, const PcgSystem& a, int k, const int* kdev, hipStream_t s, Timer* timer)
{
    if (a.kc == 0 && !a.dense) return hipSuccess;
    if (timer) timer->begin("pcg_coarse", s);
    if (a.dense) k_dense_apply<<<(unsigned)a.n_agg, kBlock, 0, s>>>(a, a.nh * d, k, kdev);
    else if (d == 3 && a.kc == 6) coarse_t<3, 6>(a, k, kdev, s);
    else if (d == 3 && a.kc == 3) coarse_t<3, 3>(a, k, kdev, s);
    else if (d == 2 && a.kc == 3) coarse_t<2, 3>(a, k, kdev, s);
    else if (d == 2 && a.kc == 2) coarse_t<2, 2>(a, k, kdev, s);
    else if (d == 1 && a.kc == 1) coarse_t<1, 1>(a, k, kdev, s);
    else return hipErrorInvalidValue;
    if (timer) timer->end("pcg_coarse", s);
    return hipGetLastError();
}

hipError_t launch_pcg_init(int d, const PcgSystem& a, hipStream_t s)
{
    const hipError_t e = update_any(d, a, -1, nullptr, true, s);
    return e != hipSuccess ? e : coarse_any(d, a, -1, nullptr, s, nullptr);
}

hipError_t launch_pcg_iteration(int d, const PcgSystem& a, int k, bool with_update, hipStream_t s, Timer* timer,
                                bool read_k)
{
    const int* kdev = read_k ? &a.sc->k : nullptr;
    if (timer) timer->begin("spmv", s);
    if (d == 1) spmv_t<1>(a, k, kdev, s);
    else if (d == 2) spmv_t<2>(a, k, kdev, s);
    else spmv_t<3>(a, k, kdev, s);
    if (timer) timer->end("spmv", s);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || !with_update) return e;
    if (timer) timer->begin("pcg_update", s);
    e = update_any(d, a, k, kdev, false, s);
    if (timer) timer->end("pcg_update", s);
    return e != hipSuccess ? e : coarse_any(d, a, k, kdev, s, timer);
}

hipError_t launch_pcg_solution(int d, const PcgSystem& a, hipStream_t s)
{
    const unsigned grid = (unsigned)std::max<int64_t>(1, std::min<int64_t>((a.nh * d + kBlock - 1) / kBlock, 1024));
    if (d == 1) k_unpermute<1><<<grid, kBlock, 0, s>>>(a.nh, a.perm, a.x, a.sol);
    else if (d == 2) k_unpermute<2><<<grid, kBlock, 0, s>>>(a.nh, a.perm, a.x, a.sol);
    else k_unpermute<3><<<grid, kBlock, 0, s>>>(a.nh, a.perm, a.x, a.sol);
    return hipGetLastError();
}

__global__ void k_pcg_advance(PcgScalars* sc)
{
    if (threadIdx.x == 0) sc->k += 1;
}

hipError_t launch_pcg_advance(PcgScalars* sc, hipStream_t s)
{
    k_pcg_advance<<<1, 64, 0, s>>>(sc);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Per-segment energy sums
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_segment_sum(const double* __restrict__ elem_f,
                                                        const int64_t* __restrict__ ranges, int n_terms,
                                                        int64_t n_seg, double* __restrict__ out)
{
    __shared__ double sh[kBlock];
    const double s = segment_total(elem_f, ranges, n_terms, n_seg, blockIdx.x, sh);
    if (threadIdx.x == 0) out[blockIdx.x] = s;
}

hipError_t launch_segment_sum(const double* elem_f, const int64_t* ranges, int n_terms, int64_t n_seg, double* out,
                              hipStream_t s)
{
    if (n_seg == 0) return hipSuccess;
    k_segment_sum<<<(unsigned)n_seg, kBlock, 0, s>>>(elem_f, ranges, n_terms, n_seg, out);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Dual self test (reference operator known answers)
// ---------------------------------------------------------------------------
__global__ void k_selftest_dual(int which, double xv, double yv, double* out)
{
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    const Dual<2, double> x = dual_var<2, double>(xv, 0), y = dual_var<2, double>(yv, 1);
    Dual<2, double> f;
    switch (which)
    {
        case 0: f = sqr(x) / y; break;
        case 1:
        {
            const Dual<2, double> a = 0.5 * sqr(x) - sqr(y) + 2.0 * x - y;
            const Dual<2, double> b = -sqr(x - 2.0) - sqr(y - 3.0) + 1.0;
            f = a / b;
            break;
        }
        case 2: f = (sqr(x) + x) * (sqr(y) - y) / (y - 1.0); break;
        default: f = -(x * y) + x - y + 2.0 * x * 3.0 - 1.0; break;
    }
    out[0] = f.v;
    out[1] = f.g[0];
    out[2] = f.g[1];
    out[3] = f.h[Sym<2>::idx(0, 0)];
    out[4] = f.h[Sym<2>::idx(0, 1)];
    out[5] = f.h[Sym<2>::idx(0, 1)];
    out[6] = f.h[Sym<2>::idx(1, 1)];
}

hipError_t launch_selftest_dual(int which, double x, double y, double* out_dev, hipStream_t s)
{
    k_selftest_dual<<<1, 64, 0, s>>>(which, x, y, out_dev);
    return hipGetLastError();
}

} // namespace tad
