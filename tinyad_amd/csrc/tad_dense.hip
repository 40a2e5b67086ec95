// Dense symmetric positive definite inverse (gfx950) for the coarse matrix of
// the two-level preconditioner: A^-1 by blocked Gauss-Jordan sweeps (the
// sweep operator, Beaton 1964 / Goodnight 1979: sweeping every pivot of an
// SPD matrix turns it into -A^-1; without pivoting, every pivot block is a
// Schur complement and stays positive definite).  Per 64 x 64 pivot block K,
// with Q = M_KK^-1, C_I = M_KI and W_J = Q M_KJ:
//   M_IJ -= C_I^T W_J  (I, J != K), M_KJ = W_J, M_IK = W_I^T, M_KK = -Q
// The matrix is padded to a multiple of 64 with identity rows and columns
// (decoupled: their part of the result is -I and is dropped) and kept as its
// lower 64 x 64 tiles, 32 KB contiguous each, column-major inside; diagonal
// tiles and pivot inverses stay symmetric to the bit at every step.  (That is
// what keeps an almost singular A usable, e.g. an unpinned mesh's coarse
// matrix with its rigid motions at the projection's eps: the rounding errors
// of one-sided updates are antisymmetric and of size kappa eps |A^-1|, and
// reading one triangle of them made the preconditioner indefinite.)  Products
// use v_mfma_f64_16x16x4_f64; every sum has a fixed order (deterministic).
// The reference factorizes its whole Hessian with SimplicialLDLT instead
// (NewtonDirection.hh:34-41); this inverse only serves the preconditioner.
//
// What bounds it: the pivot blocks follow each other, so at n = 500 .. 1,500
// the time is the chain of one pivot step (a launch, two tile products and a
// 64 x 64 inverse), not arithmetic (2 n^3 flops) or memory.  Hence one launch
// per pivot block: every workgroup forms the W_J it needs itself (64^3 flops
// more per strip, no panel launch), the tiles are read from one copy of the
// matrix and written to another (no ordering between workgroups), and the
// first workgroup of a step inverts the next pivot block as soon as it has
// updated it, beside the other tiles' updates.  Only lower tiles are kept:
// half the flops and bytes of the full square.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cstdint>
#include "tad_internal.hpp"

namespace tad {

namespace {

constexpr int kTile = 64;
constexpr int kTT = kTile * kTile;
constexpr int kSub = 16;  // pivot columns per blocked step inside a tile's inverse
typedef double tad_v4d __attribute__((ext_vector_type(4)));

// Operand tiles in LDS, both stored [outer index][k] with one double of
// padding per row: A(r, k) = As[r][k], B(k, c) = Bs[c][k].
typedef double Tile[kTile][kTile + 1];

// 1 / d by the hardware reciprocal and two Newton steps (within 1 ulp for
// normal d; the pivots are checked to be positive and finite)
__device__ __forceinline__ double pivot_rcp(double d)
{
    double y = __builtin_amdgcn_rcp(d);
    y = fma(fma(-d, y, 1.0), y, y);
    y = fma(fma(-d, y, 1.0), y, y);
    return y;
}

// lane K of every 16-lane row to all lanes of its row (DPP row_newbcast)
template <int K>
__device__ __forceinline__ double row_bcast(double v)
{
    int2 u = __builtin_bit_cast(int2, v);
    u.x = __builtin_amdgcn_update_dpp(0, u.x, 0x150 + K, 0xf, 0xf, true);
    u.y = __builtin_amdgcn_update_dpp(0, u.y, 0x150 + K, 0xf, 0xf, true);
    return __builtin_bit_cast(double, u);
}

__device__ __forceinline__ double lane_value(double v, int lane)
{
    int2 u = __builtin_bit_cast(int2, v);
    u.x = __builtin_amdgcn_readlane(u.x, lane);
    u.y = __builtin_amdgcn_readlane(u.y, lane);
    return __builtin_bit_cast(double, u);
}

// 16-lane row G of the wave to all four rows (two lane swaps in the VALU; an
// LDS permute here would add its latency to every pivot)
template <int G>
__device__ __forceinline__ unsigned rows_from(unsigned v)
{
    const auto h = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    const unsigned x = h[G / 2];  // rows 2 (G / 2), 2 (G / 2) + 1 in both halves
    const auto q = __builtin_amdgcn_permlane16_swap(x, x, false, false);
    return q[G % 2];
}

template <int G>
__device__ __forceinline__ double rows_from(double v)
{
    uint2 u = __builtin_bit_cast(uint2, v);
    u.x = rows_from<G>(u.x);
    u.y = rows_from<G>(u.y);
    return __builtin_bit_cast(double, u);
}

// One scalar sweep of a 16 x 16 block held by one wave: lane l has column
// l % 16, rows 4 m + l / 16 in a[m] (the MFMA result layout); piv collects the pivots (lane K of
// every row).  a_ij -= (a_iK a_Kj) / d, rounded in the same way for (i, j) and
// (j, i), so a symmetric block stays symmetric to the bit; the pivot column
// goes through the same product (0 - (a_iK * -1) / d): the chain of one step
// is what the whole inverse costs, so it has no branches and few selects.
template <int K>
__device__ __forceinline__ void sweep16_step(double a[4], int j, int g, double& piv)
{
    constexpr int gk = K % 4, mk = K / 4;
    const double d = lane_value(a[mk], gk * 16 + K);
    const bool is_col = j == K;
    const double row = is_col ? -1.0 : rows_from<gk>(a[mk]);
    piv = is_col ? d : piv;
    double t[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) t[m] = row_bcast<K>(a[m]) * row;
    const double rd = pivot_rcp(d);
#pragma unroll
    for (int m = 0; m < 4; ++m)
    {
        const double v = fma(-t[m], rd, is_col ? 0.0 : a[m]);
        a[m] = (m == mk && g == gk) ? row * rd : v;
    }
}

template <int K>
__device__ __forceinline__ void sweep16(double a[4], int j, int g, double& piv)
{
    sweep16_step<K>(a, j, g, piv);
    if constexpr (K + 1 < kSub) sweep16<K + 1>(a, j, g, piv);
}

// P (64 x 64, symmetric, both triangles) <- -P^-1 by four blocked sweeps of 16
// pivots; 256 threads, T is 64 x 65 doubles of scratch.  The 64 scalar sweeps
// are one chain (about 340 cycles each); wave 0 runs them in registers, and
// updates and sweeps the next pivot block while waves 1-3 write the pivot
// rows and columns and update the other 16 x 16 tiles by MFMA.  (64 scalar
// sweeps over the whole tile with a barrier each took 32 us; this form 12 us.)
__device__ __forceinline__ bool tile_inverse(Tile& P, Tile& T)
{
    typedef double Sub[kSub][kSub + 1];
    typedef double Panel[kSub][kTile + 1];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int j = lane % 16, g = lane / 16;
    Sub* Q16 = reinterpret_cast<Sub*>(&T[0][0]);          // two of 16 x 17
    Panel& Wl = *reinterpret_cast<Panel*>(&T[16][0]);     // W = Q P_K*, 16 x 65
    Panel& Cl = *reinterpret_cast<Panel*>(&T[32][0]);     // P_K*, 16 x 65
    static_assert(2 * kSub * (kSub + 1) <= 16 * (kTile + 1), "scratch layout");
    bool bad = false;
    auto sweep = [&](double a[4], Sub& Q) {
        double piv = 1.0;
        sweep16<0>(a, j, g, piv);
        bad = bad || __any(!(piv > 0.0) || !(piv < 1.0 / 0.0));
#pragma unroll
        for (int m = 0; m < 4; ++m) Q[4 * m + g][j] = -a[m];
    };
    if (w == 0)
    {
        double a[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) a[m] = P[4 * m + g][j];
        sweep(a, Q16[0]);
    }
    for (int kb = 0; kb < kTile / kSub; ++kb)
    {
        const int o = kSub * kb;
        const Sub& Q = Q16[kb & 1];
        __syncthreads();
        {
            tad_v4d acc = { 0.0, 0.0, 0.0, 0.0 };
#pragma unroll
            for (int q = 0; q < 4; ++q)
            {
                const double c = P[o + 4 * q + g][16 * w + j];
                Cl[4 * q + g][16 * w + j] = c;
                acc = __builtin_amdgcn_mfma_f64_16x16x4f64(Q[j][4 * q + g], c, acc, 0, 0, 0);
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) Wl[4 * q + g][16 * w + j] = acc[q];
        }
        __syncthreads();
        if (w == 0)
        {
            if (kb + 1 == kTile / kSub) continue;
            // the next pivot block, both D and its transpose (the same sums in
            // the same order): the lower half of D and its mirror
            const int b = 16 * (kb + 1);
            tad_v4d d, dt;
#pragma unroll
            for (int q = 0; q < 4; ++q) d[q] = P[b + 4 * q + g][b + j];
            dt = d;
#pragma unroll
            for (int q = 0; q < 4; ++q)
            {
                const double c = Cl[4 * q + g][b + j], v = Wl[4 * q + g][b + j];
                d = __builtin_amdgcn_mfma_f64_16x16x4f64(-c, v, d, 0, 0, 0);
                dt = __builtin_amdgcn_mfma_f64_16x16x4f64(v, -c, dt, 0, 0, 0);
            }
            double a[4];
#pragma unroll
            for (int m = 0; m < 4; ++m) a[m] = 4 * m + g >= j ? d[m] : dt[m];
            sweep(a, Q16[(kb + 1) & 1]);
            continue;
        }
        if (w == 1)  // pivot row and -Q
        {
#pragma unroll
            for (int J = 0; J < 4; ++J)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    P[o + 4 * q + g][16 * J + j] = J == kb ? -Q[4 * q + g][j] : Wl[4 * q + g][16 * J + j];
        }
        int turn = 0;  // lower tiles go round waves 3, 2, 1
#pragma unroll
        for (int I = 0; I < 4; ++I)
        {
            if (I == kb) continue;
            if (w == 2)
            {
#pragma unroll
                for (int q = 0; q < 4; ++q) P[16 * I + 4 * q + g][o + j] = Wl[j][16 * I + 4 * q + g];
            }
#pragma unroll
            for (int J = 0; J <= I; ++J)
            {
                if (J == kb || (I == J && I == kb + 1)) continue;
                if (turn++ % 3 != 3 - w) continue;
                tad_v4d acc;
#pragma unroll
                for (int q = 0; q < 4; ++q) acc[q] = P[16 * I + 4 * q + g][16 * J + j];
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(-Cl[4 * q + g][16 * I + j], Wl[4 * q + g][16 * J + j],
                                                               acc, 0, 0, 0);
#pragma unroll
                for (int q = 0; q < 4; ++q)
                {
                    const int r = 16 * I + 4 * q + g, c = 16 * J + j;
                    if (I == J && r < c) continue;
                    P[r][c] = acc[q];
                    P[c][r] = acc[q];
                }
            }
        }
    }
    __syncthreads();
    return bad;
}

// Q (column-major tile in memory) = P^-1 for the pivot block in LDS; info[0]
// = 1 when a pivot is not positive and finite (clear: 0 otherwise).
__device__ __forceinline__ void pivot_to(Tile& P, Tile& T, double* __restrict__ Q, int* __restrict__ info, bool clear)
{
    const bool bad = tile_inverse(P, T);  // known to wave 0
#pragma unroll
    for (int p = 0; p < 16; ++p)
    {
        const int e = threadIdx.x + 256 * p;
        Q[e] = -P[e / kTile][e % kTile];
    }
    if (threadIdx.x == 0 && (bad || clear)) info[0] = bad ? 1 : 0;
}

__host__ __device__ __forceinline__ int64_t tile_at(int64_t I, int64_t J)  // lower tile (I >= J)
{
    return (I * (I + 1) / 2 + J) * kTT;
}

// Lower tiles of A (n x n, column-major, symmetric) padded with identity, and
// the first pivot block's inverse; one workgroup per tile (I = row of the
// grid's triangle).
__global__ __launch_bounds__(256) void k_sweep_load(int64_t n, const double* __restrict__ A, double* __restrict__ S,
                                                    double* __restrict__ Q, int* __restrict__ info, bool clear)
{
    __shared__ Tile P, T;
    int64_t I = 0, J = blockIdx.x;
    while (J > I) J -= ++I;
    double* __restrict__ out = S + tile_at(I, J);
#pragma unroll
    for (int p = 0; p < 16; ++p)
    {
        const int e = threadIdx.x + 256 * p;
        const int r = e % kTile, c = e / kTile;
        const int64_t i0 = I * kTile + r, j0 = J * kTile + c;
        const int64_t i = i0 > j0 ? i0 : j0, j = i0 > j0 ? j0 : i0;  // A's lower triangle
        const double v = (i < n && j < n) ? A[i + j * n] : (i == j ? 1.0 : 0.0);
        out[e] = v;
        P[r][c] = v;
    }
    if (blockIdx.x != 0) return;
    __syncthreads();
    pivot_to(P, T, Q, info, clear);
}

// acc[c] (16 x 16 block: rows 16 w .. 16 w + 15, columns 16 c ..) = sum over
// k = 0..63 of A(r, k) B(k, c), in k order.  MFMA 16x16x4 FP64 operand
// layout: lane l holds A(l % 16, l / 16) and B(l / 16, l % 16); the result
// register q of lane l is D(4 q + l / 16, l % 16) (rows interleave across the
// lane groups).
__device__ __forceinline__ void tile_product(int w, const Tile& As, const Tile& Bs, tad_v4d acc[4])
{
    const int lane = threadIdx.x & 63;
    const int r = lane % 16, kk = lane / 16;
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[c] = tad_v4d{ 0.0, 0.0, 0.0, 0.0 };
#pragma unroll 4
    for (int k0 = 0; k0 < kTile; k0 += 4)
    {
        const double av = As[16 * w + r][k0 + kk];
#pragma unroll
        for (int c = 0; c < 4; ++c)
        {
            const double bv = Bs[16 * c + r][k0 + kk];
            acc[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, bv, acc[c], 0, 0, 0);
        }
    }
}

// X[o][k] = M_KI(k, o) from the stored lower tiles, in two halves so that the
// loads can be in flight while the LDS tile is still read.
__device__ __forceinline__ void fetch_panel(const double* __restrict__ S, int64_t K, int64_t I, double v[16])
{
    const double* __restrict__ src = S + (K >= I ? tile_at(K, I) : tile_at(I, K));
#pragma unroll
    for (int p = 0; p < 16; ++p) v[p] = src[threadIdx.x + 256 * p];
}

__device__ __forceinline__ void put_panel(const double v[16], bool low, Tile& X)
{
#pragma unroll
    for (int p = 0; p < 16; ++p)
    {
        const int e = threadIdx.x + 256 * p;
        const int a = e % kTile, b = e / kTile;
        if (low) X[b][a] = v[p];
        else X[a][b] = v[p];
    }
}

// Strips of pivot step: for tile column J the rows J .. nt - 1 in strips of L.
__host__ __device__ __forceinline__ int64_t strips_of(int64_t nt, int64_t J, int64_t L) { return (nt - J + L - 1) / L; }

// Pivot step K: S (lower tiles) -> So, Q = M_KK^-1 given; workgroup 0 updates
// the next pivot block (K + 1, K + 1) and writes its inverse to Qo, the
// others take one strip of at most L tiles of one tile column each: W_J once,
// then one product per tile.
__global__ __launch_bounds__(256, 2) void k_sweep_step(int64_t nt, int64_t K, int64_t L, const double* __restrict__ S,
                                                    const double* __restrict__ Q, double* __restrict__ So,
                                                    double* __restrict__ Qo, int* __restrict__ info)
{
    __shared__ Tile X, Y;
    const int t = threadIdx.x, w = t >> 6, lane = t & 63;
    const int g = lane / 16, j = lane % 16;
    const bool next = K + 1 < nt;
    int64_t J, I0, I1;
    const bool pivot = next && blockIdx.x == 0;
    if (pivot)
    {
        J = K + 1;
        I0 = J;
        I1 = J + 1;
    }
    else
    {
        int64_t b = (int64_t)blockIdx.x - (next ? 1 : 0);
        J = 0;
        for (int64_t ns = strips_of(nt, 0, L); b >= ns; ns = strips_of(nt, J, L))
        {
            b -= ns;
            ++J;
        }
        I0 = J + b * L;
        I1 = min(nt, I0 + L);
    }
    double v[16];
#pragma unroll
    for (int p = 0; p < 16; ++p) v[p] = Q[t + 256 * p];
    put_panel(v, true, X);  // symmetric
    tad_v4d acc[4];
    if (J == K)  // pivot column: -Q and W_I^T
    {
        for (int64_t I = I0; I < I1; ++I)
        {
            double* __restrict__ out = So + tile_at(I, K);
            if (I == K)
            {
#pragma unroll
                for (int p = 0; p < 16; ++p) out[t + 256 * p] = -Q[t + 256 * p];
                continue;
            }
            fetch_panel(S, K, I, v);
            put_panel(v, K >= I, Y);
            __syncthreads();
            tile_product(w, X, Y, acc);  // (column of tile (I, K), row)
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int q = 0; q < 4; ++q) out[(16 * c + j) + kTile * (16 * w + 4 * q + g)] = acc[c][q];
            __syncthreads();
        }
        return;
    }
    fetch_panel(S, K, J, v);
    put_panel(v, K >= J, Y);
    fetch_panel(S, K, I0, v);  // C_I of the first tile, in flight during W_J (for I0 = K: not used)
    __syncthreads();
    tile_product(w, Y, X, acc);  // W_J^T: (column of J, row of K)
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int q = 0; q < 4; ++q) Y[16 * w + 4 * q + g][16 * c + j] = acc[c][q];
    __syncthreads();
    for (int64_t I = I0; I < I1; ++I)
    {
        if (I == K)  // pivot row: W_J
        {
            double* __restrict__ out = So + tile_at(K, J);
#pragma unroll
            for (int p = 0; p < 16; ++p)
            {
                const int e = t + 256 * p;
                out[e] = Y[e / kTile][e % kTile];
            }
            continue;
        }
        if (!pivot && I == K + 1 && J == K + 1) continue;  // workgroup 0
        const double* __restrict__ in = S + tile_at(I, J);
        double* __restrict__ out = So + tile_at(I, J);
        double old[16];
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int q = 0; q < 4; ++q) old[4 * c + q] = in[(16 * c + j) + kTile * (16 * w + 4 * q + g)];
        if (I > I0) fetch_panel(S, K, I, v);
        put_panel(v, K >= I, X);
        __syncthreads();
        tile_product(w, Y, X, acc);  // (column of tile (I, J), row)
        __syncthreads();
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int q = 0; q < 4; ++q)
            {
                const int r = 16 * c + j, cc = 16 * w + 4 * q + g;
                const double v = old[4 * c + q] - acc[c][q];
                if (I > J)
                    out[r + kTile * cc] = v;
                else if (r >= cc)  // a diagonal tile mirrors its lower half
                {
                    out[r + kTile * cc] = v;
                    out[cc + kTile * r] = v;
                    if (pivot)
                    {
                        X[r][cc] = v;
                        X[cc][r] = v;
                    }
                }
            }
    }
    if (pivot)
    {
        __syncthreads();
        pivot_to(X, Y, Qo, info, false);
    }
}

// A = -S on the leading n x n part, both triangles (the sweeps leave -A^-1).
__global__ __launch_bounds__(256) void k_sweep_store(int64_t n, const double* __restrict__ S, double* __restrict__ A)
{
    __shared__ Tile P;
    int64_t I = 0, J = blockIdx.x;
    while (J > I) J -= ++I;
    const double* __restrict__ in = S + tile_at(I, J);
#pragma unroll
    for (int p = 0; p < 16; ++p)
    {
        const int e = threadIdx.x + 256 * p;
        const int r = e % kTile, c = e / kTile;
        const int64_t i = I * kTile + r, jj = J * kTile + c;
        const double v = -in[e];
        P[r][c] = v;
        // a diagonal tile's lower half is written from here, its upper half below
        if (i < n && jj < n && i >= jj) A[i + jj * n] = v;
    }
    __syncthreads();
#pragma unroll
    for (int p = 0; p < 16; ++p)
    {
        const int e = threadIdx.x + 256 * p;
        const int c = e % kTile, r = e / kTile;
        const int64_t i = I * kTile + r, jj = J * kTile + c;
        if (i < n && jj < n && i > jj) A[jj + i * n] = P[r][c];
    }
}

} // namespace

int64_t spd_inverse_work(int64_t n)
{
    const int64_t nt = (n + kTile - 1) / kTile;
    return 2 * (nt * (nt + 1) / 2) * kTT + 2 * kTT;
}

hipError_t launch_spd_inverse(int64_t n, double* A, double* work, int* info, hipStream_t s, bool cleared)
{
    if (n <= 0) return hipSuccess;
    const int64_t nt = (n + kTile - 1) / kTile;
    const int64_t tiles = nt * (nt + 1) / 2;
    double* S[2] = { work, work + tiles * kTT };
    double* Q[2] = { work + 2 * tiles * kTT, work + (2 * tiles + 1) * kTT };
    // Strip length: one tile per workgroup while the chip (two workgroups per
    // CU by LDS) holds them all, longer strips beyond, where W_J's product
    // per strip is what the extra workgroups would cost.
    const int64_t L = std::min<int64_t>(4, std::max<int64_t>(1, tiles / 512 + 1));
    int64_t strips = 0;
    for (int64_t J = 0; J < nt; ++J) strips += strips_of(nt, J, L);
    k_sweep_load<<<(unsigned)tiles, 256, 0, s>>>(n, A, S[0], Q[0], info, !cleared);
    for (int64_t K = 0; K < nt; ++K)
        k_sweep_step<<<(unsigned)(strips + (K + 1 < nt ? 1 : 0)), 256, 0, s>>>(nt, K, L, S[K & 1], Q[K & 1],
                                                                               S[(K + 1) & 1], Q[(K + 1) & 1], info);
    k_sweep_store<<<(unsigned)tiles, 256, 0, s>>>(n, S[nt & 1], A);
    return hipGetLastError();
}

} // namespace tad
