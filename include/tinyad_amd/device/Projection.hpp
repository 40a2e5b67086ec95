// In-register symmetric eigensolve and positive-definite projection for small
// packed symmetric matrices (n <= 12), one matrix per lane.
//
// Semantics follow include/TinyAD/Utils/HessianProjection.hh:48-101:
//   eps >= 0: eigenvalues below eps are raised to eps;
//   eps <  0: negative eigenvalues are replaced by their absolute value;
//   if no eigenvalue changed, the matrix is returned unchanged.
// The reference first tries a positive-diagonal-dominance early out
// (HessianProjection.hh:23-42) and otherwise runs Eigen's dense
// SelfAdjointEigenSolver.  Here the early out is a Cholesky factorization of
// A - max(eps, 0) I: it succeeds exactly when every eigenvalue exceeds the
// clamp level, which covers every matrix the diagonal-dominance test accepts
// (Gershgorin) and more, and in that case the reference also returns the
// matrix unchanged.  Otherwise a Householder tridiagonalization and implicit
// QL iteration (the two stages SelfAdjointEigenSolver also uses) give the
// spectrum, and the clamped spectrum is re-assembled.
#pragma once

#include <hip/hip_runtime.h>
#include "Dual.hpp"

namespace tad {

// True when A - shift I is positive definite (Cholesky succeeds).
template <int n, class T>
__device__ __forceinline__ bool cholesky_pd(const T* A, T shift)
{
    T L[Sym<n>::n];
    bool ok = true;
#pragma unroll
    for (int j = 0; j < n; ++j)
    {
        T djj = A[Sym<n>::idx(j, j)] - shift;
#pragma unroll
        for (int k = 0; k < j; ++k) djj -= L[Sym<n>::idx(k, j)] * L[Sym<n>::idx(k, j)];
        ok = ok && (djj > T(0));
        const T ljj = sqrt(djj > T(0) ? djj : T(1));
        const T il = T(1) / ljj;
        L[Sym<n>::idx(j, j)] = ljj;
#pragma unroll
        for (int i = j + 1; i < n; ++i)
        {
            T s = A[Sym<n>::idx(j, i)];
#pragma unroll
            for (int k = 0; k < j; ++k) s -= L[Sym<n>::idx(k, i)] * L[Sym<n>::idx(k, j)];
            L[Sym<n>::idx(j, i)] = s * il;  // L stored transposed: entry (j, i) = L_ij
        }
    }
    return ok;
}

// 1/sqrt(x), x > 0 finite: the hardware approximation refined by Newton
// steps (two in FP64: ~2^-22 -> below 1 ulp; one in FP32)
__device__ __forceinline__ double ql_rsqrt(double x)
{
    double y = __builtin_amdgcn_rsq(x);
    const double hx = 0.5 * x;
    y = y * (1.5 - hx * y * y);
    y = y * (1.5 - hx * y * y);
    return y;
}
__device__ __forceinline__ float ql_rsqrt(float x)
{
    float y = __builtin_amdgcn_rsqf(x);
    y = y * (1.5f - 0.5f * x * y * y);
    return y;
}

template <class T> struct QlTraits;
template <> struct QlTraits<double>
{
    static constexpr double eps = 2.220446049250313e-16;  // 2^-52
    static constexpr int max_iters = 30;
};
template <> struct QlTraits<float>
{
    static constexpr float eps = 1.1920929e-07f;  // 2^-23
    static constexpr int max_iters = 30;
};

// Symmetric eigensolve by Householder reduction to tridiagonal form followed
// by the implicit QL iteration with a Wilkinson-type shift (Bowdler, Martin,
// Reinsch and Wilkinson, Numer. Math. 11 (1968) 293-306, the method of EISPACK
// tql2; Eigen's SelfAdjointEigenSolver follows the same two stages).
// A (packed, n x n) is consumed; on exit Z (row-major) holds orthonormal
// eigenvectors as columns and lam the eigenvalues.  Every register index is a
// compile-time constant: data-dependent loop bounds of the QL sweep are
// applied as per-step activity masks, so nothing goes to scratch.
// Entry of e holding coupling i of the reversed tridiagonal matrix (e[n-1]
// is the zero sentinel).
__host__ __device__ constexpr int ql_rev_e(int n, int i) { return i <= n - 2 ? n - 2 - i : n - 1; }

// InMemory: the loops over Z's rows (over its columns where Q is accumulated)
// stay loops, which puts Z into scratch memory: for a rare path, whose
// registers then do not count for the kernel around it.
template <int n, class T, bool InMemory = false>
__device__ __forceinline__ void tridiag_ql_eigen(T* A, T* Z, T* lam)
{
    constexpr int kRows = InMemory ? 1 : n;
    T e[n];
    T tau[n > 2 ? n - 2 : 1];
    // 1. Householder: column k below the diagonal -> (e_k, 0, ..., 0); the
    //    reflector vector v overwrites that column (v_0 in row k + 1).
#pragma unroll
    for (int k = 0; k + 2 < n; ++k)
    {
        const int L = n - k - 1;
        T sigma = T(0);
#pragma unroll
        for (int i = 1; i < L; ++i) sigma += A[Sym<n>::idx(k, k + 1 + i)] * A[Sym<n>::idx(k, k + 1 + i)];
        const T x0 = A[Sym<n>::idx(k, k + 1)];
        const bool has = sigma > T(0);
        const T mu = sqrt(x0 * x0 + sigma);
        const T alpha = x0 > T(0) ? -mu : mu;
        const T v0 = x0 - alpha;
        const T vtv = v0 * v0 + sigma;
        const T tk = has ? T(2) / (has ? vtv : T(1)) : T(0);
        e[k] = has ? alpha : x0;
        tau[k] = tk;
        A[Sym<n>::idx(k, k + 1)] = v0;
        // p = tau B v, w = p - (tau/2)(v.p) v, B -= v w^T + w v^T
        T pv[n], vv[n];
#pragma unroll
        for (int i = 0; i < L; ++i) vv[i] = A[Sym<n>::idx(k, k + 1 + i)];
        T vp = T(0);
#pragma unroll
        for (int i = 0; i < L; ++i)
        {
            T acc = T(0);
#pragma unroll
            for (int j = 0; j < L; ++j) acc += A[Sym<n>::at(k + 1 + i, k + 1 + j)] * vv[j];
            pv[i] = tk * acc;
            vp += vv[i] * pv[i];
        }
        const T K = T(0.5) * tk * vp;
#pragma unroll
        for (int i = 0; i < L; ++i) pv[i] -= K * vv[i];
#pragma unroll
        for (int i = 0; i < L; ++i)
#pragma unroll
            for (int j = i; j < L; ++j) A[Sym<n>::idx(k + 1 + i, k + 1 + j)] -= vv[i] * pv[j] + pv[i] * vv[j];
    }
#pragma unroll
    for (int i = 0; i < n; ++i) lam[i] = A[Sym<n>::idx(i, i)];
    if (n >= 2) e[n - 2] = A[Sym<n>::idx(n - 2, n - 1)];
    e[n - 1] = T(0);
    // 2. Z = P_0 P_1 ... P_{n-3}, accumulated backwards (P_k acts on rows and
    //    columns k+1..n-1, where the partial product is non-trivial).
#pragma unroll kRows
    for (int i = 0; i < n; ++i)
#pragma unroll
        for (int j = 0; j < n; ++j) Z[i * n + j] = (i == j) ? T(1) : T(0);
#pragma unroll
    for (int k = n - 3; k >= 0; --k)
    {
        const int L = n - k - 1;
#pragma unroll kRows
        for (int j = k + 1; j < n; ++j)
        {
            T s = T(0);
#pragma unroll
            for (int i = 0; i < L; ++i) s += A[Sym<n>::idx(k, k + 1 + i)] * Z[(k + 1 + i) * n + j];
            s *= tau[k];
#pragma unroll
            for (int i = 0; i < L; ++i) Z[(k + 1 + i) * n + j] -= s * A[Sym<n>::idx(k, k + 1 + i)];
        }
    }
    // 3. implicit QL on the tridiagonal matrix in reverse order, J T J with
    //    J the reversal (lr[i] = lam[n-1-i], er[i] couples lr[i] and lr[i+1]):
    //    the reduction above runs from the first row down, and deflating the
    //    reversed matrix from the top needs fewer sweeps (element Hessians of
    //    the 60^3 twisted cube: 16.6 instead of 19.0 QL iterations per 9 x 9
    //    matrix, 18 instead of 22 for the slowest lane of a wave).  Column i
    //    of the reversed problem is column n-1-i of Z.
    // (index maps only: lr(i) is lam[n-1-i], er(i) is e[n-2-i] and er(n-1)
    // the zero sentinel e[n-1], so the sweep works on the same registers)
    const T eps = QlTraits<T>::eps;
#pragma unroll
    for (int l = 0; l + 1 < n; ++l)
    {
        for (int it = 0; it < QlTraits<T>::max_iters; ++it)
        {
            int m = n - 1;
#pragma unroll
            for (int j = n - 2; j >= l; --j)
                if (fabs(e[ql_rev_e(n, j)]) <= eps * (fabs(lam[n - 1 - (j)]) + fabs(lam[n - 1 - (j + 1)]))) m = j;
            if (m == l) break;
            T dm = lam[n - 1 - (n - 1)];
#pragma unroll
            for (int j = l; j + 1 < n; ++j)
                if (j == m) dm = lam[n - 1 - (j)];
            T g = (lam[n - 1 - (l + 1)] - lam[n - 1 - (l)]) / (T(2) * e[ql_rev_e(n, l)]);
            T r = sqrt(g * g + T(1));
            g = dm - lam[n - 1 - (l)] + e[ql_rev_e(n, l)] / (g + (g >= T(0) ? r : -r));
            T s = T(1), c = T(1), p = T(0);
            bool alive = true;  // false once a rotation underflowed (r == 0)
#pragma unroll
            for (int i = n - 2; i >= l; --i)
            {
                if (alive && i < m)
                {
                    const T f = s * e[ql_rev_e(n, i)];
                    const T b = c * e[ql_rev_e(n, i)];
                    // r = |(f, g)| and 1/r from one refined reciprocal square root
                    const T qq = f * f + g * g;
                    const T ir = qq > T(0) ? ql_rsqrt(qq) : T(0);
                    r = qq * ir;
                    e[ql_rev_e(n, i + 1)] = r;
                    if (r == T(0))
                    {
                        lam[n - 1 - (i + 1)] -= p;
#pragma unroll
                        for (int j = l; j + 1 < n; ++j)
                            if (j == m) e[ql_rev_e(n, j)] = T(0);
                        alive = false;
                    }
                    else
                    {
                        s = f * ir;
                        c = g * ir;
                        g = lam[n - 1 - (i + 1)] - p;
                        r = (lam[n - 1 - (i)] - g) * s + T(2) * c * b;
                        p = s * r;
                        lam[n - 1 - (i + 1)] = g + p;
                        g = c * r - b;
#pragma unroll kRows
                        for (int k = 0; k < n; ++k)
                        {
                            const T zi = Z[k * n + (n - 1 - i)], zi1 = Z[k * n + (n - 2 - i)];
                            Z[k * n + (n - 2 - i)] = s * zi + c * zi1;
                            Z[k * n + (n - 1 - i)] = c * zi - s * zi1;
                        }
                    }
                }
            }
            if (alive)
            {
                lam[n - 1 - (l)] -= p;
                e[ql_rev_e(n, l)] = g;
#pragma unroll
                for (int j = l; j + 1 < n; ++j)
                    if (j == m) e[ql_rev_e(n, j)] = T(0);
            }
        }
    }
}

// 1/x, x normal: the hardware approximation refined by two Newton steps
__device__ __forceinline__ double refined_rcp(double x)
{
    double y = __builtin_amdgcn_rcp(x);
    y = fma(fma(-x, y, 1.0), y, y);
    y = fma(fma(-x, y, 1.0), y, y);
    return y;
}

// |x| < 2^K, from the exponent (false for NaN): its constant stands in the
// instruction, where a double's would be held in registers through the
// persistent kernels' loop.
template <int K>
__device__ __forceinline__ bool under(double x)
{
    return ((uint32_t)(__builtin_bit_cast(uint64_t, x) >> 32) & 0x7fffffffu) < (uint32_t)(1023 + K) << 20;
}

// True when A - shift I is positive definite, from the pivots of its L D L^T
// factorization (no square roots, one reciprocal per column).
template <int n>
__device__ __forceinline__ bool ldl_pd(const double* A, double shift)
{
    double L[Sym<n>::n], D[n];
    bool ok = true;
#pragma unroll
    for (int j = 0; j < n; ++j)
    {
        double t[n];
        double dj = A[Sym<n>::idx(j, j)] - shift;
#pragma unroll
        for (int k = 0; k < j; ++k)
        {
            t[k] = L[Sym<n>::idx(k, j)] * D[k];
            dj -= t[k] * L[Sym<n>::idx(k, j)];
        }
        ok = ok && (dj > 0.0);
        D[j] = dj;
        const double ij = refined_rcp(dj > 0.0 ? dj : 1.0);
#pragma unroll
        for (int i = j + 1; i < n; ++i)
        {
            double v = A[Sym<n>::idx(j, i)];
#pragma unroll
            for (int k = 0; k < j; ++k) v -= L[Sym<n>::idx(k, i)] * t[k];
            L[Sym<n>::idx(j, i)] = v * ij;
        }
    }
    return ok;
}

// Eigenvectors project_few computes at most.  An isotropic energy of a tet has
// up to three eigenvalues below zero, one per pair of singular values; four are
// the smaller side of any level among the nine of a tet.
constexpr int kMaxClamped = 4;
// On the scaled tridiagonal (norm 1): the rounding of a root; the shift off
// roots that cannot be told apart for their vectors; the residual at which a
// vector is final, the largest accepted, and the passes it gets.
constexpr double kRootRounding = 1e-15, kSharedShift = 1e-13, kResidual = 2e-15, kResidualMax = 4e-15;
constexpr int kVectorPasses = 5;
// Distances from a known root at which the search for the next one sets out:
// the largest with no root between.  (Closer than a thousandth of the distance
// to the next root, the rounding of the known one would drown it.)
constexpr int kRootGaps = 6;
__device__ __forceinline__ double root_gap(int i)
{
    return ldexp(1.0, i == 0 ? -7 : i == 1 ? -17 : i == 2 ? -27 : i == 3 ? -37 : i == 4 ? -43 : -47);
}

// A pivot, kept from zero by less than the rounding of a matrix of norm 1 (NaN
// becomes a number).
__device__ __forceinline__ double off_zero(double x) { return copysign(fmax(fabs(x), 0x1p-56), x); }

// Number of eigenvalues of the tridiagonal (d, e2 = squared couplings) below
// x (negative pivots of T - x I), and the logarithmic derivative of
// det(T - x I) (s1) and its derivative (s2).  The pivots come from both ends
// at once and meet in the middle: two independent chains of n / 2 instead of
// one of n.
template <int n>
__device__ __forceinline__ int tridiag_count(const double* d, const double* e2, double x, double& s1, double& s2)
{
    constexpr int mid = n / 2;
    int count = 0;
    // per chain: e2 / last pivot, the pivot's first and second log-derivative parts
    double w[2] = {}, t[2] = {}, u[2] = {}, a1[2] = {}, a2[2] = {};
#pragma unroll
    for (int s = 0; s < mid; ++s)
#pragma unroll
        for (int c = 0; c < 2; ++c)
        {
            const int i = c == 0 ? s : n - 1 - s;
            if (c == 1 && i <= mid) continue;
            double q = (d[i] - x) - w[c];
            q = off_zero(q);
            const double r = refined_rcp(q);
            count += q < 0.0 ? 1 : 0;
            const double q2 = w[c] * (u[c] - 2.0 * t[c] * t[c]);
            t[c] = (w[c] * t[c] - 1.0) * r;
            u[c] = q2 * r;
            a1[c] += t[c];
            a2[c] += u[c] - t[c] * t[c];
            w[c] = e2[c == 0 ? i : i - 1] * r;
        }
    double q = ((d[mid] - x) - w[0]) - w[1];
    q = off_zero(q);
    const double r = refined_rcp(q);
    count += q < 0.0 ? 1 : 0;
    const double q2 = w[0] * (u[0] - 2.0 * t[0] * t[0]) + w[1] * (u[1] - 2.0 * t[1] * t[1]);
    const double tm = (w[0] * t[0] + (w[1] * t[1] - 1.0)) * r;
    s1 = a1[0] + a1[1] + tm;
    s2 = a2[0] + a2[1] + (q2 * r - tm * tm);
    return count;
}

// y <- (T - shift I)^-1 y for the tridiagonal (d, e) by Givens rotations: no
// element growth at any shift (a zero pivot counts as 1e-30).
template <int n>
__device__ __forceinline__ void tridiag_solve(const double* d, const double* e, double shift, double* y)
{
    double r0[n], r1[n], r2[n];  // rows of R: reciprocal diagonal, the two superdiagonals
    double a = d[0] - shift, b = e[0];
#pragma unroll
    for (int i = 0; i + 1 < n; ++i)
    {
        const double x = e[i], an = d[i + 1] - shift, bn = i + 2 < n ? e[i + 1] : 0.0;
        const double w = a * a + x * x;
        const bool zero = under<-200>(w);
        const double ih = ql_rsqrt(zero ? 1.0 : w);
        const double c = zero ? 1.0 : a * ih, s = zero ? 0.0 : x * ih;
        r0[i] = zero ? 1e30 : ih;
        r1[i] = c * b + s * an;
        r2[i] = s * bn;
        a = c * an - s * b;
        b = c * bn;
        const double t = c * y[i] + s * y[i + 1];
        y[i + 1] = c * y[i + 1] - s * y[i];
        y[i] = t;
    }
    r0[n - 1] = refined_rcp(under<-100>(a) ? 1e-30 : a);
#pragma unroll
    for (int i = n - 1; i >= 0; --i)
    {
        if (i + 1 < n) y[i] -= r1[i] * y[i + 1];
        if (i + 2 < n) y[i] -= r2[i] * y[i + 2];
        y[i] *= r0[i];
    }
}

// v / |v|, without overflow for |v| up to 1e300
template <int n>
__device__ __forceinline__ void normalize(double* v)
{
    double top = 0.0, vv = 0.0;
#pragma unroll
    for (int i = 0; i < n; ++i) top = fmax(top, fabs(v[i]));
    const double it = refined_rcp(top);
#pragma unroll
    for (int i = 0; i < n; ++i)
    {
        v[i] *= it;
        vv += v[i] * v[i];
    }
    const double iv = ql_rsqrt(vv);
#pragma unroll
    for (int i = 0; i < n; ++i) v[i] *= iv;
}

// Place of reflector k (n - 1 - k values) among the stored ones, and their
// number.
__host__ __device__ constexpr int reflector_at(int n, int k) { return k * (n - 1) - k * (k - 1) / 2; }
__host__ __device__ constexpr int reflector_values(int n) { return reflector_at(n, n - 2); }

// Projects packed symmetric A in place from the eigenvectors on the smaller
// side of the clamp level only:
//   P(A) = A + sum_j (clamped_j - lam_j) v_j v_j^T
// over the eigenvalues below it or, if more than kMaxClamped are,
//   P(A) = eps I + sum_j (lam_j - eps) v_j v_j^T    (absolute values:
//   P(A) = -A + sum_j 2 lam_j v_j v_j^T)
// over those above it, computed as the ones below it of -A.  Returns false,
// with A restored up to rounding, when a vector misses its residual; the
// caller then projects A by the full eigensolve.
//   1. Householder reduction to the tridiagonal T, scaled by a power of two
//      to norm 1, the reflectors going to `store` (in registers they do not
//      fit beside the rest); the number m of eigenvalues below the level from
//      the pivot signs (T and the level negated if those are the most).  Roots
//      within rounding of the level are not clamped (they would move by
//      rounding).
//   2. Their values from right to left by Laguerre's iteration (cubic, and
//      monotone towards the neighbouring root as all roots are real), each
//      started next to the previous root, which is divided out.  k roots that
//      look like one are approached as one k-fold root; roots within 1e-14 of
//      each other share one value.
//   3. Their vectors: a twisted factorization of T - lam I (Fernando, SIAM J.
//      Matrix Anal. Appl. 18 (1997) 1013-1034) at the index with the smallest
//      twist pivot, then inverse iteration until T z - rho z is at rounding
//      level, with two Gram-Schmidt passes against the earlier vectors.  m
//      orthonormal vectors with such residuals and m Rayleigh quotients below
//      the level are all there is below it, however close the roots are:
//      which vectors of close roots they are does not matter to P(A).
//   4. T (or eps I, or -T) + sum c w w^T, then the reflectors from both sides.
// On the CPU, 6,000 element matrices (10^3 cube) per state, eps 1e-9, 0.05, 0
// and absolute values, against 80-bit arithmetic, relative to |A|: at rest, noise
// of 1e-12 .. 0.1 mesh widths, smooth displacements, compressed and flattened
// by 1e-9 .. 0.2, twisted by 0.01 .. 60 degrees 4.1e-15 at most (full
// eigensolve 4.2e-15), at most 0.18 % of the elements given to the full
// eigensolve (0.5 % for levels in the middle of the spectrum).  Noise of 1e-13
// and 1e-14 mesh widths, whose roots are hardly above rounding: 0.4 %, and 3
// and 23 % for eps <= 0, where the level lies among them; error 1.5e-14 at most.
// 7 to 18 evaluations of step 2 per wave at eps 1e-9, where the full QL
// iteration takes 27 sweeps, 31 with the level among the eigenvalues.
// Evaluation of 1,296,000 tets: twisted by 30 and 54 degrees 0.82 and 0.81 ms,
// at rest 0.74, noise of 1e-9 and 1e-4 mesh widths 0.88 and 0.81, compressed by
// 1e-4 0.77 (with the full eigensolve, and a tail of its own launches, 1.35,
// 1.36, 1.20, 1.16, 1.26, 1.15); eps 1e-4 .. 1e-2 0.79 .. 0.90, eps above every
// eigenvalue 0.63 (full 1.19 .. 1.38; where only the side below the level is
// computed and the rest left to the full eigensolve here, 6.7 .. 8.1).
template <int n>
__device__ __forceinline__ bool project_few(double* A, double eps, double* store)
{
    static_assert(n <= 2 * kMaxClamped + 1, "one side of the level has at most kMaxClamped eigenvalues");
    double amax = 0.0;
#pragma unroll
    for (int q = 0; q < Sym<n>::n; ++q) amax = fmax(amax, fabs(A[q]));
    if (!(amax > 1e-100 && amax < 1e100)) return false;
    double d[n], e[n];
    // 1. as in tridiag_ql_eigen, with refined reciprocals; a reflector that is
    //    the identity is stored as 0
#pragma unroll
    for (int k = 0; k + 2 < n; ++k)
    {
        const int L = n - k - 1;
        double sigma = 0.0;
#pragma unroll
        for (int i = 1; i < L; ++i) sigma += A[Sym<n>::idx(k, k + 1 + i)] * A[Sym<n>::idx(k, k + 1 + i)];
        const double x0 = A[Sym<n>::idx(k, k + 1)];
        const double ss = x0 * x0 + sigma;
        const bool has = sigma > 0.0 && ss > 1e-290;
        const double mu = has ? ss * ql_rsqrt(ss) : 0.0;
        const double v0 = x0 > 0.0 ? x0 + mu : x0 - mu;
        const double tk = has ? 2.0 * refined_rcp(v0 * v0 + sigma) : 0.0;
        e[k] = has ? (x0 > 0.0 ? -mu : mu) : x0;
        A[Sym<n>::idx(k, k + 1)] = v0;
#pragma unroll
        for (int i = 0; i < L; ++i) store[(reflector_at(n, k) + i) * 64] = has ? A[Sym<n>::idx(k, k + 1 + i)] : 0.0;
        double pv[n], vp = 0.0;
#pragma unroll
        for (int i = 0; i < L; ++i)
        {
            double acc = 0.0;
#pragma unroll
            for (int j = 0; j < L; ++j) acc += A[Sym<n>::at(k + 1 + i, k + 1 + j)] * A[Sym<n>::idx(k, k + 1 + j)];
            pv[i] = tk * acc;
            vp += A[Sym<n>::idx(k, k + 1 + i)] * pv[i];
        }
        const double K = 0.5 * tk * vp;
#pragma unroll
        for (int i = 0; i < L; ++i) pv[i] -= K * A[Sym<n>::idx(k, k + 1 + i)];
#pragma unroll
        for (int i = 0; i < L; ++i)
#pragma unroll
            for (int j = i; j < L; ++j)
                A[Sym<n>::idx(k + 1 + i, k + 1 + j)] -=
                    A[Sym<n>::idx(k, k + 1 + i)] * pv[j] + pv[i] * A[Sym<n>::idx(k, k + 1 + j)];
    }
    e[n - 2] = A[Sym<n>::idx(n - 2, n - 1)];
    e[n - 1] = 0.0;
    double norm = 0.0;
#pragma unroll
    for (int i = 0; i < n; ++i)
    {
        d[i] = A[Sym<n>::idx(i, i)];
        norm = fmax(norm, fabs(d[i]) + fabs(e[i]) + (i > 0 ? fabs(e[i - 1]) : 0.0));
    }
    double nan_sum = 0.0;
#pragma unroll
    for (int i = 0; i < n; ++i) nan_sum += (d[i] + e[i]) * 0.0;
    if (!(nan_sum == 0.0)) return false;
    int ex = 0;
    (void)frexp(norm, &ex);
    bool ok = true;
    double e2[n];
#pragma unroll
    for (int i = 0; i < n; ++i)
    {
        d[i] = ldexp(d[i], -ex);
        e[i] = ldexp(e[i], -ex);
        e2[i] = e[i] * e[i];
    }
    double level = ldexp(eps > 0.0 ? eps : 0.0, -ex);
    // 2. roots r[0] >= r[1] >= ... below `start`
    double r[kMaxClamped] = {};
    double start = level - kRootRounding;
    int m = 0, found = 0;
    bool flip = false;  // more eigenvalues clamped than not: the others, of -T
    {
        double x = start, g, h;
        int below = tridiag_count<n>(d, e2, x, g, h);
        h = -h;
        if (below > kMaxClamped)
        {
            flip = true;
            below = n - below;
            g = -g;
            level = -level;
            start = x = -start;
#pragma unroll
            for (int i = 0; i < n; ++i)
            {
                d[i] = -d[i];
                e[i] = -e[i];
            }
        }
        double from = x;  // the last root (or the level)
        int gap = -1;     // >= 0: x lies root_gap(gap) below `from`
        bool fresh = true, known = true;  // m to be taken from `below`; evaluated at x already
        bool run = below > 0;
#pragma unroll 1
        for (int it = 0; run && it < 64; ++it)
        {
            if (!known)
            {
                below = tridiag_count<n>(d, e2, x, g, h);
                h = -h;
            }
            known = false;
            bool away = false;
            if (fresh)
            {
                fresh = false;
                m = below;
                run = m > 0;
                // roots right above the level: set out away from them
                away = g < 0.0 && !under<10>(g);
                if (away)
                {
                    gap = 0;
                    x = from - root_gap(0);
                }
            }
            const int inside = m - found - below;  // roots not found yet that are not below x
            int take = 0;
            double root = from;
            if (gap >= 0 && inside > 0)
            {
                // between the last root and x: closer to it, or not to be told apart from it
                if (gap + 1 < kRootGaps) x = from - root_gap(++gap);
                else take = inside;
            }
            else if (!away)
            {
                gap = -1;
#pragma unroll
                for (int j = 0; j + 1 < kMaxClamped; ++j)
                    if (j < found)
                    {
                        const double q = refined_rcp(x - r[j]);
                        g -= q;
                        h -= q * q;
                    }
                const double deg = (double)(n - found), gg = g * g;
                const double spread = deg * h - gg;  // 0 for one deg-fold root
                const double disc = (deg - 1.0) * spread;
                const double sq = disc > 0.0 ? disc * ql_rsqrt(disc) : 0.0;
                // k equal roots have g = k / (x - root), h = k / (x - root)^2
                // (g < 0: the near ones lie above x)
                const double like = gg * __builtin_amdgcn_rcp(h);
                const double fold = fmin(fmax(rint(like), 1.0), (double)(m - found));
                const double dev = fabs(like - fold);
                const bool past = inside > 0;  // x is below the next root: towards it
                const bool alike = (past ? g < 0.0 : g > 0.0) && dev < 0.01 * fold;
                double step = deg * refined_rcp(past ? g - sq : g + sq);
                // (the wrong way: rounding of the roots divided out)
                const bool lost = !(past ? step < 0.0 : step > 0.0);
                if (lost) step = past ? 0.5 * (x - from) : fmax(from - x, root_gap(1));
                else if (alike && fold == 1.0)
                    take = under<-53>(step * dev * dev) ? 1 : 0;  // (the error of root: about step dev^2)
                else if (alike)
                {
                    const double f = (deg * refined_rcp(fold) - 1.0) * spread;
                    const double sf = f > 0.0 ? f * ql_rsqrt(f) : 0.0;
                    step = deg * refined_rcp(past ? g - sf : g + sf);
                    take = under<-43>(step) ? (int)fold : 0;
                }
                if (!lost && under<-51>(step) && (past || g > 0.0)) take = max(take, 1);
                root = x - step;
                if (inside > 1)
                {
                    // beyond all but one of them, or they share a value
                    take = under<-47>(step) ? inside : 0;
                    step *= 2.0;
                }
                else if (take == 0 && alike && fold > 1.0)
                {
                    // short of the first of them (their spread is about 2 sqrt(dev / k) of the distance)
                    const double q = fmax(dev, 1e-12);
                    step *= 1.0 - 2.0 * q * ql_rsqrt(q);
                }
                x -= step;
            }
            if (take > 0)
            {
                gap = 1;
                from = root;
                if (found == 0 && !(root < start - 2.0 * kRootRounding))
                {
                    // at the level up to rounding: those below it are clamped
                    run = root > level - 4.0 * kRootRounding;
                    start = from = root - 2.0 * kRootRounding;
                    fresh = true;
                    gap = -1;
                    x = from;
                }
                else
                {
#pragma unroll
                    for (int j = 0; j < kMaxClamped; ++j)
                        if (j >= found && j < found + take) r[j] = root;
                    found += take;
                    run = found < m;
                    x = from - root_gap(1);
                }
            }
        }
    }
    ok = ok && found == m;
    // 3.
    double W[kMaxClamped][n], c[kMaxClamped];
#pragma unroll
    for (int j = 0; j < kMaxClamped; ++j)
    {
        if (ok && j < m)
        {
            double lam = r[j], z[n];
            bool shared = false;
#pragma unroll
            for (int q = 0; q < kMaxClamped; ++q) shared = shared || (q != j && q < m && r[q] == r[j]);
            if (shared) lam -= kSharedShift;
            {
                // pivots from the top (dp) and from the bottom (dm), side by side
                double l[n], u[n], dp[n], dm[n];
                dp[0] = d[0] - lam;
                dm[n - 1] = d[n - 1] - lam;
#pragma unroll
                for (int i = 0; i + 1 < n; ++i)
                {
                    const int b = n - 1 - i;
                    dp[i] = off_zero(dp[i]);
                    dm[b] = off_zero(dm[b]);
                    l[i] = e[i] * refined_rcp(dp[i]);
                    u[b - 1] = e[b - 1] * refined_rcp(dm[b]);
                    dp[i + 1] = (d[i + 1] - lam) - e[i] * l[i];
                    dm[b - 1] = (d[b - 1] - lam) - e[b - 1] * u[b - 1];
                }
                // the smallest twist pivot's vector (of roots close to an
                // earlier one, not the earlier vector again)
                double best = 1e300;
                int k = n - 1;
#pragma unroll
                for (int i = n - 1; i >= 0; --i)
                {
                    const double gi = fabs(dp[i] + (dm[i] - (d[i] - lam)));
                    double used = 0.0;
#pragma unroll
                    for (int q = 0; q < j; ++q) used += W[q][i] * W[q][i];
                    if (used < 0.5 && gi < best)
                    {
                        best = gi;
                        k = i;
                    }
                }
                z[n - 1] = k == n - 1 ? 1.0 : 0.0;
#pragma unroll
                for (int i = n - 2; i >= 0; --i) z[i] = i == k ? 1.0 : (i < k ? -l[i] * z[i + 1] : 0.0);
#pragma unroll
                for (int i = 0; i + 1 < n; ++i)
                    if (i >= k) z[i + 1] = -u[i] * z[i];
                double zz = 0.0;
#pragma unroll
                for (int i = 0; i < n; ++i) zz += z[i] * z[i];
                const double iz = ql_rsqrt(zz);
#pragma unroll
                for (int i = 0; i < n; ++i) z[i] *= iz;
            }
            double rho = 0.0, rr = 0.0;  // Rayleigh quotient, squared residual
#pragma unroll 1
            for (int pass = 0; pass < kVectorPasses; ++pass)
            {
                if (pass > 0)
                {
                    tridiag_solve<n>(d, e, pass == 1 ? lam : rho, z);
                    normalize<n>(z);
                }
                double zz = 1.0;  // what the second orthogonalization kept
                if (j > 0)
#pragma unroll
                    for (int t = 0; t < 2; ++t)
                    {
#pragma unroll
                        for (int q = 0; q < j; ++q)
                        {
                            double s = 0.0;
#pragma unroll
                            for (int i = 0; i < n; ++i) s += W[q][i] * z[i];
#pragma unroll
                            for (int i = 0; i < n; ++i) z[i] -= s * W[q][i];
                        }
                        zz = 0.0;
#pragma unroll
                        for (int i = 0; i < n; ++i) zz += z[i] * z[i];
                        const double iz = ql_rsqrt(zz);
#pragma unroll
                        for (int i = 0; i < n; ++i) z[i] *= iz;
                    }
                double tz[n];
                rho = 0.0;
                rr = 0.0;
#pragma unroll
                for (int i = 0; i < n; ++i)
                {
                    tz[i] = d[i] * z[i] + (i + 1 < n ? e[i] * z[i + 1] : 0.0) + (i > 0 ? e[i - 1] * z[i - 1] : 0.0);
                    rho += z[i] * tz[i];
                }
#pragma unroll
                for (int i = 0; i < n; ++i)
                {
                    const double t = tz[i] - rho * z[i];
                    rr += t * t;
                }
                if (!(zz > 0.5)) rr = 1.0;
                if (rr < kResidual * kResidual) break;
            }
#pragma unroll
            for (int i = 0; i < n; ++i) W[j][i] = z[i];
            ok = ok && rr < kResidualMax * kResidualMax && rho < start - kRootRounding;
            c[j] = fmax(eps < 0.0 ? -2.0 * rho : level - rho, 0.0);
        }
    }
    // 4. (the reflectors are read, not kept: the compiler does not look past this)
    asm volatile("" ::: "memory");
    double P[Sym<n>::n];
    {
        const bool all = ok && flip && !(eps < 0.0);  // all at the level but for the others' vectors
        const double sign = flip && !ok ? -1.0 : 1.0;   // (A as it was)
#pragma unroll
        for (int i = 0; i < n; ++i)
#pragma unroll
            for (int j = i; j < n; ++j)
                P[Sym<n>::idx(i, j)] = i == j       ? ldexp(all ? -level : sign * d[i], ex)
                                       : j == i + 1 ? ldexp(all ? 0.0 : sign * e[i], ex)
                                                    : 0.0;
    }
#pragma unroll
    for (int q = 0; q < kMaxClamped; ++q)
        if (ok && q < m)
        {
            const double cq = ldexp(c[q], ex);
#pragma unroll
            for (int i = 0; i < n; ++i)
            {
                const double ci = cq * W[q][i];
#pragma unroll
                for (int j = i; j < n; ++j) P[Sym<n>::idx(i, j)] += ci * W[q][j];
            }
        }
#pragma unroll
    for (int k = n - 3; k >= 0; --k)
    {
        const int L = n - k - 1;
        double v[n], vv = 0.0;
#pragma unroll
        for (int i = 0; i < L; ++i) v[i] = store[(reflector_at(n, k) + i) * 64];
#pragma unroll
        for (int i = 1; i < L; ++i) vv += v[i] * v[i];
        vv += v[0] * v[0];
        const double tau = vv > 0.0 ? 2.0 * refined_rcp(vv) : 0.0;
#pragma unroll
        for (int row = 0; row <= k; ++row)
        {
            double s = 0.0;
#pragma unroll
            for (int i = 0; i < L; ++i) s += P[Sym<n>::idx(row, k + 1 + i)] * v[i];
            s *= tau;
#pragma unroll
            for (int i = 0; i < L; ++i) P[Sym<n>::idx(row, k + 1 + i)] -= s * v[i];
        }
        double pv[n], vp = 0.0;
#pragma unroll
        for (int i = 0; i < L; ++i)
        {
            double acc = 0.0;
#pragma unroll
            for (int j = 0; j < L; ++j) acc += P[Sym<n>::at(k + 1 + i, k + 1 + j)] * v[j];
            pv[i] = tau * acc;
            vp += v[i] * pv[i];
        }
        const double K = 0.5 * tau * vp;
#pragma unroll
        for (int i = 0; i < L; ++i) pv[i] -= K * v[i];
#pragma unroll
        for (int i = 0; i < L; ++i)
#pragma unroll
            for (int j = i; j < L; ++j)
                P[Sym<n>::idx(k + 1 + i, k + 1 + j)] -=
                    v[i] * pv[j] + pv[i] * v[j];
    }
#pragma unroll
    for (int q = 0; q < Sym<n>::n; ++q) A[q] = P[q];
    return ok;
}

// Projects packed symmetric A in place through its whole spectrum; returns
// true when A was modified.
template <int n, class T, bool KeepUnchanged, bool InMemory = false>
__device__ __forceinline__ bool project_spectrum(T* A, T eps)
{
    T Wbuf[KeepUnchanged ? Sym<n>::n : 1];
    T* W = A;
    if constexpr (KeepUnchanged)
    {
#pragma unroll
        for (int i = 0; i < Sym<n>::n; ++i) Wbuf[i] = A[i];
        W = Wbuf;
    }
    T V[n * n];
    T lam[n];
    tridiag_ql_eigen<n, T, InMemory>(W, V, lam);
    bool changed = false;
#pragma unroll
    for (int i = 0; i < n; ++i)
    {
        T l = lam[i];
        if (eps < T(0))
        {
            changed = changed || (l < T(0));
            l = l < T(0) ? -l : l;
        }
        else
        {
            changed = changed || (l < eps);
            l = l < eps ? eps : l;
        }
        lam[i] = l;
    }
    if constexpr (KeepUnchanged)
        if (!changed)
            return false;
    constexpr int kRows = InMemory ? 1 : n;
    T P[InMemory ? n * n : 1];
#pragma unroll kRows
    for (int i = 0; i < n; ++i)
#pragma unroll kRows
        for (int j = i; j < n; ++j)
        {
            T acc = T(0);
#pragma unroll
            for (int m = 0; m < n; ++m) acc += V[i * n + m] * lam[m] * V[j * n + m];
            if constexpr (InMemory) P[i * n + j] = acc;
            else A[Sym<n>::idx(i, j)] = acc;
        }
    if constexpr (InMemory)
    {
#pragma unroll
        for (int i = 0; i < n; ++i)
#pragma unroll
            for (int j = i; j < n; ++j) A[Sym<n>::idx(i, j)] = P[i * n + j];
    }
    return true;
}

// Projects packed symmetric A in place.  Returns true when A was modified.
// KeepUnchanged: when no eigenvalue needs clamping, A is left bit-identical
// (the reference returns its input untouched then); this keeps a copy of A
// alive through the eigensolve.  Without it the spectrum is re-assembled
// whenever the Cholesky test failed (equal to A up to rounding when nothing
// was clamped), which saves n(n+1)/2 registers during the eigensolve.
template <int n, class T, bool KeepUnchanged = true>
__device__ __forceinline__ bool project_psd(T* A, T eps)
{
    if (cholesky_pd<n, T>(A, eps > T(0) ? eps : T(0))) return false;
    return project_spectrum<n, T, KeepUnchanged>(A, eps);
}

// The same, without KeepUnchanged, for a wave that holds one matrix per lane
// and has reflector_values(n) x 64 values of LDS for it (store: this lane's
// first, the others 64 apart).
template <int n>
__device__ __forceinline__ void project_psd_few(double* A, double eps, double* store)
{
    if (ldl_pd<n>(A, eps > 0.0 ? eps : 0.0)) return;
    if (!project_few<n>(A, eps, store)) project_spectrum<n, double, false, true>(A, eps);
}

} // namespace tad
