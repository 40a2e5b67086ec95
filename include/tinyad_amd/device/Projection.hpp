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

// Most eigenvalues project_few clamps (three bounds what an
// isotropic energy of a tet has below zero: one per pair of singular values).
constexpr int kMaxClamped = 3;
// On the scaled tridiagonal: where the search for the next root starts below
// the last one; the Laguerre step at which a root is final; the distance from
// the level below which a root counts as the level itself, and where the
// count starts then; how far equal roots may be moved, the other roots' share
// of the log-derivative they allow per step, and the shift off them for their
// vectors; the residual at which a vector is final and the largest accepted.
constexpr double kRootGap = 1e-5, kRootStep = 1e-7, kRootApart = 1e-13, kLevelShift = 1e-9,
                 kWeakMove = 1e-7, kWeakShare = 1e4, kWeakShift = 1e-9, kResidual = 2e-15, kResidualMax = 1e-14;

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
            q = fabs(q) < 1e-100 ? -1e-100 : q;
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
    q = fabs(q) < 1e-100 ? -1e-100 : q;
    const double r = refined_rcp(q);
    count += q < 0.0 ? 1 : 0;
    const double q2 = w[0] * (u[0] - 2.0 * t[0] * t[0]) + w[1] * (u[1] - 2.0 * t[1] * t[1]);
    const double tm = (w[0] * t[0] + (w[1] * t[1] - 1.0)) * r;
    s1 = a1[0] + a1[1] + tm;
    s2 = a2[0] + a2[1] + (q2 * r - tm * tm);
    return count;
}

// Place of reflector k (n - 1 - k values) among the stored ones, and their
// number.
__host__ __device__ constexpr int reflector_at(int n, int k) { return k * (n - 1) - k * (k - 1) / 2; }
__host__ __device__ constexpr int reflector_values(int n) { return reflector_at(n, n - 2); }

// Projects packed symmetric A in place when few eigenvalues are clamped:
//   P(A) = A + sum_j (clamped_j - lam_j) v_j v_j^T
// over the eigenvalues below the clamp level only, so no other eigenvector
// and no full spectrum is computed.  Returns false, with A restored up to
// rounding, when more than kMaxClamped eigenvalues are clamped or a vector
// misses its residual or orthogonality bound; the caller then projects A by
// the full eigensolve (none of 24,000 elements of the 16^3 twisted cube, 0.1 %
// of those within 1e-4 of a rest state).
//   1. Householder reduction to the tridiagonal T, scaled by a power of two
//      to norm 1, the reflectors going to `store` (in registers they do not
//      fit beside the rest); the number m of clamped eigenvalues from the
//      pivot signs.
//   2. Their values from right to left by Laguerre's iteration (cubic, and
//      monotone towards the neighbouring root as all roots are real), each
//      started below the previous root, which is divided out: 6.7 evaluations
//      per matrix, 10.7 for the slowest lane of a wave, where the full QL
//      iteration takes 27.5 sweeps of a wave.
//   3. Their vectors from twisted factorizations of T - lam I (Fernando,
//      SIAM J. Matrix Anal. Appl. 18 (1997) 1013-1034) at the index with the
//      smallest twist pivot, which gives the residual; Rayleigh quotient
//      steps until it is at rounding level; two Gram-Schmidt passes, so that
//      close eigenvalues (whose vectors are determined as a set only) give
//      orthonormal vectors of their common space.
//   4. T + sum c w w^T, then the reflectors from both sides.
// Error against 80-bit arithmetic on those elements, relative to |A|: 7e-16
// in the mean, 3e-15 at most (full eigensolve: 1.4e-15 and 5e-15).
template <int n>
__device__ __forceinline__ bool project_few(double* A, double eps, double* store)
{
    double amax = 0.0;
#pragma unroll
    for (int q = 0; q < Sym<n>::n; ++q) amax = fmax(amax, fabs(A[q]));
    if (!(amax > 1e-100 && amax < 1e100)) return false;
    double d[n], e[n], tau[n - 2];
    // 1. as in tridiag_ql_eigen, with refined reciprocals
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
        tau[k] = tk;
        A[Sym<n>::idx(k, k + 1)] = v0;
#pragma unroll
        for (int i = 0; i < L; ++i) store[(reflector_at(n, k) + i) * 64] = A[Sym<n>::idx(k, k + 1 + i)];
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
    const double level = ldexp(eps > 0.0 ? eps : 0.0, -ex);
    // 2. roots r[0] >= r[1] >= ... below the level
    double r[kMaxClamped] = {};
    int m = 0, found = 0;
    bool weak = false;     // roots that count as one value
    double start = level;  // the roots below it are clamped
    {
        double x = level;
        bool fresh = false, run = true, first = true;
#pragma unroll 1
        for (int it = 0; run && it < 48; ++it)
        {
            double g, h;
            const int below = tridiag_count<n>(d, e2, x, g, h);
            h = -h;
            if (first)
            {
                m = below;
                if (m == 0 || m > kMaxClamped) break;
                first = false;
            }
            if (below < m - found)
            {
                // a root between x and the last one found: too close to tell
                // apart from it; or x itself, passed by rounding
                if (fresh) break;
            }
#pragma unroll
            for (int j = 0; j + 1 < kMaxClamped; ++j)
                if (j < found)
                {
                    const double q = refined_rcp(x - r[j]);
                    g -= q;
                    h -= q * q;
                }
            const double deg = (double)(n - found);
            const double gg = g * g;
            const double disc = (deg - 1.0) * (deg * h - gg);
            const double sq = disc > 0.0 ? disc * ql_rsqrt(disc) : 0.0;
            const double step = deg * refined_rcp(g + sq);
            // next to k equal roots g = k / (x - root), h = k / (x - root)^2, up
            // to the other roots' share (g < 0: the near ones lie above x)
            int take = 0;
            double share = 1.0;
            if (g > 0.0 && step < kRootStep)
#pragma unroll
                for (int k = kMaxClamped; k >= 1; --k)
                    if (k <= m - found && fabs(gg - k * h) < 0.01 * gg)
                    {
                        take = k;
                        share = fabs(gg - k * h);
                    }
            if (take > 1)
            {
                // equal roots: only where the clamping moves them by next to
                // nothing and the others are well apart
                const double move = eps < 0.0 ? -2.0 * x : level - x;
                if (!(move < kWeakMove && share < gg * fabs(step) * kWeakShare)) break;
                weak = true;
            }
            else if (below < m - found || (g > 0.0 && step < 2e-16))
                take = 1;
            const double root = x - (take > 1 ? take * refined_rcp(g) : step);
            if (take > 0 && found == 0 && !(root < start - kRootApart))
            {
                // the level itself is an eigenvalue up to rounding: count
                // (and clamp, by nothing) it as one of those below
                if (start != level) break;
                start = level + kLevelShift;
                x = start;
                first = true;
                continue;
            }
            x -= step;
            fresh = false;
            if (take > 0)
            {
#pragma unroll
                for (int j = 0; j < kMaxClamped; ++j)
                    if (j >= found && j < found + take) r[j] = root;
                found += take;
                run = found < m;
                x = root - kRootGap;
                fresh = true;
            }
        }
    }
    ok = ok && m <= kMaxClamped && found == m;
    // the lowest first: the vectors of equal roots next to the level (which
    // need not be accurate, they move by next to nothing) are made orthogonal
    // to the others, not the others to them
    static_assert(kMaxClamped == 3, "the order of up to three roots is reversed");
    const double top = r[0];
    r[0] = m == 3 ? r[2] : (m == 2 ? r[1] : r[0]);
    r[1] = m == 2 ? top : r[1];
    r[2] = m == 3 ? top : r[2];
    // 3.
    double W[kMaxClamped][n], c[kMaxClamped];
#pragma unroll
    for (int j = 0; j < kMaxClamped; ++j)
    {
        c[j] = 0.0;
#pragma unroll
        for (int i = 0; i < n; ++i) W[j][i] = 0.0;
        if (ok && j < m)
        {
            double lam = r[j], res = 0.0, z[n];
            bool shared = false;
#pragma unroll
            for (int q = 0; q < kMaxClamped; ++q) shared = shared || (weak && q != j && q < m && r[q] == r[j]);
            if (shared) lam -= kWeakShift;
#pragma unroll 1
            for (int pass = 0; pass < 3; ++pass)
            {
                // pivots from the top (dp) and from the bottom (dm), side by side
                double l[n], u[n], dp[n], dm[n];
                dp[0] = d[0] - lam;
                dm[n - 1] = d[n - 1] - lam;
#pragma unroll
                for (int i = 0; i + 1 < n; ++i)
                {
                    const int b = n - 1 - i;
                    dp[i] = fabs(dp[i]) < 1e-100 ? -1e-100 : dp[i];
                    dm[b] = fabs(dm[b]) < 1e-100 ? -1e-100 : dm[b];
                    l[i] = e[i] * refined_rcp(dp[i]);
                    u[b - 1] = e[b - 1] * refined_rcp(dm[b]);
                    dp[i + 1] = (d[i + 1] - lam) - e[i] * l[i];
                    dm[b - 1] = (d[b - 1] - lam) - e[b - 1] * u[b - 1];
                }
                double gamma = 0.0, best = 1e300;
                int k = n - 1;
#pragma unroll
                for (int i = n - 1; i >= 0; --i)
                {
                    const double gi = dp[i] + (dm[i] - (d[i] - lam));
                    double used = 0.0;
#pragma unroll
                    for (int q = 0; q < j; ++q) used += W[q][i] * W[q][i];
                    // the smallest pivot's vector; of equal roots the one with
                    // the largest part (shift / pivot) outside the earlier ones
                    const double rank = shared ? used - kWeakShift * refined_rcp(fmax(fabs(gi), 1e-30))
                                               : (used < 0.5 ? fabs(gi) : 1e300);
                    if (rank < best)
                    {
                        best = rank;
                        gamma = gi;
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
                res = shared ? 0.0 : fabs(gamma) * iz;
                lam += gamma * iz * iz;
                if (res < kResidual) break;
            }
            double zz = 1.0;
            if (j > 0)
            {
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
                    ok = ok && zz > 0.01;
                    const double iz = ql_rsqrt(zz);
#pragma unroll
                    for (int i = 0; i < n; ++i) z[i] *= iz;
                }
            }
                        double rho = 0.0;
#pragma unroll
            for (int i = 0; i < n; ++i)
            {
                W[j][i] = z[i];
                rho += z[i] * (d[i] * z[i] + (i + 1 < n ? 2.0 * e[i] * z[i + 1] : 0.0));
            }
            ok = ok && res < kResidualMax && rho < start + kResidualMax;
            c[j] = fmax(eps < 0.0 ? -2.0 * rho : level - rho, 0.0);
        }
    }
    // 4. (the reflectors are read, not kept: the compiler does not look past this)
    asm volatile("" ::: "memory");
    double P[Sym<n>::n];
#pragma unroll
    for (int i = 0; i < n; ++i)
#pragma unroll
        for (int j = i; j < n; ++j)
        {
            double s = i == j ? d[i] : (j == i + 1 ? e[i] : 0.0);
#pragma unroll
            for (int q = 0; q < kMaxClamped; ++q) s += ok ? c[q] * W[q][i] * W[q][j] : 0.0;
            P[Sym<n>::idx(i, j)] = ldexp(s, ex);
        }
#pragma unroll
    for (int k = n - 3; k >= 0; --k)
    {
        const int L = n - k - 1;
        double v[n];
#pragma unroll
        for (int i = 0; i < L; ++i) v[i] = store[(reflector_at(n, k) + i) * 64];
#pragma unroll
        for (int row = 0; row <= k; ++row)
        {
            double s = 0.0;
#pragma unroll
            for (int i = 0; i < L; ++i) s += P[Sym<n>::idx(row, k + 1 + i)] * v[i];
            s *= tau[k];
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
            pv[i] = tau[k] * acc;
            vp += v[i] * pv[i];
        }
        const double K = 0.5 * tau[k] * vp;
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
