"""The few-eigenvalue projection of FP64 tets (Projection.hpp), compiled for the
host, on element matrices near and at rest, compressed, flattened and twisted,
and on spectra with close roots around the clamp level: its error against a
full eigendecomposition, and how often it hands a matrix to the full
eigensolve.  The kernels run the same code, one matrix per lane."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from tinyad_amd import configs

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

STUB = """
#pragma once
#include <algorithm>
#include <cmath>
#include <cstdint>
#define __device__
#define __host__
#define __forceinline__ inline
using std::max; using std::copysign; using std::fabs; using std::fma; using std::fmax; using std::frexp; using std::ldexp; using std::rint; using std::sqrt;
// (single precision accuracy, as the hardware's approximations have)
inline double __builtin_amdgcn_rcp(double x) { return 1.0 / x * (1 + 3e-8); }
inline double __builtin_amdgcn_rsq(double x) { return 1.0 / std::sqrt(x) * (1 + 3e-8); }
inline float __builtin_amdgcn_rsqf(float x) { return 1.0f / std::sqrt(x); }
inline double rsqrt(double x) { return 1.0 / std::sqrt(x); }
"""

HARNESS = """
#include "tinyad_amd/device/Projection.hpp"
// status per matrix: 0 positive definite, 1 projected, 2 given to the full eigensolve
extern "C" void project(long n, double eps, double* A, int* status)
{
    static double store[64 * 64];
    for (long q = 0; q < n; ++q)
    {
        double* a = A + 45 * q;
        if (tad::ldl_pd<9>(a, eps > 0.0 ? eps : 0.0)) status[q] = 0;
        else status[q] = tad::project_few<9>(a, eps, store) ? 1 : 2;
    }
}
"""

IU = np.triu_indices(9)


@pytest.fixture(scope="module")
def project(tmp_path_factory):
    d = tmp_path_factory.mktemp("projection")
    os.makedirs(d / "hip")
    (d / "hip" / "hip_runtime.h").write_text(STUB)
    (d / "harness.cpp").write_text(HARNESS)
    so = str(d / "projection.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-Wno-unknown-pragmas", f"-I{d}",
                    "-I" + os.path.join(ROOT, "include"), str(d / "harness.cpp"), "-o", so], check=True)
    f = ctypes.CDLL(so).project
    f.argtypes = [ctypes.c_long, ctypes.c_double, ctypes.c_void_p, ctypes.c_void_p]
    f.restype = None

    def run(K, eps):
        A = np.ascontiguousarray(K[:, IU[0], IU[1]])
        status = np.zeros(len(K), dtype=np.int32)
        f(len(K), eps, A.ctypes.data, status.ctypes.data)
        P = np.zeros_like(K)
        P[:, IU[0], IU[1]] = A
        P[:, IU[1], IU[0]] = A
        return P, status

    return run


def reference(K, eps):
    lam, V = np.linalg.eigh(K)
    lam = np.abs(lam) if eps < 0 else np.maximum(lam, eps)
    return np.einsum("nik,nk,njk->nij", V, lam, V)


def check(project, K, eps, fallback):
    """numpy's eigendecomposition of a 9 x 9 matrix is accurate to about 20 eps
    = 4e-15 |A|; the accepted residual is 4e-15 of T's norm, at most 3 |A| here,
    and counts up to three times (once per clamped vector), twice for absolute
    values: 4e-15 + 7.2e-14 < 1e-13 (the largest entry for |A|)."""
    P, status = project(K, eps)
    scale = np.maximum(np.abs(K).max(axis=(1, 2)), eps)
    few = status == 1
    err = np.abs(P - reference(K, eps)).max(axis=(1, 2)) / scale
    assert err[few].max(initial=0.0) <= 1e-13, eps
    # the others are A unchanged up to rounding (Householder there and back)
    back = np.abs(P - K).max(axis=(1, 2)) / scale
    assert back[status != 1].max(initial=0.0) <= 1e-13
    assert np.count_nonzero(status == 2) <= fallback * np.count_nonzero(status), (eps, np.bincount(status))


def tets():
    P = configs.twist_cube(m=7)
    t = [t for t in P.terms if t.valence == 4][0]
    return P.info["rest"].reshape(-1, 3), P.info["h"], t.conn, t.params


def element_matrices(x, conn, params):
    """Hessians of the symmetric-Dirichlet tets in the nine directions
    orthogonal to the translations."""
    R, w = params[:, :9].reshape(-1, 3, 3), params[:, 9]
    J = (x[conn[:, 1:]] - x[conn[:, :1]]).transpose(0, 2, 1) @ R
    A = np.linalg.inv(J)
    At = A.transpose(0, 2, 1)
    C = At @ A @ At
    H = 2.0 * np.einsum("nik,njl->nijkl", At @ A, A @ At)
    H += 2.0 * np.einsum("ik,jl->ijkl", np.eye(3), np.eye(3))
    H += 2.0 * np.einsum("nil,njk->nijkl", C, A) + 2.0 * np.einsum("nkj,nli->nijkl", C, A)
    D = np.concatenate([-R.sum(1, keepdims=True), R], axis=1)
    Q = np.linalg.qr(np.concatenate([np.ones((4, 1)), np.eye(4)[:, :3]], axis=1))[0][:, 1:]
    E = Q.T @ D
    return np.einsum("n,naj,nbk,nijlk->naibl", w, E, E, H, optimize=True).reshape(-1, 9, 9)


def moved(rest, h, state):
    kind, a = state
    if kind == "noise":
        return rest + a * h * np.random.default_rng(3).standard_normal(rest.shape)
    if kind == "smooth":
        return rest + a * np.sin(np.pi * rest[:, [1, 2, 0]] + 0.3)
    if kind == "compressed":
        return rest * (1.0 - a)
    if kind == "flattened":
        return rest * np.array([1.0, 1.0, 1.0 - a])
    th = np.radians(a) * rest[:, 2]
    px, py = rest[:, 0] - 0.5, rest[:, 1] - 0.5
    return np.stack([0.5 + np.cos(th) * px - np.sin(th) * py, 0.5 + np.sin(th) * px + np.cos(th) * py, rest[:, 2]], axis=1)


# where the clamped roots are apart by more than a few roundings
@pytest.mark.parametrize("state", [("noise", 0.0)] + [("noise", 10.0 ** -k) for k in (12, 11, 10, 9, 8, 7, 6, 5, 4, 3, 2)]
                         + [("smooth", 10.0 ** -k) for k in (8, 5, 4, 3)]
                         + [("compressed", a) for a in (1e-9, 1e-7, 1e-5, 1e-4, 1e-3, 0.1, 0.2)]
                         + [("flattened", a) for a in (1e-9, 1e-7, 1e-4, 0.1, 0.2)]
                         + [("twisted", a) for a in (0.01, 1.0, 30.0, 60.0)], ids=lambda s: f"{s[0]}_{s[1]:g}")
def test_element_states(project, state):
    """At most 1 % of the elements (0.3 % measured) go to the full eigensolve."""
    rest, h, conn, params = tets()
    K = element_matrices(moved(rest, h, state), conn, params)
    for eps in (1e-9, 0.0, -1.0):
        check(project, K, eps, 0.01)


@pytest.mark.parametrize("spread", [0.0, 1e-16, 1e-14, 1e-12, 1e-11, 1e-10, 1e-9, 1e-8, 1e-6, 1e-4])
@pytest.mark.parametrize("near", [2, 3])
@pytest.mark.parametrize("base", [-0.5, 0.0, 1e-9])
def test_close_roots(project, base, near, spread):
    """Two or three roots within `spread` of each other, clamped or around the
    level, in random directions; any number of them may be given back."""
    rng = np.random.default_rng(11)
    n = 400
    Q = np.linalg.qr(rng.standard_normal((n, 9, 9)))[0]
    lam = 0.05 + np.abs(rng.standard_normal((n, 9)))
    lam[:, :near] = base + spread * rng.standard_normal((n, near))
    K = np.einsum("nik,nk,njk->nij", Q, lam, Q)
    K = 0.5 * (K + K.transpose(0, 2, 1))
    for eps in (1e-9, 0.0, -1.0):
        check(project, K, eps, 0.05 if base < 0.0 else 1.0)


@pytest.mark.parametrize("state", [("noise", 0.0), ("noise", 1e-6), ("noise", 1e-2), ("compressed", 0.1), ("twisted", 54.0)],
                         ids=lambda s: f"{s[0]}_{s[1]:g}")
@pytest.mark.parametrize("eps", [0.02, 0.1, 0.2, 0.3, 0.5, 0.8, 5.0, 1e6])
def test_large_clamp_levels(project, state, eps):
    """Levels among and above the eigenvalues (0.1 .. 1 here): four to all nine
    of them are clamped; still at most 1 % go to the full eigensolve."""
    rest, h, conn, params = tets()
    check(project, element_matrices(moved(rest, h, state), conn, params), eps, 0.01)


def test_absolute_values_of_mostly_negative_matrices(project):
    """Any number of negative eigenvalues, with and without close ones."""
    rng = np.random.default_rng(4)
    for negative in range(10):
        Q = np.linalg.qr(rng.standard_normal((200, 9, 9)))[0]
        lam = 0.05 + np.abs(rng.standard_normal((200, 9)))
        lam[:, :negative] *= -1.0
        lam[:100, 1] = lam[:100, 0] * (1.0 + 1e-9)
        K = np.einsum("nik,nk,njk->nij", Q, lam, Q)
        for eps in (-1.0, 0.0, 1e-9):
            check(project, 0.5 * (K + K.transpose(0, 2, 1)), eps, 0.01)
