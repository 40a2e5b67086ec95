"""Kernels at the edges of their tiles and dispatch ranges, through the public
entry points, against direct solves and the CPU oracle."""
import numpy as np
import pytest

import tinyad_amd as tad
from tinyad_amd import configs

pytestmark = pytest.mark.gpu


def nrel(a, b):
    a, b = np.asarray(a, dtype=np.float64), np.asarray(b, dtype=np.float64)
    return float(np.abs(a - b).max(initial=0.0) / max(np.abs(b).max(initial=0.0), 1e-300))


def pinned_grid(n, seed=1):
    """grid_param with its left and right columns pinned (a definite Hessian)."""
    P = configs.grid_param(n, seed)
    cols = np.concatenate([np.arange(n) * n, np.arange(n) * n + n - 1]).astype(np.int32)
    pins = configs.Term(configs.E_PENALTY, cols[:, None].copy(),
                        np.concatenate([P.x0.reshape(-1, 2)[cols], np.ones((cols.size, 1))], axis=1))
    return configs.Problem(f"grid_pinned_{n}", 2, P.n_handles, [P.terms[0], pins], P.x0)


# unknowns below, at and past the 64-column pivot tiles, and a size whose tile
# columns are cut into several strips
@pytest.mark.parametrize("n", [4, 5, 8, 9, 16, 22, 40])
def test_dense_inverse_tile_edges(ctx, n):
    """The coarse inverse with one aggregate per handle and translations only
    (no Hessian evaluated by the solving function): P = I, so A_c = H and the
    preconditioned matrix is I + D^-1 H, with a spectrum in (1, 1 + 3.2] for
    block-Jacobi on triangles (measured bound of lambda_max(D^-1 H): 2.3).
    Chebyshev's bound for that interval gives 1e-12 within 21 iterations; a
    wrong inverse does not."""
    import scipy.sparse.linalg as spla
    P = pinned_grid(n)
    f, g, H = tad.ScalarFunction.from_problem(P, ctx).eval_with_hessian_proj(P.x0)
    fn = tad.ScalarFunction.from_problem(P, ctx)
    d, st = fn.solve(g, H=H, tol=1e-12, coarse_aggregate=1)
    assert st.converged and st.coarse_unknowns == 2 * n * n
    assert st.iters <= 24
    assert nrel(d, spla.spsolve(H.tocsc(), g)) <= 1e-9


def quadratic_chain(d, n, seed=0):
    """Quadratic elements on the handle pairs (i, i + 1) and (i, i + 5), permuted
    handles, the last handle in no element; every element Hessian has its
    spectrum in [1, 3]."""
    rng = np.random.default_rng(seed)
    perm = rng.permutation(n)
    pairs = [(i, i + 1) for i in range(n - 2)] + [(i, i + 5) for i in range(n - 6)]
    conn = perm[np.array(pairs, dtype=np.int64).reshape(-1, 2)].astype(np.int32)
    K = 2 * d
    Q = np.linalg.qr(rng.normal(size=(conn.shape[0], K, K)))[0]
    A = np.einsum("eik,ek,ejk->eij", Q, rng.uniform(1.0, 3.0, (conn.shape[0], K)), Q)
    A = 0.5 * (A + A.transpose(0, 2, 1))
    params = np.concatenate([A.reshape(-1, K * K), np.zeros((conn.shape[0], K + 1))], axis=1)
    return configs.Problem("quadratic_chain", d, n, [configs.Term(configs.E_QUADRATIC, conn, params)],
                           rng.normal(size=d * n))


# handles around the update kernel's chunks of 64 and the product's groups of
# 32 rows; aggregates smaller than, equal to and larger than a chunk, and off
@pytest.mark.parametrize("d", [1, 2, 3])
@pytest.mark.parametrize("n", [3, 33, 64, 65, 200, 700])
@pytest.mark.parametrize("agg", [0, 3, 64, 150])
def test_solver_order_edges(ctx, d, n, agg):
    """Solves in solver order (aggregates, parts, chunks; a handle without
    elements; a free-variable mask) against direct solves of w I + H.  The
    condition number is at most 40 (element spectra in [1, 3], at most four
    elements per handle, w = 0.3), so a relative residual of 1e-13 bounds the
    solution error by 4e-12."""
    import scipy.sparse as sp
    import scipy.sparse.linalg as spla
    fn = tad.ScalarFunction.from_problem(quadratic_chain(d, n), ctx)
    rng = np.random.default_rng(n)
    _, _, H = fn.eval_with_derivatives(rng.normal(size=d * n))
    A = (H + 0.3 * sp.identity(d * n)).tocsc()
    b = rng.normal(size=d * n)
    x, st = fn.solve(b, tol=1e-13, w_identity=0.3, coarse_aggregate=agg)
    assert st.converged and nrel(x, spla.spsolve(A, b)) <= 1e-10
    free = (rng.random(d * n) < 0.7).astype(np.uint8)
    free[0] = 1
    fi = np.nonzero(free)[0]
    ref = np.zeros(d * n)
    ref[fi] = np.atleast_1d(spla.spsolve(A[fi][:, fi].tocsc(), b[fi]))
    x, st = fn.solve(b, free=free, tol=1e-13, w_identity=0.3, coarse_aggregate=agg)
    assert st.converged and nrel(x, ref) <= 1e-10 and np.all(x[free == 0] == 0.0)
    x2, st2 = fn.solve(b, free=free, tol=1e-13, w_identity=0.3, coarse_aggregate=agg)
    assert np.array_equal(x, x2) and st.iters == st2.iters


# one pivot tile and less, a tile boundary, several tiles, and the largest
# sizes the dense preconditioner takes (2,400 variables, 1,536 in 3D)
@pytest.mark.parametrize("kind,n", [("grid", 3), ("grid", 8), ("grid", 17), ("grid", 34), ("cube", 2), ("cube", 3),
                                    ("cube", 7)])
def test_small_systems_dense_preconditioner(ctx, kind, n):
    """Automatic solves of small systems: the dense inverse makes the
    preconditioned matrix the identity to rounding (condition numbers below
    1e6), so two CG iterations reach 1e-12; against direct solves, with a
    free-variable mask, with w, and with a reused inverse of another Hessian
    (whose preconditioned spectrum is a few percent wide here)."""
    import scipy.sparse as sp
    import scipy.sparse.linalg as spla
    P = pinned_grid(n) if kind == "grid" else configs.twist_cube(m=n, seed=2)
    fn = tad.ScalarFunction.from_problem(P, ctx)
    f, g, H = fn.eval_with_hessian_proj(P.x0)
    nv = g.size
    for w in (0.0, 0.3):
        d, st = fn.solve(g, tol=1e-12, w_identity=w)
        assert st.converged and st.coarse_unknowns == nv and st.iters <= 2
        assert nrel(d, spla.spsolve((H + w * sp.identity(nv)).tocsc(), g)) <= 1e-9
    free = np.ones(nv, dtype=np.uint8)
    free[: nv // 3] = 0
    fi = np.nonzero(free)[0]
    d, st = fn.solve(g, free=free, tol=1e-12)
    ref = np.zeros(nv)
    ref[fi] = spla.spsolve(H.tocsr()[fi][:, fi].tocsc(), g[fi])
    assert st.converged and st.iters <= 2 and nrel(d, ref) <= 1e-9 and np.all(d[free == 0] == 0.0)
    fn.solve(g, tol=1e-12)
    scale = 1.0 + 0.05 * np.cos(np.arange(nv))
    S = sp.diags(scale)
    H2 = (S @ H @ S).tocsr()  # same pattern, still positive definite
    H2.sort_indices()
    d, st = fn.solve(g, H=H2.data, tol=1e-12, coarse_reuse=1)
    assert st.converged and st.coarse_reused == 1
    assert nrel(d, spla.spsolve(H2.tocsc(), g)) <= 1e-9


def star_quadratic(d, n, seed=0):
    """Quadratic pairs (0, i): handle 0's block row holds n blocks."""
    rng = np.random.default_rng(seed)
    conn = np.stack([np.zeros(n - 1, dtype=np.int32), np.arange(1, n, dtype=np.int32)], axis=1)
    K = 2 * d
    A = rng.normal(size=(n - 1, K, K))
    A = A + A.transpose(0, 2, 1)
    params = np.concatenate([A.reshape(-1, K * K), rng.normal(size=(n - 1, K + 1))], axis=1)
    return configs.Problem("star", d, n, [configs.Term(configs.E_QUADRATIC, conn, params)], rng.normal(size=d * n))


# block rows below, at and above a tile of 256 blocks, and tiles that end in
# the middle of the chip's eight-fold split
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("d", [1, 2, 3])
@pytest.mark.parametrize("n", [2, 255, 256, 257, 300, 2000])
def test_assembly_tiles(ctx, d, n, precision):
    """Assembly by tiles of rows against one thread per block (the same sums in
    the same order: identical bits) and against the sum of the element
    matrices; the second term interleaves short rows."""
    P = star_quadratic(d, n)
    Q = quadratic_chain(d, max(n, 8), seed=1)
    P = configs.Problem("both", d, max(n, 8), P.terms + Q.terms, Q.x0)
    fn = tad.ScalarFunction.from_problem(P, ctx, precision)
    x = P.x0
    out = []
    for shape in (0, 1):
        fn.assembly_shape = shape
        f, g, H = fn.eval_with_derivatives(x)
        out.append((f, g, H.toarray()))
    assert out[0][0] == out[1][0] and np.array_equal(out[0][1], out[1][1]) and np.array_equal(out[0][2], out[1][2])
    ref = np.zeros((x.size, x.size))
    for t in P.terms:
        K = t.valence * d
        A = t.params[:, : K * K].reshape(-1, K, K)
        idx = (t.conn[:, :, None] * d + np.arange(d)).reshape(-1, K)
        np.add.at(ref, (idx[:, :, None], idx[:, None, :]), A)
    # FP64: sums of at most 2,000 terms; mixed: FP32 contributions, FP64 sums
    assert np.abs(out[0][2] - ref).max() <= (1e-12 if precision == "fp64" else 1e-6) * np.abs(ref).max()


def tet_states(P, state):
    rest = P.info["rest"].reshape(-1, 3)
    rng = np.random.default_rng(5)
    if state == "rest":            # three eigenvalues 0 to rounding
        x = rest.copy()
    elif state == "noise":         # three small ones of either sign, close together
        x = rest + 1e-4 * P.info["h"] * rng.normal(size=rest.shape)
    elif state == "compressed":    # three below 0
        x = 0.9 * rest
    elif state == "flattened":     # two below 0, one at 0 to rounding
        x = rest * np.array([1.0, 1.0, 0.8])
    elif state == "stretched":     # none to clamp
        x = 1.2 * rest
    else:                          # some elements inverted (zero Hessian)
        x = rest + 0.1 * P.info["h"] * rng.normal(size=rest.shape)
        x[::5] += 1.5 * P.info["h"]
    return np.ascontiguousarray(x).reshape(-1)


# 6, 48, 162 and 384 tets: one short group of 64, a full and a short one, ...
@pytest.mark.parametrize("state", ["rest", "noise", "compressed", "flattened", "stretched", "inverted"])
@pytest.mark.parametrize("m", [1, 2, 3, 4])
def test_tet_projection_cases(ctx, m, state):
    """FP64 tets projected through their clamped eigenvalues against the
    oracle's full eigensolve, also with a level that clamps more than three of
    them and with absolute values, plain and persistent launches.  Each side's
    element error is below 30 eps |H_e| (7e-15), a block sums at most 24
    elements: 24 * 2 * 7e-15 < 1e-12."""
    import oracle
    P = configs.twist_cube(m=m)
    x = tet_states(P, state)
    fg = tad.ScalarFunction.from_problem(P, ctx)
    fo = oracle.Function.from_problem(P)
    for eps in (1e-9, 0.05, -1.0, 0.0):
        ref = fo.eval_with_hessian_proj(x, eps)[2]
        for shape in [(0, 0, 0), (64, 8, 1), (256, 1, 0)]:
            fg.set_launch_shape(0, *shape)
            f, g, H = fg.eval_with_hessian_proj(x, eps)
            assert nrel(H.toarray(), ref.toarray()) <= 1e-12, (eps, shape)


@pytest.mark.parametrize("batch", [1, 2, 3, 4, 8])
def test_line_search_batches(ctx, batch):
    """The step accepted on the device does not depend on the batch size, and
    a limit on the trials holds inside a batch: one trial fewer than needed
    accepts nothing and returns x0."""
    import torch
    P = configs.twist_cube(m=3, seed=5)
    fg = tad.ScalarFunction.from_problem(P, ctx)
    f, g, H = fg.eval_with_hessian_proj(P.x0)
    d, _ = fg.solve(g, w=1e-6)
    x, dt, gt = (torch.tensor(a, device="cuda:0") for a in (P.x0, -200.0 * np.asarray(d), g))
    ref, f_ref, s_ref, n_ref = fg.line_search(x, dt, f, gt, opts=tad.newton_default_opts(ls_batch=1))
    assert n_ref > 8
    out, f_new, s, n = fg.line_search(x, dt, f, gt, opts=tad.newton_default_opts(ls_batch=batch))
    assert (f_new, s, n) == (f_ref, s_ref, n_ref) and torch.equal(out, ref)
    out, f_new, s, n = fg.line_search(x, dt, f, gt, opts=tad.newton_default_opts(ls_batch=batch, ls_max_iters=n_ref))
    assert (f_new, s, n) == (f_ref, s_ref, n_ref) and torch.equal(out, ref)
    out, f_new, s, n = fg.line_search(x, dt, f, gt,
                                      opts=tad.newton_default_opts(ls_batch=batch, ls_max_iters=n_ref - 1))
    assert n < 0 and s == 0.0 and torch.equal(out, x)
