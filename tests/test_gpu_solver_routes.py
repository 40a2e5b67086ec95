"""Which preconditioner a solve takes and keeps, through the public entry points."""
import numpy as np
import pytest

import tinyad_amd as tad
from tinyad_amd import configs

pytestmark = pytest.mark.gpu


def pinned_grid(n, seed=1):
    """grid_param with its left and right columns pinned (a definite Hessian)."""
    P = configs.grid_param(n, seed)
    cols = np.concatenate([np.arange(n) * n, np.arange(n) * n + n - 1]).astype(np.int32)
    pins = configs.Term(configs.E_PENALTY, cols[:, None].copy(),
                        np.concatenate([P.x0.reshape(-1, 2)[cols], np.ones((cols.size, 1))], axis=1))
    return configs.Problem(f"grid_pinned_{n}", 2, P.n_handles, [P.terms[0], pins], P.x0)


def indefinite(ctx, n):
    """(function, H, A, b): A = H - s I, of H's pattern, with one negative
    eigenvalue, and right-hand sides b with b . A^-1 b of either sign."""
    import scipy.sparse as sp
    P = pinned_grid(n)
    fn = tad.ScalarFunction.from_problem(P, ctx)
    _, _, H = fn.eval_with_hessian_proj(P.x0)
    lam, V = np.linalg.eigh(H.toarray())
    A = (H - 0.5 * (lam[0] + lam[1]) * sp.identity(H.shape[0])).tocsr()
    A.sort_indices()
    assert np.array_equal(A.indices, H.indices)
    mu = lam - 0.5 * (lam[0] + lam[1])
    c = np.random.default_rng(5).standard_normal(lam.size)
    rest = float(np.sum(c[1:] ** 2 / mu[1:]))
    b = {}
    for sign in (1.0, -1.0):
        c[0] = np.sqrt(-mu[0] * rest * (0.25 if sign > 0 else 4.0))
        b[sign] = V @ c
        assert sign * (b[sign] @ np.linalg.solve(A.toarray(), b[sign])) > 0.0
    return fn, H, A, b


# the dense preconditioner of small systems, and the two-level one
@pytest.mark.parametrize("n", [6, 16, 33])
def test_indefinite_systems_are_refused(ctx, n):
    """w I + H must be positive definite, whatever the right-hand side: also
    where b . A^-1 b > 0, so that the curvature along A^-1 b is positive."""
    fn, H, A, b = indefinite(ctx, n)
    for sign in (1.0, -1.0):
        with pytest.raises(tad.TadError):
            _, st = fn.solve(b[sign], H=A.data, tol=1e-10)
            if not st.converged:
                raise tad.TadError(0, "not converged")
        # the definite system of the same function still takes the dense inverse
        x, st = fn.solve(b[sign], H=H.data, tol=1e-10)
        assert st.converged and st.coarse_unknowns == (2 * n * n if 2 * n * n <= 2400 else st.coarse_unknowns)
        assert np.linalg.norm(H @ x - b[sign]) <= 1e-9 * np.linalg.norm(b[sign])


def test_inverse_of_an_indefinite_matrix_is_not_kept(ctx):
    """A solve with b = 0 converges at once; the inverse it formed is kept for
    a later solve only when its matrix was positive definite."""
    fn, H, A, b = indefinite(ctx, 16)
    x, st = fn.solve(np.zeros(H.shape[0]), H=A.data)
    assert st.converged and not np.any(x)
    x, st = fn.solve(b[1.0], H=H.data, tol=1e-10, coarse_reuse=1)
    assert st.converged and st.coarse_reused == 0 and st.iters <= 2
    _, st = fn.solve(b[1.0], H=H.data, tol=1e-10, coarse_reuse=1)
    assert st.converged and st.coarse_reused == 1 and st.iters <= 2


def test_destroyed_functions_leave_no_device_memory(ctx):
    """Create, evaluate, solve (with a mask as well), destroy: every
    buffer is given back.  One vector of a round is 4 MB, so a buffer left per
    round shows as 40 MB after ten."""
    import torch
    nh = 500000

    def one():
        pins = configs.Term(configs.E_PENALTY, np.arange(nh, dtype=np.int32)[:, None],
                            np.concatenate([np.zeros((nh, 1)), np.ones((nh, 1))], axis=1))
        P = configs.Problem("pins", 1, nh, [pins], np.ones(nh))
        fn = tad.ScalarFunction.from_problem(P, ctx)
        fn.eval_with_hessian_proj(np.ones(nh))
        x, st = fn.solve(np.ones(nh), coarse_aggregate=0)
        assert st.converged
        free = np.ones(nh, dtype=np.uint8)
        free[1] = 0
        _, st = fn.solve(np.ones(nh), free=free, coarse_aggregate=0)
        assert st.converged
        fn.close()

    one()  # pools of the runtime are filled
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    for _ in range(10):
        one()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    assert before - torch.cuda.mem_get_info()[0] <= 16 << 20


def lagged_size(ctx, P):
    """Coarse unknowns of a Newton loop that keeps its coarse space."""
    fn = tad.ScalarFunction.from_problem(P, ctx)
    return fn.newton_step(P.x0.copy(), tad.newton_default_opts(coarse_refresh=3))["coarse_unknowns"]


def test_solves_between_lagged_newton_steps_share_the_coarse_space(ctx):
    """Automatic solves between the steps neither replace the steps' aggregates
    nor make the next step rebuild what it was going to keep."""
    P = configs.twist_cube(m=16)
    fn = tad.ScalarFunction.from_problem(P, ctx)
    opts = tad.newton_default_opts(coarse_refresh=5)
    x = P.x0.copy()
    n = fn.newton_step(x, opts)["coarse_unknowns"]
    g = np.random.default_rng(0).standard_normal(x.size)
    for _ in range(2):
        _, st = fn.solve(g, tol=1e-8, w_identity=0.0)
        assert st.converged and st.coarse_unknowns == n
        s = fn.newton_step(x, opts)
        assert s["coarse_reused"] == 1 and s["coarse_unknowns"] == n


def test_callers_own_reuse_schedule_gets_the_lagged_size(ctx):
    """A caller that asks for reuse solve by solve gets, from the next rebuild
    on, the size of a space that serves several solves; the solves that only
    keep what is there keep it."""
    P = configs.twist_cube(m=16)
    big = lagged_size(ctx, P)
    fn = tad.ScalarFunction.from_problem(P, ctx)
    _, g, _ = fn.eval_with_hessian_proj(P.x0)
    sizes = []
    for reuse in (0, 1, 1, 0, 1, 0):
        _, st = fn.solve(g, tol=1e-8, coarse_reuse=reuse)
        assert st.converged and st.coarse_reused == reuse
        sizes.append(st.coarse_unknowns)
    assert sizes[0] == sizes[1] == sizes[2] < big
    assert sizes[3] == sizes[4] == sizes[5] == big
