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
