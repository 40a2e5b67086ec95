"""FP64 tets near and at rest: the projection through the clamped eigenvalues
against the oracle's full eigensolve where those eigenvalues are close to each
other and to the clamp level."""
import numpy as np
import pytest

import tinyad_amd as tad
from tinyad_amd import configs

pytestmark = pytest.mark.gpu


# displacement noise in mesh widths, uniform and one-axis compression
@pytest.mark.parametrize("state", [("noise", 10.0 ** -k) for k in (13, 12, 11, 10, 9, 8, 6, 5)]
                         + [("compressed", a) for a in (1e-9, 1e-5, 1e-4)]
                         + [("flattened", a) for a in (1e-7, 1e-4, 0.2)], ids=lambda s: f"{s[0]}_{s[1]:g}")
def test_tets_near_rest(ctx, state):
    """Each side's element error is below 30 eps |H_e| (7e-15), a block sums at
    most 24 elements: 24 * 2 * 7e-15 < 4e-13."""
    import oracle
    P = configs.twist_cube(m=4)
    rest = P.info["rest"].reshape(-1, 3)
    kind, a = state
    if kind == "noise":
        x = rest + a * P.info["h"] * np.random.default_rng(3).standard_normal(rest.shape)
    else:
        x = rest * ((1.0 - a) if kind == "compressed" else np.array([1.0, 1.0, 1.0 - a]))
    x = np.ascontiguousarray(x).reshape(-1)
    fg = tad.ScalarFunction.from_problem(P, ctx)
    fo = oracle.Function.from_problem(P)
    for eps in (1e-9, 0.0, -1.0):
        ref = fo.eval_with_hessian_proj(x, eps)[2].toarray()
        for shape in [(0, 0, 0), (256, 1, 0)]:
            fg.set_launch_shape(0, *shape)
            H = fg.eval_with_hessian_proj(x, eps)[2].toarray()
            assert np.abs(H - ref).max() <= 4e-13 * np.abs(ref).max(), (eps, shape)


@pytest.mark.parametrize("eps", [0.02, 0.1, 0.3, 1.0, 30.0])
@pytest.mark.parametrize("state", ["rest", "noise", "twisted"])
def test_levels_that_clamp_most_eigenvalues(ctx, state, eps):
    """Four to all nine of an element's eigenvalues below the level (they are
    0.1 .. 3 here), against the oracle; the error bound of test_tets_near_rest,
    relative to the level where that is larger."""
    import oracle
    P = configs.twist_cube(m=3)
    rest = P.info["rest"].reshape(-1, 3)
    x = rest.copy()
    if state == "noise":
        x = x + 0.02 * P.info["h"] * np.random.default_rng(3).standard_normal(rest.shape)
    elif state == "twisted":
        th = np.radians(50.0) * rest[:, 2]
        px, py = rest[:, 0] - 0.5, rest[:, 1] - 0.5
        x = np.stack([0.5 + np.cos(th) * px - np.sin(th) * py, 0.5 + np.sin(th) * px + np.cos(th) * py, rest[:, 2]], axis=1)
    x = np.ascontiguousarray(x).reshape(-1)
    fg = tad.ScalarFunction.from_problem(P, ctx)
    fo = oracle.Function.from_problem(P)
    ref = fo.eval_with_hessian_proj(x, eps)[2].toarray()
    for shape in [(0, 0, 0), (256, 1, 0)]:
        fg.set_launch_shape(0, *shape)
        H = fg.eval_with_hessian_proj(x, eps)[2].toarray()
        assert np.abs(H - ref).max() <= 4e-13 * max(np.abs(ref).max(), eps), shape
