"""The Hessian assembly a function reports is the one that runs."""
import numpy as np
import pytest

import tinyad_amd as tad
from tinyad_amd import configs

pytestmark = pytest.mark.gpu


def launches(ctx, fn, x):
    """Launches of an assembly of its own in one evaluation (tiles have none)."""
    ctx.enable_timing(True)
    ctx.reset_stats()
    fn.eval_with_hessian_proj(x)
    n = ctx.kernel_stats("assemble_hessian")[0]
    ctx.enable_timing(False)
    return n


# 3D from 200,000 blocks on, where the automatic choice is not the tiles, and below
@pytest.mark.parametrize("m", [6, 24])
def test_reported_shape_is_the_one_that_runs(ctx, m):
    P = configs.twist_cube(m=m)
    fn = tad.ScalarFunction.from_problem(P, ctx)
    fn.pattern()
    auto = fn.assembly_shape
    assert auto == (0 if m == 6 else 2)
    assert launches(ctx, fn, P.x0) == (0 if auto == 0 else 1)
    ref = fn.eval_with_hessian_proj(P.x0)
    for shape in range(4):
        fn.assembly_shape = shape
        assert fn.assembly_shape == shape
        assert launches(ctx, fn, P.x0) == (0 if shape == 0 else 1), shape
        f, g, H = fn.eval_with_hessian_proj(P.x0)
        assert f == ref[0] and np.array_equal(g, ref[1]) and np.array_equal(H.data, ref[2].data)
    fn.autotune(P.x0)
    assert launches(ctx, fn, P.x0) == (0 if fn.assembly_shape == 0 else 1)
