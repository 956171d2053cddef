"""The multigrid-preconditioned iteration on problems whose values leave FP32's
range.  Every step of the FP64 solve is homogeneous, so inputs scaled by a power
of two give the same bits, scaled.
"""
import numpy as np
import pytest

from suli_amd import cases

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def solver():
    from suli_amd.solver import PressureSolver
    s = PressureSolver(verbose=False)
    yield s
    s.close()


def solve(s, c, fields):
    df = s.upload(c.grid, fields)
    try:
        st = s.graddin_dev(c.grid, df)
        return df.download("prd1"), st
    finally:
        df.free()


@pytest.mark.parametrize("shape", [(40, 32, 24), (70, 60, 40)], ids=["bricks", "marched"])
def test_fp64_residuals_beyond_fp32(solver, shape):
    """Right-hand sides of 1e-120 to 1e120: FP32 holds 1e-45 to 3e38."""
    c = cases.random_case(*shape, 91)
    solver.configure(precision="fp64", stop_rule="relative", tol=1e-12, verbose=False)
    print(f"multigrid range {shape}", flush=True)
    p0, st0 = solve(solver, c, c.fields)
    assert st0.status == 0 and st0.iters < 40, st0.as_dict()
    for e in (-400, -150, -100, 100, 140, 400):
        p, st = solve(solver, c, cases.scale_velocity(c.fields, 2.0 ** e))
        assert st.status == 0 and st.iters == st0.iters, (e, st.as_dict())
        np.testing.assert_array_equal(p, p0 * 2.0 ** e)
