"""The multigrid-preconditioned iteration on problems whose values leave FP32's
range.  Every step of the FP64 solve is homogeneous, so inputs scaled by a power
of two give the same bits, scaled.
"""
import numpy as np
import pytest

import oracle
from suli_amd import cases
from tests import helpers

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


def breaking(shape, seed):
    """A density so small that the operator's diagonal is beyond FP32 (2^280): the
    V-cycle's weights are infinite and the iteration breaks down in its first step.
    The velocity is scaled so that the scaled system's vectors are the plain case's,
    and the pressure is 2^-140 times its."""
    c = cases.random_case(*shape, seed)
    fields = cases.scale_velocity(c.fields, 2.0 ** 140)
    fields.rho = np.asfortranarray(fields.rho * 2.0 ** -280)
    c.plain, c.fields = c.fields, fields
    return c


BREAKING = [(40, 32, 24), (70, 60, 40)]   # bricks, marched


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("mixed", 1e-11)], ids=["fp64", "mixed"])
def test_breakdown_is_solved_again_by_plain_cg(solver, precision, tol):
    """Alone, without allocation, in a batch beside problems that do not break
    down, and through the server: plain CG's solution, and every neighbour as it
    is alone.  (The second set-up happens with another chunk of steps in flight.)"""
    from suli_amd.server import PressureServer
    cs = [breaking(BREAKING[0], 92), cases.random_case(48, 40, 36, 93), breaking(BREAKING[1], 94),
          cases.random_case(66, 50, 44, 95), cases.random_case(20, 16, 12, 96)]
    print(f"multigrid breakdown {precision}", flush=True)
    solver.configure(precision=precision, stop_rule="relative", tol=tol, verbose=False)
    alone = [solve(solver, c, c.fields) for c in cs]
    for c, (p, st) in zip(cs, alone):
        assert st.status == 0, st.as_dict()
        if hasattr(c, "plain"):
            p_or, _, rc = oracle.graddin(c.grid, c.plain, stop_rule=oracle.STOP_RELATIVE, tol=1e-12,
                                         project_null=True)
            assert rc == 0 and st.iters > 150   # plain CG's count
            assert helpers.rel_diff(p * 2.0 ** 140, p_or, helpers.face_mask(p.shape)) <= 1e-8
    df = solver.upload(cs[0].grid, cs[0].fields)
    st = solver.graddin_noalloc_dev(cs[0].grid, df)
    assert st.iters == alone[0][1].iters
    np.testing.assert_array_equal(df.download("prd1"), alone[0][0])
    df.free()
    for _ in range(2):   # the slots serve again
        dfs = [solver.upload(c.grid, c.fields) for c in cs]
        sts = solver.graddin_batch_dev([(c.grid, df) for c, df in zip(cs, dfs)])
        for i, (df, st) in enumerate(zip(dfs, sts)):
            assert st.status == 0 and st.iters == alone[i][1].iters, (i, st.as_dict())
            np.testing.assert_array_equal(df.download("prd1"), alone[i][0])
            df.free()
    with PressureServer(precision=precision, stop_rule="relative", tol=tol) as srv:
        fields = [c.fields.copy() for c in cs]
        tickets = [srv.submit(c.grid, f) for c, f in zip(cs, fields)]
        for i, (f, t) in enumerate(zip(fields, tickets)):
            st = srv.wait(t)
            assert st.status == 0 and st.iters == alone[i][1].iters, i
            np.testing.assert_array_equal(f.prd1, alone[i][0])


def test_stalled_replacements_end_by_plain_cg(solver):
    """A tolerance below what FP64 resolves: after three replacements that do not
    halve the residual the solve is plain CG's, which runs to its cap."""
    c = cases.random_case(36, 30, 22, 97)
    print("multigrid stalls", flush=True)
    solver.configure(precision="mixed", stop_rule="relative", tol=1e-19, max_iter=300, verbose=False)
    p, st = solve(solver, c, c.fields)
    assert st.status == 1 and st.iters == 300, st.as_dict()
    solver.configure(precision="fp64", stop_rule="relative", tol=1e-12, verbose=False)
    p64, st64 = solve(solver, c, c.fields)
    assert st64.status == 0
    # 300 plain iterations: a residual of about 1e-8
    assert st.rel_true < 1e-6 and helpers.rel_diff(p, p64, helpers.face_mask(p.shape)) < 1e-4


def flat(shape, ax, ay, seed):
    c = cases.random_case(*shape, seed)
    c.grid.dx *= ax
    c.grid.dy *= ay
    return c


# (grid, dx / dz, dy / dz, most iterations to 1e-12).  On cells of unequal sides the
# point smoother and the 2x2x2 coarsening take more: 40x32x24 took 24, 73, 143 and 212
# for 2, 4, 8 and 16 (plain CG 560, 1024, 2184, 10000 mixed), 77, 132 and 231 for
# 1/4, 1/8 and 1/16 (656, 1024, 2584).
FLAT = [((40, 32, 24), a, a, most) for a, most in
        ((1, 20), (2, 35), (4, 100), (8, 190), (16, 300), (1 / 4, 110), (1 / 8, 180), (1 / 16, 320))]
FLAT += [((64, 48, 40), 4, 4, 150), ((64, 48, 40), 1 / 4, 1 / 4, 150)]      # marched tiles
# thin grids of cubes
FLAT += [((160, 160, 2), 1, 1, 40), ((200, 2, 130), 1, 1, 40), ((3, 130, 128), 1, 1, 40)]


@pytest.mark.parametrize("shape,ax,ay,most", FLAT)
def test_iterations_on_flat_and_thin_cells(solver, shape, ax, ay, most):
    c = flat(shape, ax, ay, 98)
    for precision, tol in (("fp64", 1e-12), ("mixed", 1e-11)):
        print(f"multigrid flat {shape} {ax} {ay} {precision}", flush=True)
        solver.configure(precision=precision, stop_rule="relative", tol=tol, verbose=False)
        _, st = solve(solver, c, c.fields)
        assert st.status == 0 and st.iters <= most, (precision, st.as_dict())
        solver.configure(precision=precision, stop_rule="relative", tol=tol, verbose=False, keep_null=True)
        _, plain = solve(solver, c, c.fields)
        assert st.iters < 0.5 * plain.iters, (st.iters, plain.iters)
