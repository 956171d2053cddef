"""The multigrid-preconditioned iteration (mixed solves, and FP64 ones by the
relative rule, on grids of 4096 cells or more) against the CPU oracle.

Sizes where its kernels can go wrong: the first size it serves, rows of 16,
32 and 64 lanes with whole and partial last lanes, rows of several segments,
an odd number of rows and planes (half-filled coarse cells), thin grids (coarse
levels one cell wide), every boundary and operator kind.  Mixed solves to a
1e-11 relative residual, FP64 and the oracle to 1e-12; the pressure agrees
within 1e-8 as in the plain CG tests.  The options that name properties of
plain CG keep it.
"""
import numpy as np
import pytest

import oracle
from suli_amd import cases
from tests import helpers

pytestmark = pytest.mark.gpu

PRESSURE_RTOL = 1e-8
PRECISIONS = [("fp64", 1e-12), ("mixed", 1e-11)]


@pytest.fixture(scope="module")
def solver():
    from suli_amd.solver import PressureSolver
    s = PressureSolver(precision="mixed", stop_rule="relative", tol=1e-11, verbose=False)
    yield s
    s.close()


def lid(c):
    c.grid.top_bc = 1
    return c


def ipa(c):
    c.grid.t_press, c.grid.rho_f1 = 2, 1000.0
    return c


def cylinder(nx, ny, nz, seed):
    c = cases.config3(seed=seed, nx=nx, ny=ny, nz=nz)
    cases.make_stretched_compatible(c)
    return c


def two_parts(nx, ny, nz, seed):
    """A solid wall one cell thick cuts the fluid in two."""
    c = cases.random_case(nx, ny, nz, seed)
    c.fields.solid = np.zeros((nx, ny, nz), np.uint8, order="F")
    c.fields.solid[nx // 3, :, :] = 1
    return c


R = cases.random_case
CASES = [
    ("first_size", lambda: R(16, 16, 16, 1)),             # the bottom kernel takes every coarse level
    ("one_coarse_grid", lambda: R(37, 37, 33, 23)),       # 6137 cells on level 1
    ("two_coarse_grids", lambda: R(37, 37, 36, 24)),      # 6498: one more level of its own
    ("rows_of_64", lambda: R(64, 33, 25, 2)),
    ("rows_of_65", lambda: R(65, 40, 21, 3, periodic_x=True)),
    ("rows_of_130", lambda: R(130, 21, 20, 4)),
    ("two_segments", lambda: R(257, 17, 13, 5)),
    ("three_segments_px", lambda: R(515, 11, 10, 6, periodic_x=True, periodic_y=True)),
    ("four_aligned_px", lambda: R(128, 24, 18, 7, periodic_x=True)),
    ("py", lambda: R(52, 40, 25, 8, periodic_y=True)),
    ("thin_z", lambda: R(160, 160, 2, 9)),
    ("thin_y", lambda: R(200, 2, 130, 10)),
    ("thin_x", lambda: R(3, 130, 128, 11, periodic_x=True)),
    ("ratio_1000", lambda: R(64, 64, 40, 22, ratio=1000.0, surface=0.45)),
    ("ratio_1", lambda: R(48, 41, 31, 12, ratio=1.0)),
    ("lid", lambda: lid(R(50, 40, 33, 13))),
    ("ipa", lambda: ipa(R(63, 31, 29, 14))),
    ("ibm_rhs", lambda: R(56, 48, 24, 15, ibm=True)),
    ("cylinder", lambda: cylinder(72, 40, 24, 16)),
    ("flat_cells", lambda: R(64, 48, 20, 17, dx=5e-3)),
    ("last_brick", lambda: R(64, 64, 32, 25, periodic_x=True)),      # 131072 cells: up to here bricks
    ("brick_edges", lambda: R(17, 9, 41, 26, periodic_y=True)),
    ("first_march", lambda: lid(R(61, 43, 50, 27))),                 # 131150
    ("march_two_segments", lambda: R(257, 27, 19, 28)),
    ("march_three_segments_px", lambda: R(515, 17, 15, 29, periodic_x=True, periodic_y=True)),
    ("march_four_aligned_px", lambda: R(128, 33, 32, 30, periodic_x=True)),
    ("march_cylinder", lambda: cylinder(96, 44, 33, 32)),
]


@pytest.mark.parametrize("precision,tol", PRECISIONS, ids=["fp64", "mixed"])
@pytest.mark.parametrize("name,make", CASES, ids=[n for n, _ in CASES])
def test_vs_oracle(solver, name, make, precision, tol):
    c = make()
    if name == "flat_cells":
        c.grid.dx = c.grid.dy = 4e-2     # 8 times as wide as high
    print(f"multigrid {name} {precision}", flush=True)
    p_or, _, rc = oracle.graddin(c.grid, c.fields, stop_rule=oracle.STOP_RELATIVE, tol=1e-12, project_null=True)
    assert rc == 0
    solver.configure(precision=precision, stop_rule="relative", tol=tol, verbose=False)
    df = solver.upload(c.grid, c.fields)
    try:
        st = solver.graddin_dev(c.grid, df)
        p = df.download("prd1")
    finally:
        df.free()
    print(f"  {st.iters} iterations", flush=True)
    assert st.status == 0 and st.rel_true <= (tol if precision == "mixed" else 10 * tol), st.as_dict()
    # far fewer than plain CG's several hundred: the iteration itself ran
    assert st.iters < 150 or name in ("thin_z", "thin_y", "thin_x", "flat_cells"), st.iters
    assert helpers.rel_diff(p, p_or, helpers.face_mask(p.shape)) <= PRESSURE_RTOL


@pytest.mark.parametrize("precision,tol", PRECISIONS, ids=["fp64", "mixed"])
@pytest.mark.parametrize("shape", [(40, 37, 36), (130, 40, 11)])
def test_suli_it_vs_oracle(solver, shape, precision, tol):
    g, f = cases.it_case(*shape, seed=21)
    print(f"multigrid suli-it {shape} {precision}", flush=True)
    f_or = f.copy()
    p_or, _, rc = oracle.it_graddin(g, f_or, stop_rule=oracle.STOP_RELATIVE, tol=1e-12)
    assert rc == 0
    solver.configure(precision=precision, stop_rule="relative", tol=tol, verbose=False)
    st = solver.it_graddin(g, f)
    assert st.status == 0 and st.iters < 150, st.as_dict()
    assert helpers.rel_diff(f.prd1, p_or, helpers.face_mask(f.prd1.shape)) <= PRESSURE_RTOL


@pytest.mark.parametrize("precision,tol", PRECISIONS, ids=["fp64", "mixed"])
def test_two_parts_keep_their_gauges(solver, precision, tol):
    """Fluid cut in two by a solid wall: each part's pressure keeps the mean
    that plain CG (the oracle) gives it."""
    c = two_parts(48, 40, 30, 31)
    print(f"multigrid two parts {precision}", flush=True)
    p_or, _, rc = oracle.graddin(c.grid, c.fields, stop_rule=oracle.STOP_RELATIVE, tol=1e-12, project_null=True)
    assert rc == 0
    solver.configure(precision=precision, stop_rule="relative", tol=tol, verbose=False)
    df = solver.upload(c.grid, c.fields)
    try:
        st = solver.graddin_dev(c.grid, df)
        p = df.download("prd1")
    finally:
        df.free()
    assert st.status == 0, st.as_dict()
    assert helpers.rel_diff(p, p_or, helpers.face_mask(p.shape)) <= PRESSURE_RTOL


def test_options_that_keep_plain_cg(solver):
    """A small iteration cap returns plain CG's iterate, also at this size;
    keep_null and stored_residual take plain CG's iteration counts, and so
    does FP64 by the reference rule."""
    c = cases.random_case(48, 40, 30, 41)
    print("multigrid options", flush=True)

    def run(**kw):
        solver.configure(stop_rule="relative", verbose=False, **kw)
        df = solver.upload(c.grid, c.fields)
        try:
            st = solver.graddin_dev(c.grid, df)
            return df.download("prd1"), st
        finally:
            df.free()

    p64, _ = run(precision="fp64", tol=1e-14, max_iter=37)
    p32, st = run(precision="mixed", tol=1e-14, max_iter=37)
    assert st.status == 1 and st.iters == 37
    assert helpers.rel_diff(p32, p64, helpers.face_mask(p64.shape)) <= 1e-5
    _, st64 = run(precision="fp64", tol=1e-8, keep_null=True)
    assert st64.iters > 150
    for kw in (dict(keep_null=True), dict(stored_residual=True)):
        _, st = run(precision="mixed", tol=1e-8, **kw)
        assert st.status == 0 and st.iters >= 0.5 * st64.iters, (kw, st.iters, st64.iters)
    f = cases.scale_velocity(c.fields, 2.0 ** 14)
    _, st_or, _ = oracle.graddin(c.grid, f, project_null=True)
    solver.configure(precision="fp64", stop_rule="reference", verbose=False)
    st = solver.graddin(c.grid, f)
    assert abs(st.iters - st_or.iters) <= 1, (st.iters, st_or.iters)


@pytest.mark.parametrize("precision,tol", PRECISIONS, ids=["fp64", "mixed"])
def test_batch_and_server_equal_alone(precision, tol):
    """Problems of both iterations in one batch, and through the server: each
    bit for bit as alone."""
    from suli_amd.server import PressureServer
    from suli_amd.solver import PressureSolver
    cs = [R(40, 24, 16, 51), R(66, 40, 30, 52), cylinder(72, 40, 24, 53), ipa(R(61, 33, 31, 54)),
          R(130, 40, 33, 55, periodic_x=True), R(24, 20, 16, 56)]
    with PressureSolver(precision=precision, stop_rule="relative", tol=tol, verbose=False) as s:
        alone = []
        for c in cs:
            df = s.upload(c.grid, c.fields)
            st = s.graddin_dev(c.grid, df)
            assert st.status == 0
            alone.append((df.download("prd1"), st.iters))
            df.free()
        dfs = [s.upload(c.grid, c.fields) for c in cs]
        sts = s.graddin_batch_dev([(c.grid, df) for c, df in zip(cs, dfs)])
        for i, (df, st) in enumerate(zip(dfs, sts)):
            assert st.iters == alone[i][1], i
            np.testing.assert_array_equal(df.download("prd1"), alone[i][0])
            df.free()
    with PressureServer(precision=precision, stop_rule="relative", tol=tol) as srv:
        todo = [i for i, c in enumerate(cs) if c.fields.solid is None]
        fields = [cs[i].fields.copy() for i in todo]
        tickets = [srv.submit(cs[i].grid, f) for i, f in zip(todo, fields)]
        for i, f, t in zip(todo, fields, tickets):
            st = srv.wait(t)
            assert st.status == 0 and st.iters == alone[i][1], i
            np.testing.assert_array_equal(f.prd1, alone[i][0])


@pytest.mark.parametrize("precision,tol", PRECISIONS, ids=["fp64", "mixed"])
@pytest.mark.parametrize("shape", [(72, 50, 40), (110, 79, 72)])
def test_noalloc_equals_alone(solver, shape, precision, tol):
    """Small, and near the largest state the call accepts."""
    c = R(*shape, 61)
    print(f"multigrid noalloc {shape} {precision}", flush=True)
    solver.configure(precision=precision, stop_rule="relative", tol=tol, verbose=False)
    out = []
    for noalloc in (False, True):
        df = solver.upload(c.grid, c.fields)
        try:
            st = solver.graddin_noalloc_dev(c.grid, df) if noalloc else solver.graddin_dev(c.grid, df)
            out.append((df.download("prd1"), st.iters, st.refreshes))
        finally:
            df.free()
    assert out[0][1:] == out[1][1:]
    assert out[0][1] < 150
    np.testing.assert_array_equal(out[0][0], out[1][0])


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("shape", [(40, 32, 24), (70, 60, 40)], ids=["bricks", "marched"])
def test_step_is_timed(solver, shape, precision):
    """opts.timing measures the step however few of them a solve takes."""
    c = R(*shape, 71)
    print(f"multigrid timing {shape} {precision}", flush=True)
    solver.configure(precision=precision, stop_rule="relative", tol=1e-8, verbose=False, timing=True)
    df = solver.upload(c.grid, c.fields)
    try:
        for _ in range(2):   # windows at both alignments of the step counter
            df.zero("prd1")
            st = solver.graddin_dev(c.grid, df)
            assert st.spmv_timed > 0 and 0.0 < st.spmv_ms < st.solve_ms, st.as_dict()
    finally:
        df.free()


def masked(name):
    """(case, number of connected fluid parts)"""
    nx, ny, nz = 70, 26, 20
    px = name.endswith("_px")
    c = cases.random_case(nx, ny, nz, 81, periodic_x=px)
    m = np.zeros((nx, ny, nz), np.uint8, order="F")
    base = name.removesuffix("_px")
    if base == "wall_x_at_64":
        m[64] = 1
    elif base == "wall_y":
        m[:, 12] = 1
    elif base == "wall_z":
        m[:, :, 9] = 1
    elif base == "gap_in_x":       # two runs of a row, joined by its last rows
        m[31, :ny - 4] = 1
    elif base == "gap_in_y":       # two stretches, joined in the last columns
        m[:nx - 5, 12] = 1
    elif base == "gap_in_z":
        m[:, :ny - 4, 9] = 1
    elif base == "blocks":
        m[10:20, 5:15, 3:12] = m[40:66, 10:22, 6:20] = 1
    c.fields.solid = m
    parts = 2 if base in ("wall_y", "wall_z") or name == "wall_x_at_64" else 1
    return c, parts


@pytest.mark.parametrize("name", ["wall_x_at_64", "wall_x_at_64_px", "wall_y", "wall_z", "gap_in_x", "gap_in_x_px",
                                  "gap_in_y", "gap_in_z", "blocks", "blocks_px"])
def test_parts_of_a_mask(solver, name):
    """Fluid in one part is solved by the multigrid iteration, in several by
    plain CG (hundreds of iterations); either agrees with the oracle.  (In FP64:
    plain CG's mixed iteration lets each part's mean drift with FP32's rounding,
    3e-7 of the pressure over wall_z.)"""
    c, parts = masked(name)
    print(f"multigrid mask {name}", flush=True)
    p_or, _, rc = oracle.graddin(c.grid, c.fields, stop_rule=oracle.STOP_RELATIVE, tol=1e-12, project_null=True)
    assert rc == 0
    solver.configure(precision="fp64", stop_rule="relative", tol=1e-12, verbose=False)
    df = solver.upload(c.grid, c.fields)
    try:
        st = solver.graddin_dev(c.grid, df)
        p = df.download("prd1")
    finally:
        df.free()
    assert st.status == 0 and (st.iters < 60) == (parts == 1), (name, st.as_dict())
    assert helpers.rel_diff(p, p_or, helpers.face_mask(p.shape)) <= PRESSURE_RTOL
