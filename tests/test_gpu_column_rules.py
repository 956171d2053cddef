"""The column sweeps pressh and posdin_hydro on both sides of the lines between a
lane per column and a workgroup per chunk of planes (ps_setup.hip,
pressh_in_chunks and hydro_w_in_chunks): bit for bit the C oracle's, whose operation
order both keep."""
import numpy as np
import pytest

import oracle
from suli_amd import cases

pytestmark = pytest.mark.gpu

GZ = 9.80665


@pytest.fixture(scope="module")
def solver():
    from suli_amd.solver import PressureSolver
    s = PressureSolver(verbose=False)
    yield s
    s.close()


@pytest.mark.parametrize("stretched", [False, True], ids=["uniform", "stretched"])
@pytest.mark.parametrize("nx,ny,nz", [
    (9, 7, 2), (9, 7, 3), (31, 17, 7), (31, 17, 8),      # pressh: 8 planes
    (128, 128, 8), (127, 129, 8), (128, 129, 8), (128, 129, 9),   # w: 16384 columns, 8 planes
    (256, 128, 15), (256, 128, 16),                      # pressh: a plane for 2048 columns
    (320, 256, 41), (321, 256, 41),                      # pressh: 81920 columns
    (640, 512, 9), (640, 512, 10),                       # w: a plane for 32768 columns
    (300, 257, 1 + 1)])
def test_column_rules(solver, nx, ny, nz, stretched):
    c = cases.random_case(nx, ny, nz, seed=nz, stretched=stretched, surface=0.55)
    c.grid.t_press = 0
    hs = np.clip((c.fields.rho - 1.2) / (1000.0 - 1.2), 0.0, 1.0)
    hs[hs < 1e-3] = 0.0
    c.fields.hs = np.asfortranarray(hs)
    print(f"columns {nx}x{ny}x{nz} {stretched}", flush=True)
    p = oracle.pressh(c.grid, c.fields.rho, GZ, c.fields.prd1)
    f = c.fields.copy()
    f.prd1[...] = p
    u, v, w, _ = oracle.posdin_hydro(c.grid, f, f.hs, p)
    df = solver.upload(c.grid, c.fields)
    try:
        solver.pressh_dev(c.grid, df, GZ)
        np.testing.assert_array_equal(df.download("prd1"), p)
        solver.posdin_hydro_dev(c.grid, df)
        for name, want in (("u", u), ("v", v), ("w", w)):
            np.testing.assert_array_equal(df.download(name), want)
    finally:
        df.free()
