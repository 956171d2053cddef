"""The column sweeps pressh and posdin_hydro at the edges of their chunks of 16
and 32 planes and of their 64 columns: bit for bit the C oracle's, whose
operation order they keep."""
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
@pytest.mark.parametrize("nx,ny,nz", [(8, 8, 16), (9, 7, 17), (16, 8, 31), (13, 5, 32), (11, 6, 33), (7, 9, 34),
                                      (62, 3, 64), (5, 13, 65), (17, 3, 100)])
def test_column_chunks(solver, nx, ny, nz, stretched):
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
