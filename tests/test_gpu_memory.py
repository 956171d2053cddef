"""Allocations that fail, and device memory that holds plain CG's state only.
(The engine's own shortages: test_engine_host.py.)"""
import pytest

from suli_amd import cases
from tests import helpers

pytestmark = pytest.mark.gpu


def test_failed_allocation_does_not_fail_the_next_solve():
    from suli_amd.solver import PressureSolver
    c = cases.random_case(20, 18, 16, 3)
    print("failed allocation", flush=True)
    with PressureSolver(stop_rule="relative", tol=1e-8, verbose=False) as s:
        df = s.upload(c.grid, c.fields)
        assert s.lib.suli_ps_dev_alloc(s.ctx, 1 << 46) is None   # 64 TiB
        st = s.graddin_dev(c.grid, df)
        assert st.status == 0
        s.posdin_dev(c.grid, df)
        df.free()


def test_server_budget_chooses_the_iteration():
    """An FP64 request of 40^3 cells: 2.9 MB of fields, 8 MiB of state, or 6 MiB
    for plain CG."""
    from suli_amd.server import PressureServer
    c = cases.random_case(40, 40, 40, 5)
    print("server budget", flush=True)
    out = []
    for budget in (12 << 20, 10 << 20):
        with PressureServer(precision="fp64", stop_rule="relative", tol=1e-12, hbm_budget=budget) as srv:
            f = c.fields.copy()
            st = srv.wait(srv.submit(c.grid, f))
            assert st.status == 0
            out.append((f.prd1, st.iters))
    assert out[0][1] < 40 and out[1][1] > 150, (out[0][1], out[1][1])
    assert helpers.rel_diff(out[1][0], out[0][0], helpers.face_mask(out[0][0].shape)) <= 1e-8
