"""A failed allocation is reported to the call that made it, and to no other."""
import pytest

from suli_amd import cases

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
