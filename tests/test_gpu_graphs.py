"""Replayed graphs of plain CG steps against direct launches, on problems that take
the plain iteration (multigrid steps are launched directly)."""
import numpy as np
import pytest

from suli_amd import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("mixed", 1e-11)], ids=["fp64", "mixed"])
def test_replay_equals_direct_launches(precision, tol):
    from suli_amd.solver import PressureSolver
    # keep_null: plain CG at any size; and below 4096 cells
    runs = [(dict(keep_null=True), [cases.random_case(40, 24, 16, 61), cases.random_case(33, 20, 18, 62)]),
            (dict(), [cases.random_case(17, 15, 14, 63), cases.random_case(20, 16, 12, 64, periodic_x=True)])]
    with PressureSolver(verbose=False) as s:
        for opts, cs in runs:
            want = None
            for graphs in (False, True, True, True):   # replays with the program's own work between
                print(f"graphs {graphs} {precision} {opts}", flush=True)
                s.configure(precision=precision, stop_rule="relative", tol=tol, verbose=False, graphs=graphs, **opts)
                dfs = [s.upload(c.grid, c.fields) for c in cs]
                sts = s.graddin_batch_dev([(c.grid, df) for c, df in zip(cs, dfs)])
                got = [(df.download("prd1"), st.iters) for df, st in zip(dfs, sts)]
                for df in dfs:
                    df.free()
                assert all(st.status == 0 and (st.graph_replays > 0) == graphs for st in sts)
                want = want or got
                for (p, it), (p0, it0) in zip(got, want):
                    assert it == it0
                    np.testing.assert_array_equal(p, p0)
