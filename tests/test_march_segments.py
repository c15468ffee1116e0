"""The y and z passes cut the lines of small grids into march segments (from
8 cells a line on).  Lines of every remainder of the 4-row march step, from
the longest line that stays whole to lines of several segments, over one and
several 64-column groups: the right-hand side and one SSPRK3 step (whose z
pass updates the state as well) against the oracle."""
import dataclasses

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

TOL = 1e-12


@pytest.mark.parametrize("dims", [(6, 7, 8), (9, 10, 11), (66, 12, 13), (5, 47, 23), (64, 31, 16)])
@pytest.mark.parametrize("interp,upwind,Re", [("characteristic", "roe", 1600.0), ("components", "rusanov", -1.0)])
def test_segments_match_oracle(dims, interp, upwind, Re):
    from hypar_amd import decks
    from hypar_amd.solver import NS3D
    from oracle.oracle import Oracle
    w = dataclasses.replace(decks.config1(16, 1), dims=dims, interp=interp, upwind=upwind, Re=Re, dt=None)
    print(f"[gpu] march segments {interp}/{upwind}/Re={Re} dims={dims}", flush=True)
    u0, dt = decks.prepare(w)
    o = Oracle.for_workload(w)
    s = NS3D.from_workload(w)
    u = s.to_device(u0)
    err = decks.rel_l2(s.to_host(s.rhs(u)), o.rhs(u0))
    assert err <= TOL, err
    s.ssprk3(u, dt, 1)
    err = decks.rel_l2(s.to_host(u), o.step(u0, dt, 1, "ssprk3"))
    s.close()
    assert err <= TOL, err
