"""A cell without mass: the flux kernels take its velocity as zero, so that the
flux and its neighbours' right-hand side stay finite.  The adjoint may be
without a value only where the forward's upwinding is: at the two interfaces
of the empty cell, whose stencils reach three cells along the three lines
through it.  Everywhere else it is finite and is the derivative of the
oracle's right-hand side.

The difference quotient's step h = 1e-7 is 1e-4 of the smallest scale on which
the weights change (sqrt(eps) = 1e-3): error 1e-8, rounding 1e-16/h = 1e-9;
1e-5 leaves the third derivative a factor of a thousand."""
import dataclasses

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

H = 1e-7


@pytest.mark.parametrize("interp,upwind", [("components", "roe"), ("components", "rusanov"),
                                           ("characteristic", "roe"), ("characteristic", "rusanov")])
def test_adjoint_around_an_empty_cell(interp, upwind):
    from hypar_amd import decks
    from hypar_amd.solver import NS3D
    from oracle.oracle import Oracle
    dims, at = (16, 17, 18), (9, 8, 7)  # at: (z, y, x)
    w = dataclasses.replace(decks.config1(16, 1), dims=dims, interp=interp, upwind=upwind, Re=-1.0, dt=None)
    u = decks.initial_state(w)
    u[at] = 0.0
    near = np.zeros(u.shape[:3], dtype=bool)
    for ax in range(3):
        for k in range(-3, 4):
            c = list(at)
            c[ax] = (c[ax] + k) % u.shape[ax]
            near[tuple(c)] = True
    rng = np.random.default_rng(17)
    d, lam = (rng.normal(size=u.shape) * ~near[..., None] for _ in range(2))
    o = Oracle.for_workload(w)
    dr = (o.rhs(u + H * d) - o.rhs(u - H * d)) / (2 * H)
    ref = float((lam * dr)[~near].sum())
    print(f"[gpu] adjoint around an empty cell, {interp}/{upwind}", flush=True)
    s = NS3D.from_workload(w)
    g = s.to_host(s.rhs_vjp(s.to_device(u), s.to_device(lam)))
    s.close()
    assert np.isfinite(g[~near]).all(), int((~np.isfinite(g[~near])).sum())
    got = float((g * d)[~near].sum())
    assert abs(got - ref) <= 1e-5 * abs(ref), (got, ref)
