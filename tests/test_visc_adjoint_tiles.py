"""The viscous adjoint takes the grid in tiles of 64 x 8 columns and z segments
whose length depends on the grid: sides one below, at and one above a tile,
grids of one and of several segments, with both cotangents of a step's
stages, against autograd through the FP64 reference.  The ghost-layer kernels
take the ten cells at a line's ends at once from 10 cells on: sides of 9, 10
and 11 as well."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

TOL = 1e-12


@pytest.mark.parametrize("dims", [(64, 8, 5), (63, 7, 6), (65, 9, 7), (66, 17, 40), (10, 9, 11)])
def test_step_vjp_at_tile_edges(dims):
    from hypar_amd.solver import NS3D
    from oracle import torch_ref as T
    from test_adjoint import _hm, _rel, _scheme_case
    w, u0, dt, dx, sch = _scheme_case("components", "rusanov", 1000.0, dims)
    x = T.to_soa(u0).requires_grad_(True)
    lam = torch.randn(x.shape, dtype=x.dtype, generator=torch.Generator().manual_seed(3))
    (ref,) = torch.autograd.grad(T.rk4_step(x, dt, dx, **sch), x, lam)
    print(f"[gpu] viscous adjoint tiles dims={dims}", flush=True)
    s = NS3D.from_workload(w)
    g = _hm(lam)
    s.rk4_vjp(_hm(x), dt, g)
    err = _rel(g.cpu().view_as(ref) - lam, ref - lam)  # without the identity part
    s.close()
    assert err <= TOL, err
