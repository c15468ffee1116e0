"""The right-hand side's adjoint is linear in its cotangent: a cotangent times
2^100 (1.3e30) gives 2^100 times the result, to the bit, as long as nothing
leaves double's range.  With the smallest epsilons in use, and in a uniform
region, where the smoothness indicators are epsilon alone, the derivative of
the weights divides by up to its ninth power."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("interp,upwind", [("components", "rusanov"), ("components", "roe"), ("characteristic", "roe")])
@pytest.mark.parametrize("weno,eps", [("js", 1e-40), ("mapped", 1e-40), ("borges", 1e-32), ("yc", 1e-32)])
def test_vjp_scales_with_its_cotangent(interp, upwind, weno, eps):
    from hypar_amd.solver import NS3D
    dims = (14, 12, 13)
    n = dims[0] * dims[1] * dims[2]
    u = torch.tensor([1.0, 0.25, -0.125, 0.5, 2.5], dtype=torch.float64).repeat_interleave(n).view(5, *dims[::-1])
    u[0, 2:4, 5, 6] *= 1.125  # a bump; the rest is uniform
    lam = torch.randn(5 * n, dtype=torch.float64, generator=torch.Generator().manual_seed(5)).cuda()
    print(f"[gpu] scale of the adjoint, {interp}/{upwind}/{weno} eps={eps}", flush=True)
    s = NS3D(dims, interp, upwind, eps=eps, weno_type=weno)
    u = u.reshape(-1).cuda()
    a = s.rhs_vjp(u, lam)
    b = s.rhs_vjp(u, lam * 2.0 ** 100)
    s.close()
    assert bool(torch.isfinite(a).all())
    assert torch.equal(b, a * 2.0 ** 100)
