"""A solver used for single step adjoints holds the three stage states and the
three scratch states these need, and no more: six states of 10 MiB at 64^3,
each a whole number of the driver's 2 MiB pages."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def test_step_vjp_holds_six_states():
    from hypar_amd.solver import NS3D
    n = 64
    state = 5 * n ** 3 * 8

    def solver():
        return NS3D((n, n, n))

    u = torch.tensor([1.0, 0.1, 0.0, 0.0, 2.5], dtype=torch.float64, device="cuda").repeat_interleave(n ** 3)
    lam = torch.ones_like(u)
    first = solver()  # loads the kernels
    first.rk4_vjp(u, 1e-3, lam)
    s = solver()
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    s.rk4_vjp(u, 1e-3, lam)
    torch.cuda.synchronize()
    held = free - torch.cuda.mem_get_info()[0]
    print(f"[gpu] step adjoint holds {held / state:.2f} states", flush=True)
    s.close()
    first.close()
    assert held <= 6 * state + (4 << 20), held / state
