"""The viscous term of a uniform flow is zero.  With a state of few bits every
product and sum of the derivative stencils, whose weights are whole numbers
over 12, is exact, in the interior and in the ghost layers of a line's ends,
if the weights are applied before the scale: the term is zero to the bit, on
grids of one and of several tiles and segments."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(5, 5, 5), (9, 10, 11), (70, 20, 40)])
def test_viscous_term_of_uniform_flow(dims):
    from hypar_amd.solver import NS3D
    n = dims[0] * dims[1] * dims[2]
    # gamma = 3/2: T = gamma P / rho has 12 bits
    u = torch.tensor([1.0, 0.25, -0.5, 0.125, 2.0], dtype=torch.float64, device="cuda").repeat_interleave(n)
    print(f"[gpu] viscous term of a uniform flow, dims={dims}", flush=True)
    s = NS3D(dims, Re=1000.0, Minf=0.1, gamma=1.5)
    par = s.parabolic(u)
    s.close()
    assert int(torch.count_nonzero(par)) == 0, float(par.abs().max())
