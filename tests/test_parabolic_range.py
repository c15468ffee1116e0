"""The viscosity T^0.76 over temperatures of several powers of two, on both
sides of the mantissa sqrt(1/2) where its logarithm's interval begins: the
viscous term against the oracle, whose pow is correct to a few units of 2^-52;
the derivatives of fields of scale one lose no more than a factor of 100."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

GAMMA = 1.4


@pytest.mark.parametrize("k", [-40, -21, -1, 0, 1, 22, 40])
def test_viscous_term_over_powers_of_two(k):
    from hypar_amd import decks
    from hypar_amd.solver import NS3D
    from oracle.oracle import Oracle
    dims = (12, 10, 14)
    rng = np.random.default_rng(100 + k)
    shape = dims[::-1]
    T = np.sqrt(0.5) * 2.0 ** (k + rng.uniform(-1.0, 1.0, shape))
    rho = rng.uniform(0.5, 2.0, shape)
    v = 2.0 ** (k / 2) * rng.uniform(-0.3, 0.3, (3, *shape))
    p = T * rho / GAMMA
    u = np.stack([rho, *(rho * v), p / (GAMMA - 1) + 0.5 * rho * (v ** 2).sum(0)], axis=-1)
    print(f"[gpu] viscous term around T = 2^{k}", flush=True)
    s = NS3D(dims, Re=1000.0, Minf=0.1)
    got = s.to_host(s.parabolic(s.to_device(u)))
    s.close()
    ref = Oracle(dims, Re=1000.0, Minf=0.1).parabolic(u)
    for c in range(1, 5):
        assert decks.rel_l2(got[..., c], ref[..., c]) <= 1e-13
