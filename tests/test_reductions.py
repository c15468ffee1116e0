"""CFL number, step norm and volume integrals walk the cells from a thread's
first one by additions with a carry: grids of a few cells, of less than a
block, and of more cells than a launch has threads (2^19), with another
spacing at every point, against numpy.

A product of the integrals has 6 roundings and a sum no more than 600 terms in
a row (2e-16 x 600 = 1.2e-13 of the sum of magnitudes, which no sum reaches);
a CFL number has 20 roundings, at most 4.4e-15."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

GAMMA = 1.4


@pytest.mark.parametrize("dims", [(5, 5, 5), (7, 11, 13), (130, 6, 5), (5, 6, 301), (101, 97, 61)])
def test_reductions_match_numpy(dims):
    from hypar_amd.solver import NS3D
    rng = np.random.default_rng(11)
    nx, ny, nz = dims
    dxinv = [rng.uniform(1.0, 3.0, n + 6) for n in dims]
    rho, p = (rng.uniform(0.5, 2.0, (nz, ny, nx)) for _ in range(2))
    vel = rng.uniform(-1.0, 1.0, (3, nz, ny, nx))
    u = np.stack([rho, *(rho * vel), p / (GAMMA - 1) + 0.5 * rho * (vel ** 2).sum(0)])
    v = u + rng.uniform(-1.0, 1.0, u.shape)
    d = [a[3:-3].reshape([-1 if k == 2 - i else 1 for k in range(3)]) for i, a in enumerate(dxinv)]
    q = u[1:4] / u[0]
    c = np.sqrt(GAMMA * (u[4] - 0.5 * u[0] * (q ** 2).sum(0)) * (GAMMA - 1) / u[0])
    cfl = max(float(((np.abs(q[i]) + c) * 0.01 * d[i]).max()) for i in range(3))
    dV = 1 / (d[0] * d[1] * d[2])
    print(f"[gpu] reductions dims={dims}", flush=True)
    s = NS3D(dims, gamma=GAMMA, dxinv=np.concatenate(dxinv))
    ud, vd = (torch.tensor(a.reshape(-1), device="cuda") for a in (u, v))
    got = s.cfl(ud, 0.01), s.step_norm(ud, vd), s.volume_integral(ud)
    s.close()
    assert abs(got[0] - cfl) <= 1e-14 * cfl
    norm = np.sqrt(((u - v) ** 2).sum() / (nx * ny * nz))
    assert abs(got[1] - norm) <= 1e-13 * norm
    for k in range(5):
        assert abs(got[2][k] - (u[k] * dV).sum()) <= 1e-13 * np.abs(u[k] * dV).sum()
