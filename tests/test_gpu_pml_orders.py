"""The PML in the stage at every order against the oracle: where a level's
loads are requested and when the RK register is read differ with the order.

Tolerance: the two sum the same products in other orders (1e-14 relative at
most per residual); 25 stages of a random state, the aux fields fed by the
fields: below 1e-11 of the largest value, the bound of the other parity tests.
"""
import numpy as np
import pytest

from nekcem_amd.maxwell import MaxwellSolver
from nekcem_amd.mesh import BoxMesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("material", ["element", "node"])
@pytest.mark.parametrize("N", range(3, 10))
def test_steps_against_the_oracle(oracle, N, material):
    print(f"[case] PML against the oracle N={N} {material}", flush=True)
    rng = np.random.default_rng(N)
    nel = (4, 3, 4)
    mesh = BoxMesh(nel, N, (0, 0, 0), (1, 1, 1), ("PEC", "P", "PEC"))
    n, n3 = mesh.npts, mesh.n1 ** 3
    if material == "element":
        eps, mu = np.repeat(rng.uniform(1, 2, mesh.nelt), n3), np.repeat(rng.uniform(1, 2, mesh.nelt), n3)
    else:
        eps, mu = rng.uniform(1, 2, n), rng.uniform(1, 2, n)
    ref = oracle.BoxCase(oracle.BoxSpec(nel=nel, N=N, lo=(0, 0, 0), hi=(1, 1, 1), bc=("PML", "P", "PML")),
                         eps=eps, mu=mu)
    ref.set_pml(1, 2.0, 1e-4)
    H, E = rng.standard_normal((3, n)), rng.standard_normal((3, n))
    on = np.repeat(ref.pmltag != 0, n3)
    P = rng.standard_normal((6, n)) * on
    s = MaxwellSolver(mesh, eps=eps, mu=mu)
    s.set_state(H, E)
    s.set_pml(ref.pmlptr, ref.pmlsigma.reshape(3, n), P[:3], P[3:])
    dt = mesh.dt(0.05)
    s.step(dt, 5)
    want = ref.run(H, E, dt, 5, P=P)
    got = np.concatenate(s.get_state())
    both = np.concatenate([want["H"], want["E"]])
    assert np.max(np.abs(got - both)) <= 1e-11 * np.max(np.abs(both))
    gP, wP = s.get_pml("state")[:, on], want["P"][:, on]
    assert np.max(np.abs(gP - wP)) <= 1e-11 * np.max(np.abs(wP))
    s.close()
