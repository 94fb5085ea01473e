"""Equal-work element ranges under a PML: a PML on the outer elements against
one that lists every element, with sigma zero inside.  The second costs the
same everywhere, so its ranges differ; the physics does not, and adding the
zeros rounds nothing: equal bit for bit.  Meshes just above the size from which the
ranges are used, with elements left over.
"""
import numpy as np
import pytest

from nekcem_amd.maxwell import MaxwellSolver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,nel", [(3, (13, 13, 13)), (5, (11, 10, 11)), (7, (9, 11, 12)), (8, (8, 9, 8)), (9, (9, 7, 9))])
@pytest.mark.parametrize("drude", [False, True])
def test_ranges_do_not_change_the_fields(N, nel, drude):
    print(f"[case] PML ranges N={N} nel={nel} drude={drude}", flush=True)
    rng = np.random.default_rng(N)
    n3, ne = (N + 1) ** 3, nel[0] * nel[1] * nel[2]
    at = [v.reshape(-1) for v in np.meshgrid(*(np.arange(n) for n in nel[::-1]), indexing="ij")]
    outer = np.zeros(ne, bool)
    for v, n in zip(at, nel[::-1], strict=True):
        outer |= (v == 0) | (v == n - 1)
    sigma = rng.uniform(0, 5, (3, ne, n3)) * outer[None, :, None]
    U = rng.standard_normal((6, ne * n3))
    out = []
    for listed in (np.nonzero(outer)[0], np.arange(ne)):
        s = MaxwellSolver.from_box(nel, N, (0.0,) * 3, (1.0,) * 3, ("PEC",) * 3)
        s.set_state(U[:3], U[3:])
        s.set_pml(listed, sigma.reshape(3, -1))
        if drude:
            el = np.arange(ne // 2, ne // 2 + 3)
            s.set_drude((el[:, None] * n3 + np.arange(n3)).reshape(-1), 0.3, 4.0)
        s.step(1e-4, 2)
        out.append(np.concatenate(s.get_state()))
        s.close()
    assert np.array_equal(out[0], out[1])
