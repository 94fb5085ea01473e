"""The stage with an element in several workgroups (slabs of its levels, small
meshes) against whole elements: a large box that repeats a small one, at every
order and slab count, plain, with a Drude and Lorentz region and a source, and
with a PML.  Every copy must give the small box's fields and currents.

Tolerance: the same operations in the same order; the two meshes' element
tables are built from different extents and may round differently (relative
1e-16 per entry); over ten stages below 1e-13 of the largest value.
"""
import numpy as np
import pytest

from nekcem_amd.maxwell import MaxwellSolver

pytestmark = pytest.mark.gpu

# (order, small box): from 5 slabs down to 2
SMALL = [(5, (4, 4, 8)), (5, (1, 2, 2)), (6, (4, 4, 8)), (7, (4, 4, 4)), (7, (5, 5, 4)), (7, (8, 8, 8)), (8, (5, 4, 4)),
         (8, (4, 4, 6)), (9, (3, 4, 4)), (9, (5, 4, 4)), (9, (4, 4, 6))]


@pytest.mark.parametrize("physics", ["none", "dispersive", "pml"])
@pytest.mark.parametrize("N,small", SMALL)
def test_slabs_equal_whole_elements(N, small, physics):
    print(f"[case] stage slabs N={N} nel={small} {physics}", flush=True)
    rng = np.random.default_rng(N)
    n1, (sx, sy, sz) = N + 1, small
    n3, ne = n1 ** 3, sx * sy * sz
    copies = 513 // ne + 1                       # along z: more than 512 elements, where there are no slabs
    U = rng.standard_normal((6, ne * n3))
    eps = rng.uniform(1, 4, ne)
    some = np.nonzero(rng.uniform(size=ne) < 0.5)[0]
    some = some if len(some) else np.array([0])
    sigma, amp = rng.uniform(0, 5, (3, len(some), n3)), rng.uniform(0, 1, (len(some), n3))
    out = []
    for c in (1, copies):
        s = MaxwellSolver.from_box((sx, sy, sz * c), N, (0.0,) * 3, (0.5 * sx, 0.5 * sy, 0.5 * sz * c), ("P",) * 3,
                                   eps_elem=np.tile(eps, c))
        V = np.ascontiguousarray(np.tile(U, (1, c)))
        s.set_state(V[:3], V[3:])
        listed = (some[None, :] + ne * np.arange(c)[:, None]).reshape(-1)
        nodes = (listed[:, None] * n3 + np.arange(n3)).reshape(-1)
        if physics == "dispersive":
            s.set_drude(nodes, 0.3, 4.0)
            s.set_lorentz(nodes, 0.2, 3.0, 1.0)
        if physics == "pml":
            sig = np.zeros((3, ne * c, n3))
            sig[:, listed] = np.tile(sigma, (1, c, 1))
            s.set_pml(listed, sig.reshape(3, -1))
        if physics != "none":
            a = np.zeros(ne * c * n3)
            a[nodes] = np.tile(amp, (c, 1)).reshape(-1) * 1e-3
            s.set_source(a, (0.3, 0.5, 0.8), 1e-3, 1e-3)
        s.step(1e-3, 2)
        got = [np.concatenate(s.get_state()).reshape(6, c, -1)]
        if physics == "dispersive":
            got += [v.reshape(v.shape[0], c, -1) for v in (s.get_drude()[0], s.get_lorentz()[0])]
        if physics == "pml":
            got.append(s.get_pml().reshape(6, c, -1))
        out.append(got)
        s.close()
    for want, got in zip(*out, strict=True):
        assert np.max(np.abs(got - want)) <= 1e-13 * np.max(np.abs(want))
