"""The general kernel with an element in several workgroups (slabs of its
levels) against whole elements: a curved periodic-free box repeated side by
side.  Meshes of few elements take slabs, of many elements none; every copy
of the small mesh's element block in a larger, disconnected mesh must give
the same fields (each order's uneven slabs, first and last level in different
workgroups).

Tolerance: the same operations on the same values, summed alike; the block's
coordinates are shifted, which rounds the metrics anew (1e-15 relative at
shifts of order 10), over two steps below 1e-11 of the largest value.
"""
import numpy as np
import pytest

from nekcem_amd.hexmesh import HexMesh
from nekcem_amd.maxwell import MaxwellSolver
from nekcem_amd.mesh import box_coords

pytestmark = pytest.mark.gpu


def _mesh(N, copies):
    x, y, z = box_coords((2, 1, 2), N, (0.0,) * 3, (1.0,) * 3)
    w = 0.06 * np.sin(np.pi * x) * np.sin(np.pi * y) * np.sin(np.pi * z)
    x, y, z = x + w, y - w, z + 0.5 * w
    # disjoint blocks: a wall on every outer face
    return HexMesh.from_coords(N, *(np.concatenate([v + s * 1.5 * c for c in range(copies)])
                                    for v, s in ((x, 1.0), (y, 0.0), (z, 0.0))))


@pytest.mark.parametrize("N,copies", [(3, 70), (4, 70), (6, 66), (7, 66), (8, 66), (9, 70), (10, 35), (11, 35)])
def test_slabs_equal_whole_elements(N, copies):
    """4 elements (4 to 8 slabs each) against 140 or more (one or two)."""
    print(f"[case] general slabs N={N}", flush=True)
    rng = np.random.default_rng(N)
    n = 4 * (N + 1) ** 3
    F = rng.standard_normal((6, n))
    out = []
    for c in (1, copies):
        mesh = _mesh(N, c)
        s = MaxwellSolver(mesh, eps=np.tile(np.linspace(1.0, 3.0, n), c))
        U = np.tile(F, (1, c))
        s.set_state(U[:3], U[3:])
        s.step(1e-4, 2)
        H, E = s.get_state()
        out.append(np.concatenate([H, E]).reshape(6, c, n))
        s.close()
    assert np.max(np.abs(out[1] - out[0])) <= 1e-11 * np.max(np.abs(out[0]))
