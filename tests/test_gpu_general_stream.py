"""The general kernel at N = 7 on a mesh whose stages stream past the caches
(workgroups of four waves) against the first of its elements on a mesh that
does not (eight waves): blocks of a curved mesh side by side, unconnected.
The blocks both meshes have lie at the same coordinates and every node sums
in the same order, so they are equal bit for bit.
"""
import numpy as np
import pytest

from nekcem_amd.maxwell import MaxwellSolver

from .test_gpu_general_slabs import _mesh

pytestmark = pytest.mark.gpu


def test_streamed_mesh_equals_small_mesh():
    print("[case] general stream N=7", flush=True)
    N, few, many = 7, 70, 912
    rng = np.random.default_rng(1)
    n = 4 * (N + 1) ** 3
    F = rng.standard_normal((6, n))
    out = []
    for c in (few, many):
        mesh = _mesh(N, c)
        s = MaxwellSolver(mesh)
        assert (s.npts * 18 * 8 > 256 * 2 ** 20) == (c == many)
        V = np.tile(F, (1, c))
        s.set_state(V[:3], V[3:])
        s.step(1e-4, 2)
        out.append(np.concatenate(s.get_state()).reshape(6, c, n)[:, :few])
        s.close()
    assert np.array_equal(out[0], out[1])
