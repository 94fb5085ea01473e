"""The general kernel at N = 7 on a mesh whose stages stream past the caches
(workgroups of four waves) against the same elements on a small mesh (eight
waves): blocks of a curved mesh side by side, unconnected.

Tolerance: coordinates shifted by up to 1400 round at 2e-13, which is 1e-11 of
a metric at a node spacing of 0.03; a step changes the fields by dt times their
derivative, about a hundredth, so two steps stay below 1e-12; 1e-11 is asked.
"""
import numpy as np
import pytest

from nekcem_amd.maxwell import MaxwellSolver

from .test_gpu_general_slabs import _mesh

pytestmark = pytest.mark.gpu


def test_streamed_mesh_equals_small_mesh():
    print("[case] general stream N=7", flush=True)
    N, copies = 7, 912
    rng = np.random.default_rng(1)
    n = 4 * (N + 1) ** 3
    F = rng.standard_normal((6, n))
    out = []
    for c in (70, copies):
        mesh = _mesh(N, c)
        s = MaxwellSolver(mesh)
        assert (s.npts * 18 * 8 > 256 * 2 ** 20) == (c == copies)
        V = np.tile(F, (1, c))
        s.set_state(V[:3], V[3:])
        s.step(1e-4, 2)
        out.append(np.concatenate(s.get_state()).reshape(6, c, n))
        s.close()
    want = out[0][:, :1]
    assert np.max(np.abs(out[1] - want)) <= 1e-11 * np.max(np.abs(want))
