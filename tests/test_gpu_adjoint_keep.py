"""Adjoint passes that take over the buffers of the pass before
(adjoint_buffers_kept): the gradients are those of a fresh solver, bit for
bit, whatever ran in between."""
import numpy as np
import pytest

from nekcem_amd.maxwell import MaxwellSolver
from tests.test_gpu_adjoint_buffers import PASSES, _mesh, _pass

pytestmark = pytest.mark.gpu


def test_passes_that_take_over_buffers_equal_fresh_solvers():
    mesh = _mesh()
    a, b = MaxwellSolver(mesh), MaxwellSolver(mesh)
    for p in PASSES:
        print(f"[case] adjoint buffers taken over {p}", flush=True)
        fresh = MaxwellSolver(mesh)
        want = _pass(fresh, mesh, p)
        fresh.close()
        # two solvers in turn: neither may take the other's buffers
        for s in (a, b, a):
            with s.adjoint_buffers_kept():
                got = _pass(s, mesh, p)
            for g, w in zip(got, want, strict=True):
                assert np.array_equal(g, w)
    a.close()
    b.close()
