"""Adjoint passes that take the buffers of the pass before: the gradients are
those of a fresh solver, bit for bit, whatever ran in between, and the memory
comes back with adjoint_release and close."""
import ctypes as C

import numpy as np
import pytest

from nekcem_amd.maxwell import MaxwellSolver
from nekcem_amd.mesh import BoxMesh

pytestmark = pytest.mark.gpu


def _mesh():
    return BoxMesh((3, 2, 2), 5, (0, 0, 0), (1, 1, 1), ("PEC", "P", "PEC"))


def _pass(s, mesh, p):
    """One pass with parameters p = (seed, Drude elements, steps, every, eps/mu gradients)."""
    seed, nd, steps, every, grads = p
    rng = np.random.default_rng(seed)
    n, n3 = mesh.npts, mesh.n1 ** 3
    s.adjoint_set_grads(grads)
    s.set_materials(rng.uniform(1, 2, n), rng.uniform(1, 2, n))
    d = np.arange(nd * n3)
    s.set_drude(d, rng.uniform(0.1, 1, len(d)), rng.uniform(1, 2, len(d)))
    s.time = 0.0
    s.set_state(rng.standard_normal((3, n)), rng.standard_normal((3, n)))
    s.adjoint_forward(mesh.dt(0.2), steps, every)
    out = list(s.adjoint_backward(rng.standard_normal((3, n)), rng.standard_normal((3, n))))
    if nd:
        out += list(s.adjoint_drude_grad())
    return out


def _free(s):
    """Free device memory, asked of the runtime the library runs on."""
    free, total = C.c_size_t(), C.c_size_t()
    assert s._L.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


PASSES = [(1, 0, 6, 3, True), (2, 0, 6, 3, True), (3, 2, 6, 3, True), (4, 2, 6, 3, False), (5, 1, 7, 2, False),
          (6, 0, 4, 4, True), (7, 0, 4, 4, True)]


def test_passes_on_one_solver_equal_fresh_solvers():
    mesh = _mesh()
    a, b = MaxwellSolver(mesh), MaxwellSolver(mesh)
    for p in PASSES:
        print(f"[case] adjoint buffers {p}", flush=True)
        fresh = MaxwellSolver(mesh)
        want = _pass(fresh, mesh, p)
        fresh.close()
        # two solvers in turn: neither may take the other's buffers
        for s in (a, b, a):
            for g, w in zip(_pass(s, mesh, p), want, strict=True):
                assert np.array_equal(g, w)
    a.close()
    b.close()


def test_buffers_are_given_back():
    mesh = BoxMesh((8, 8, 8), 7, (0, 0, 0), (1, 1, 1), ("PEC",) * 3)
    print("[case] adjoint buffers given back", flush=True)
    s = MaxwellSolver(mesh)
    _pass(s, mesh, (1, 0, 2, 2, True))
    s.adjoint_release()
    free = _free(s)
    for again in (False, True):
        _pass(s, mesh, (1, 0, 8, 8, True))
        held = s.adjoint_info()["bytes"]
        assert held > 1 << 29
        s.set_materials(np.ones(mesh.npts))       # drops the pass: its buffers wait
        assert s.adjoint_info()["bytes"] == 0
        if again:
            s.adjoint_release()
        else:
            s.set_lorentz(np.zeros(0, int), *[np.zeros(0)] * 3)
        assert _free(s) > free - held // 4
    s.close()
