"""Material tables formed on the device, and node lists instead of whole
states: the same values as the tables of nkc_create and as whole states.

The tables are the host's divisions and square roots in the host's order, so
every comparison is of the same bits, except the adjoint's seeds: one at a
listed node is that node's entry of a whole state of seeds, again the same
bits; a node listed twice sums its two seeds (one rounding of a sum of two).
"""
import ctypes as C

import numpy as np
import pytest

from nekcem_amd import _lib
from nekcem_amd.maxwell import MaxwellSolver
from nekcem_amd.mesh import BoxMesh

pytestmark = pytest.mark.gpu


def _dp(a):
    return a.ctypes.data_as(C.POINTER(C.c_double))


def _ip(a):
    return a.ctypes.data_as(C.POINTER(C.c_int64))


@pytest.mark.parametrize("N,nel,bc", [(3, (1, 1, 1), ("PEC",) * 3), (4, (3, 1, 2), ("P", "PEC", "P")),
                                      (7, (2, 3, 2), ("PEC", "P", "PEC")), (9, (5, 3, 3), ("P",) * 3)])
def test_tables_equal_the_hosts(N, nel, bc):
    print(f"[case] material tables N={N} nel={nel}", flush=True)
    rng = np.random.default_rng(N)
    mesh = BoxMesh(nel, N, (0, 0, 0), (1, 1, 1), bc)
    n = mesh.npts
    eps, mu = 10.0 ** rng.uniform(-6, 6, n), 10.0 ** rng.uniform(-6, 6, n)
    H, E = rng.standard_normal((3, n)), rng.standard_normal((3, n))
    made = MaxwellSolver(mesh, eps=eps, mu=mu)
    made.set_state(H, E)
    want = made.residual()
    for s in (MaxwellSolver(mesh), MaxwellSolver(mesh, eps=np.ones(n), mu=rng.uniform(1, 2, n))):
        s.set_materials(eps, mu)
        for bad, node in ((0.0, n - 1), (-1.0, 0), (np.nan, n // 2)):
            e2, m2 = eps.copy(), mu.copy()
            (e2 if node else m2)[node] = bad
            if node + 1 < n:
                e2[node + 1] = -1.0
            with pytest.raises(Exception, match=rf"material not positive at node {node}$"):
                s.set_materials(e2, m2)
        s.set_state(H, E)
        for g, w in zip(s.residual(), want, strict=True):
            assert np.array_equal(g, w)
        # the adjoint's admittances come from the same tables
        k = (rng.standard_normal((3, n)), rng.standard_normal((3, n)))
        for g, w in zip(s.adjoint_apply(*k), made.adjoint_apply(*k), strict=True):
            assert np.array_equal(g, w)
        s.close()
    made.close()


@pytest.mark.parametrize("nlist", [1, 7, 300, 70000])
def test_node_lists_equal_whole_states(nlist):
    print(f"[case] node lists of {nlist}", flush=True)
    rng = np.random.default_rng(nlist)
    mesh = BoxMesh((3, 2, 2), 7, (0, 0, 0), (1, 1, 1), ("PEC", "P", "PEC"))
    n = mesh.npts
    s = MaxwellSolver(mesh)
    s.set_materials(rng.uniform(1, 2, n), rng.uniform(1, 2, n))
    s.set_state(rng.standard_normal((3, n)), rng.standard_normal((3, n)))
    s.adjoint_forward(mesh.dt(0.2), 4, 2)
    whole = np.concatenate(s.get_state())
    nodes = rng.integers(0, n, nlist)               # with repeats
    nodes[0] = n - 1
    out = np.empty((6, nlist))
    _lib.check(s._L.nkc_get_state_at(s._h, nlist, _ip(nodes), _dp(out)))
    assert np.array_equal(out, whole[:, nodes])
    # distinct nodes, then the first one twice
    nodes = np.unique(nodes)
    seeds = rng.standard_normal((6, len(nodes)))
    lam = np.zeros((6, n))
    lam[:, nodes] = seeds
    for twice in (False, True):
        if twice:
            nodes = np.append(nodes, nodes[0])
            seeds = np.concatenate([seeds, rng.standard_normal((6, 1))], axis=1)
            lam[:, nodes[0]] += seeds[:, -1]
        want = s.adjoint_backward(lam[:3], lam[3:])
        got = [np.empty(n), np.empty(n)]
        _lib.check(s._L.nkc_adjoint_backward_at(s._h, len(nodes), _ip(nodes), _dp(np.ascontiguousarray(seeds)),
                                                _dp(got[0]), _dp(got[1])))
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
    for bad in (-1, n):
        with pytest.raises(Exception, match="is not a node"):
            _lib.check(s._L.nkc_get_state_at(s._h, 1, _ip(np.array([bad])), _dp(out)))
    s.close()
