"""The reversed stage at every order: both ways of storing (through the caches,
or past them on large meshes), with and without the eps/mu gradients, with a
Drude region in some elements (equal-work element ranges, lanes that repeat
an element's first or last node).

* against the oracle's adjoint on a small box (walls and wrap-around faces).
  Tolerance: the two sum the same products in other orders; a gradient is a
  sum over 15 stages of terms of like size, each a few sums of up to 60
  products, 1e-14 relative at most; with the growth of the adjoint state over
  three short steps below 1e-11 of the largest value.
* a large box that repeats a small one: every copy's gradients equal the
  small box's.  Tolerance: the element tables are built from other extents
  (1e-16 per entry), ten stages: below 1e-12 of the largest value.
"""
import numpy as np
import pytest

from nekcem_amd.maxwell import MaxwellSolver
from nekcem_amd.mesh import BoxMesh

pytestmark = pytest.mark.gpu

ORDERS = range(3, 10)
# copies per axis of a 2 x 3 x 2 box: just past 256 MB of 18 doubles a node
COPIES = {3: (15, 12, 14), 4: (10, 10, 13), 5: (9, 9, 9), 6: (8, 8, 8), 7: (7, 7, 7), 8: (6, 6, 6), 9: (6, 6, 5)}


def _close(got, want, rel):
    for g, w in zip(got, want, strict=True):
        assert np.max(np.abs(g - w)) <= rel * np.max(np.abs(w))


@pytest.mark.parametrize("N", ORDERS)
def test_gradients_against_the_oracle(oracle, N):
    print(f"[case] reversed stage against the oracle N={N}", flush=True)
    rng = np.random.default_rng(N)
    nel, bc, steps = (2, 3, 2), ("PEC", "P", "PEC"), 3
    mesh = BoxMesh(nel, N, (0, 0, 0), (1, 1, 1), bc)
    n, n3 = mesh.npts, mesh.n1 ** 3
    eps, mu = rng.uniform(1, 4, n), rng.uniform(1, 2, n)
    el = np.array([0, 3, 4, mesh.nelt - 1])
    d = (el[:, None] * n3 + np.arange(n3)).ravel()
    a, b = rng.uniform(0.1, 1, len(d)), rng.uniform(1, 4, len(d))
    H0, E0 = rng.standard_normal((3, n)), rng.standard_normal((3, n))
    probes = rng.choice(n, n // 3, replace=False)
    target = rng.standard_normal(len(probes))
    dt = mesh.dt(0.1)
    ref = oracle.BoxCase(oracle.BoxSpec(nel=nel, N=N, lo=(0, 0, 0), hi=(1, 1, 1), bc=bc), eps=eps, mu=mu)
    ref.set_drude(d, a, b)
    _, ge, gm, _, ga, gb = ref.loss_and_grad(H0, E0, dt, steps, probes, target, drude=True)
    s = MaxwellSolver(mesh, eps=eps, mu=mu)
    s.set_materials(eps, mu)
    for grads in (True, False):
        s.adjoint_set_grads(grads)
        s.set_drude(d, a, b)
        s.time = 0.0
        s.set_state(H0, E0)
        s.adjoint_forward(dt, steps, 2)
        lamE = np.zeros((3, n))
        lamE[2, probes] = 2 * (s.get_state()[1][2, probes] - target)
        got = s.adjoint_backward(np.zeros((3, n)), lamE)
        if grads:
            _close(got, (ge, gm), 1e-11)
        _close(s.adjoint_drude_grad(), (ga, gb), 1e-11)
    s.close()


@pytest.mark.parametrize("grads", [True, False])
@pytest.mark.parametrize("N", ORDERS)
def test_large_box_repeats_small_box(N, grads):
    print(f"[case] streamed reversed stage N={N} gradients={grads}", flush=True)
    rng = np.random.default_rng(N)
    n1, (sx, sy, sz), (cx, cy, cz) = N + 1, (2, 3, 2), COPIES[N]
    shape = (sz, sy, sx, n1, n1, n1)
    U, L = rng.standard_normal((6,) + shape), rng.standard_normal((6,) + shape)
    eps, mu = rng.uniform(1, 4, shape), rng.uniform(1, 2, shape)
    dense = rng.uniform(size=(sz, sy, sx)) < 0.4
    dense[0, 0, 0] = True
    out = {}
    for name, (a, b, c) in (("small", (1, 1, 1)), ("large", (cx, cy, cz))):
        nel = (sx * a, sy * b, sz * c)
        tile = lambda v, lead: np.tile(v, (1,) * lead + (c, b, a) + (1,) * (v.ndim - 3 - lead))
        flat = lambda v: np.ascontiguousarray(tile(v, 1)).reshape(6, -1)
        s = MaxwellSolver.from_box(nel, N, (0.0,) * 3, tuple(0.5 * v for v in nel), ("P",) * 3)
        assert (s.npts * 18 * 8 > 256 * 2 ** 20) == (name == "large")
        s.adjoint_set_grads(grads)
        if grads:
            s.set_materials(tile(eps, 0).reshape(-1), tile(mu, 0).reshape(-1))
        el = np.nonzero(tile(dense, 0).reshape(-1))[0]
        nodes = (el[:, None] * n1 ** 3 + np.arange(n1 ** 3)[None, :]).reshape(-1)
        s.set_drude(nodes, 0.3, 4.0)
        F = flat(U)
        s.set_state(F[:3], F[3:])
        s.adjoint_forward(1e-3, 2, 2)
        F = flat(L)
        g = list(s.adjoint_backward(F[:3], F[3:])) if grads else []
        if not grads:
            s.adjoint_backward(F[:3], F[3:])
        for v in s.adjoint_drude_grad():
            w = np.zeros(s.npts)
            w[nodes] = v
            g.append(w)
        out[name] = [v.reshape((c, sz, b, sy, a, sx, n1 ** 3)) for v in g]
        s.close()
    _close(out["large"], out["small"], 1e-12)
