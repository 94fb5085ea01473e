"""The stage kernel's two ways of storing (through the caches, or past them
once the working set outgrows the Infinity Cache) on the same physics: a box
whose state repeats a small box's.  Every element of the large box then sees
what its image in the small one sees, so after two steps each copy must equal
the small box, at every order (ragged chunks, partial cache lines at the
elements' ends, both workgroup shapes).

Tolerance: the two meshes' element tables are built from different extents
and may round differently (relative 1e-16 per entry); over two steps of ten
stages that stays below 1e-13 of the field's largest value.
"""
import numpy as np
import pytest

from nekcem_amd.maxwell import MaxwellSolver

pytestmark = pytest.mark.gpu

SMALL = (2, 3, 2)
# copies per axis: just past 256 MB of u, k and output (18 doubles a node)
COPIES = {3: (15, 12, 14), 4: (10, 10, 13), 5: (9, 9, 9), 6: (8, 8, 8), 7: (7, 7, 7), 8: (6, 6, 6), 9: (6, 6, 5)}


@pytest.mark.parametrize("drude", [False, True])
@pytest.mark.parametrize("N", sorted(COPIES))
def test_large_box_repeats_small_box(N, drude):
    print(f"[case] streamed stage N={N} drude={drude}", flush=True)
    rng = np.random.default_rng(N)
    n1, (sx, sy, sz), (cx, cy, cz) = N + 1, SMALL, COPIES[N]
    eps = rng.uniform(1, 4, (sz, sy, sx))
    F = rng.standard_normal((6, sz, sy, sx, n1, n1, n1))
    dense = rng.uniform(size=(sz, sy, sx)) < 0.4
    dense[0, 0, 0] = True
    out = {}
    for name, (a, b, c) in (("small", (1, 1, 1)), ("large", (cx, cy, cz))):
        nel = (sx * a, sy * b, sz * c)
        tile = lambda v, lead: np.tile(v, (1,) * lead + (c, b, a) + (1,) * (v.ndim - 3 - lead))
        s = MaxwellSolver.from_box(nel, N, (0.0,) * 3, tuple(0.5 * v for v in nel), ("P",) * 3,
                                   eps_elem=tile(eps, 0).reshape(-1))
        assert (s.npts * 18 * 8 > 256 * 2 ** 20) == (name == "large")
        U = np.ascontiguousarray(tile(F, 1)).reshape(6, -1)
        s.set_state(U[:3], U[3:])
        if drude:
            el = np.nonzero(tile(dense, 0).reshape(-1))[0]
            nodes = (el[:, None] * n1 ** 3 + np.arange(n1 ** 3)[None, :]).reshape(-1)
            s.set_drude(nodes, 0.3, 4.0)
        s.step(1e-3, 2)
        H, E = s.get_state()
        out[name] = np.concatenate([H, E]).reshape((6, c, sz, b, sy, a, sx, n1 ** 3))
        s.close()
    want = out["small"]
    tol = 1e-13 * np.max(np.abs(want))
    assert np.max(np.abs(out["large"] - want)) <= tol
