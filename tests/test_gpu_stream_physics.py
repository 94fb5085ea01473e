"""The instances of the stage that test_gpu_box_stream does not take, streamed
(large) against cached and in slabs (small): per-node materials, alone, with a
PML, with an incident wave and with a sheet.  A box whose materials, regions,
waves and state repeat a small box's must give each copy the small box's fields.

Tolerance: that of test_gpu_box_stream (the element tables round differently
with the extents, 1e-16 per entry, over ten stages below 1e-13 of the largest
value); the incident wave's phase at the far copies is known to 1e-16 of up to
a few hundred, 1e-13 of the wave, which a step adds to the fields times dt
times the lift, at most a tenth.
"""
import numpy as np
import pytest

from nekcem_amd.maxwell import MaxwellSolver
from tests.test_gpu_box_stream import COPIES, SMALL

pytestmark = pytest.mark.gpu

CASES = [(N, p) for N in sorted(COPIES) for p in ("none", "pml", "incident")] + [(N, "sheet") for N in (3, 5, 8)]


@pytest.mark.parametrize("N,physics", CASES)
def test_large_box_repeats_small_box(N, physics):
    print(f"[case] streamed stage, per-node materials, N={N} {physics}", flush=True)
    rng = np.random.default_rng(N)
    n1, (sx, sy, sz) = N + 1, SMALL
    n2, n3 = n1 * n1, n1 ** 3
    shape = (sz, sy, sx)
    eps, mu = rng.uniform(1, 4, shape + (n3,)), rng.uniform(1, 2, shape + (n3,))
    F = rng.standard_normal((6,) + shape + (n3,))
    some = rng.uniform(size=shape) < 0.4
    some[0, 0, 0] = True
    sigma = rng.uniform(0, 5, (3,) + shape + (n3,)) * some[..., None]
    lit = rng.uniform(size=(6,) + shape) < 0.3
    par = np.array([0.5, 1.0, -0.1, 30.0, 2.0, 0.5, 2.0, -0.1, 30.0, 2.0, -0.5, 1.0]) * rng.uniform(0.5, 1, 12)
    out = []
    for copies in ((1, 1, 1), COPIES[N]):
        nel = tuple(s * c for s, c in zip(SMALL, copies))
        a, b, c = copies
        tile = lambda v, lead: np.tile(v, (1,) * lead + (c, b, a) + (1,) * (v.ndim - 3 - lead))
        s = MaxwellSolver.from_box(nel, N, (0.0,) * 3, tuple(0.5 * v for v in nel), ("P",) * 3)
        s.set_materials(tile(eps, 0).reshape(-1), tile(mu, 0).reshape(-1))
        U = np.ascontiguousarray(tile(F, 1)).reshape(6, -1)
        s.set_state(U[:3], U[3:])
        if physics == "pml":
            s.set_pml(np.nonzero(tile(some, 0).reshape(-1))[0], tile(sigma, 1).reshape(3, -1), U[:3], U[3:])
        faces = np.argwhere(tile(lit, 1).reshape(6, -1))           # (face - 1, element)
        if physics == "incident":
            # one wavelength a copy, so that every copy sees the same wave
            k = tuple(2 * np.pi / (0.5 * v) for v in SMALL)
            s.set_incident([(e, f + 1) for f, e in faces], k, 3.0, (0.3, 0.5, -0.2), (-0.4, 0.1, 0.6))
        if physics == "sheet":
            g = (faces[:, 1:] * 6 * n2 + faces[:, :1] * n2 + np.arange(n2)).reshape(-1)
            s.set_graphene(np.sort(g), par)
        s.step(1e-3, 2)
        got = [np.concatenate(s.get_state()).reshape(6, c, sz, b, sy, a, sx, n3)]
        if physics == "pml":
            got.append(s.get_pml().reshape(6, c, sz, b, sy, a, sx, n3))
        out.append(got)
        s.close()
    for want, got in zip(*out, strict=True):
        assert np.max(np.abs(got - want)) <= 1e-13 * np.max(np.abs(want))
