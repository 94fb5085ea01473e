"""Which stages stream their outputs past the caches, from the instances
launched on the stand-in runtime: once what a stage touches (u, k, the output,
per-node materials and their face coefficients, source amplitudes, dispersive
regions) is more than 256 MB, whatever order it was set in."""
from tests.fake_hip import fake_hip, needs_gxx  # noqa: F401

pytestmark = needs_gxx


def test_what_counts(fake_hip):  # noqa: F811
    fake_hip("""
def streams(s):
    log()
    s.step(1e-3, 1)
    k = {l.split("box_kernel<")[1].split(">")[0].split(", ")[4] for l in launches("box_kernel")}
    assert len(k) == 1
    return k.pop() == "true"
N, n3 = 3, 64
def box(nel): return MaxwellSolver.from_box((nel, nel, nel), N)
s = box(28)                     # 202 MB
n = s.npts
assert not streams(s)
s.set_source(np.full(n, 1e-3), (0, 0, 1.), 1.0, 0.5)                      # 214
assert not streams(s)
nodes = np.arange(28 ** 3 * n3)
s.set_drude(nodes[:28 ** 3 * n3 // 2], 0.1, 4.0)                          # 259
assert not streams(s)
s.set_drude(nodes, 0.1, 4.0)                                              # 304
assert streams(s)
s.set_drude(nodes[:0], 0.1, 4.0)
assert not streams(s)
s.set_lorentz(nodes[:28 ** 3 * n3 // 2], 0.1, 4.0, 1.0)                   # 298
assert streams(s)
s.set_lorentz(nodes[:0], 0.1, 4.0, 1.0)
assert not streams(s)
s.set_materials(np.ones(n))                                               # 303
assert streams(s)
s.set_source(None)
assert streams(s)                                                         # 292
s.close()
s = box(26)                     # per-node materials 234
s.set_materials(np.ones(s.npts))
assert not streams(s)
s.close()
s = box(32)                     # 302
assert streams(s)
""")
