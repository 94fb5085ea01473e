"""Into how many slabs a small mesh's elements go, from the instances and grids
launched on the stand-in runtime: N = 9 with and without a dispersive region."""
from tests.fake_hip import fake_hip, needs_gxx  # noqa: F401

pytestmark = needs_gxx


def test_slabs_at_n9(fake_hip):  # noqa: F811
    fake_hip("""
def slabs(s):
    log()
    s.step(1e-3, 1)
    l = launches("box_kernel")[0]
    sl = int(l.split("box_kernel<")[1].split(">")[0].split(", ")[6])
    assert int(l.split("grid ")[1].split()[0]) == sl * 8 * ((s.mesh.nelt + 7) // 8), l
    return sl
for nelt, plain, dispersive in ((51, 5, 5), (85, 3, 3), (128, 2, 2), (129, 1, 3), (200, 1, 3), (201, 1, 2), (352, 1, 2),
                                (353, 1, 1), (512, 1, 1)):
    s = MaxwellSolver.from_box((nelt, 1, 1), 9)
    assert slabs(s) == plain, nelt
    s.set_source(np.full(s.npts, 1e-3), (0, 0, 1.), 1.0, 0.5)
    assert slabs(s) == plain, nelt
    s.set_drude(np.arange(1000), 0.1, 4.0)
    assert slabs(s) == dispersive, nelt
    s.set_drude(np.arange(0), 0.1, 4.0)
    assert slabs(s) == plain, nelt
    s.set_lorentz(np.arange(1000), 0.1, 4.0, 1.0)
    assert slabs(s) == dispersive, nelt
    s.close()
""")
