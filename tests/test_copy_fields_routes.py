"""Which way the six fields go between a caller's arrays and the library
(nkc_set_state, nkc_get_state), on the stand-in runtime: one launch where a
kernel of the current device reaches everything, copies by the runtime, with
its checks, everywhere else."""
from tests.fake_hip import fake_hip, needs_gxx  # noqa: F401

pytestmark = needs_gxx

SETUP = """
s = MaxwellSolver.from_box((2, 1, 2), 5)
n = s.npts
def get(H, E, ld=n): return s._L.nkc_get_state(s._h, H, E, None, None, ld)
def put(H, E, ld=n): return s._L.nkc_set_state(s._h, H, E, None, None, ld)
def routes():
    l = log()
    return sum("copy_fields_kernel" in x for x in l), sum(x.startswith("copy") for x in l), l[-1]
"""


def test_device_arrays_of_the_right_size_go_in_one_launch(fake_hip):  # noqa: F811
    fake_hip(SETUP + """
for ld in (n, n + 7):
    H, E = dev_array(2 * ld + n), dev_array(2 * ld + n)
    for f in (get, put):
        log()
        assert f(H, E, ld) == 0 and routes() == (1, 0, "wait 0")
""")


def test_short_arrays_are_refused_by_the_runtime(fake_hip):  # noqa: F811
    fake_hip(SETUP + """
H, E = dev_array(3 * n), dev_array(3 * n - 1)
for a, b in ((H, E), (E, H)):
    for f in (get, put):
        log()
        assert f(a, b) == _lib.NKC_ERR_HIP
        assert not any("copy_fields_kernel" in x for x in log())
""")


def test_arrays_of_another_device_are_copied_by_the_runtime(fake_hip):  # noqa: F811
    fake_hip(SETUP + """
H, E = dev_array(3 * n), dev_array(3 * n)
assert fake.hipSetDevice(1) == 0
H1, E1 = dev_array(3 * n), dev_array(3 * n)
# current device, arrays: the handle's blocks are on device 0
for dev, a, b in ((1, H1, E1), (1, H, E), (0, H1, E1), (0, H, E1), (0, H1, E)):
    fake.hipSetDevice(dev)
    for f in (get, put):
        log()
        assert f(a, b) == 0 and routes() == (0, 6, "wait 0")
fake.hipSetDevice(0)
log()
assert get(H, E) == 0 and routes()[0] == 1
""")


def test_host_arrays_are_copied_by_the_runtime(fake_hip):  # noqa: F811
    fake_hip(SETUP + """
s.set_state(np.ones((3, n)), 2 * np.ones((3, n)))
log()
H, E = s.get_state()
assert routes() == (0, 6, "wait 0")
assert (H == 1).all() and (E == 2).all()
# one of each
d = dev_array(3 * n)
log()
assert get(H.ctypes.data_as(_lib._dp), d) == 0 and routes() == (0, 6, "wait 0")
""")
