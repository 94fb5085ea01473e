"""Steps whose n-th kernel launch fails, on the stand-in runtime: what was
queued by then is ordered before what follows, and the handle's buffers and
times are those of the steps that were queued whole."""
from tests.fake_hip import fake_hip, needs_gxx  # noqa: F401

pytestmark = needs_gxx


def test_batch_joins_its_streams_after_a_failed_launch(fake_hip):  # noqa: F811
    fake_hip("""
b = BatchSolver([dict(nel=(2, 2, 2), N=N, lo=(0.,) * 3, hi=(1.,) * 3) for N in (5, 6, 7, 8)])
dt = np.full(4, 1e-3)
def put(v):
    for c in range(4):
        n = 8 * (c + 6) ** 3
        b.set_state(c, np.full((3, n), v), np.full((3, n), v))
b.step(dt, 1)
l = log()
lanes = sorted({x.split()[-1] for x in l if "box_kernel" in x})
assert len(lanes) == 3
per_step = sum("box_kernel" in x for x in l)
assert per_step == 20
for k, good in enumerate((0, 7, per_step, per_step + 3, 2 * per_step)):
    put(1.0 + k)
    fake.fake_fail_launch(good)
    log()
    try:
        b.step(dt, 3)
        assert False
    except _lib.NkcError as e:
        assert e.code == _lib.NKC_ERR_HIP
    fake.fake_fail_launch(-1)
    l = log()
    at = next(i for i, x in enumerate(l) if x.startswith("failed launch"))
    joined = set()
    for x in l[at:]:
        if x.startswith("event"):
            ev, st = x.split()[1], x.split()[-1]
        elif "waits for event" in x:
            assert x.split()[-1] == ev
            joined.add(st)
    assert joined == set(lanes), (l[at:], lanes)
    # no kernel runs here: the state read back is the one put if an even number of steps was queued whole
    H, E = b.get_state(0)
    assert (H == 1.0 + k).all() == (good // per_step % 2 == 0)
b.step(dt, 1)
""")


def test_step_keeps_its_time_after_a_failed_launch(fake_hip):  # noqa: F811
    fake_hip("""
s = MaxwellSolver.from_box((2, 2, 2), 5)
s.set_source(np.ones(s.npts) * 1e-3, (0, 0, 1.), 1.0, 0.5)
t, dt = C.c_double(0.25), 0.125
def step(n): return s._L.nkc_step(s._h, C.byref(t), dt, n)
assert step(2) == 0 and t.value == 0.5
l = launches()
assert sum("put_time" in x for x in l) == 1                       # the caller's start time
per_step = sum("put_time" not in x for x in l) // 2
assert per_step == 6                                              # stage_times and five stages
assert step(1) == 0 and not launches("put_time")                  # the device's time is current
for good, whole in ((0, 0), (1, 0), (4, 0), (per_step, 1), (2 * per_step + 3, 2)):
    t0 = t.value
    fake.fake_fail_launch(good)
    assert step(3) == _lib.NKC_ERR_HIP
    fake.fake_fail_launch(-1)
    assert t.value == t0 + whole * dt
    log()
    assert step(1) == 0 and t.value == t0 + (whole + 1) * dt
    assert len(launches("put_time")) == 1                         # put right before the next stages read it
    assert step(1) == 0 and not launches("put_time")
""")
