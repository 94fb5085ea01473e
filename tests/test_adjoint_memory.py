"""What memory the adjoint holds, and when, on the stand-in runtime: a dropped
trajectory is freed at once, or taken over by the next forward inside a pass
that asks for it, and never counts against another handle."""
from tests.fake_hip import fake_hip, needs_gxx  # noqa: F401

pytestmark = needs_gxx

SETUP = """
def solver(): return MaxwellSolver.from_box((3, 2, 2), 5, (0.,) * 3, (1.,) * 3, ("PEC",) * 3)
def forward(s, steps=8): s.adjoint_forward(1e-3, steps, 4)
def used(): return fake.fake_used(0)
s = solver()
n = s.npts
drops = [lambda s: s.set_materials(np.ones(n)), lambda s: s.set_source(np.ones(n), (0, 0, 1.), 1.0, 0.5),
         lambda s: s._L.nkc_set_source_time(s._h, 0, 0.0, 0.0), lambda s: s.set_drude(np.arange(216), 0.3, 4.0)]
for d in drops: d(s)         # the tables these calls make are there from now on
base = used()
"""


def test_a_dropped_trajectory_is_freed_at_once(fake_hip):  # noqa: F811
    fake_hip(SETUP + """
for d in drops:
    forward(s)
    assert used() > base + 8 * 6 * n * 40 and s.adjoint_info()["bytes"] == used() - base
    d(s)
    assert used() == base and s.adjoint_info()["bytes"] == 0
""")


def test_a_pass_takes_over_the_buffers(fake_hip):  # noqa: F811
    fake_hip(SETUP + """
forward(s)
held = used() - base
for d in drops:
    with s.adjoint_buffers_kept():
        d(s)
        assert used() == base + held and s.adjoint_info()["bytes"] == held
        forward(s)
        assert used() == base + held
    assert used() == base + held
# other sizes: what the forward has no use for is freed
with s.adjoint_buffers_kept():
    drops[0](s)
    forward(s, 3)
assert used() - base == s.adjoint_info()["bytes"] < held
# no forward: nothing waits past the end, whatever ends it
for error in (False, True):
    forward(s)
    try:
        with s.adjoint_buffers_kept():
            drops[0](s)
            assert used() == base + held
            if error: raise ValueError
    except ValueError:
        pass
    assert used() == base and s.adjoint_info()["bytes"] == 0
for give_back in (lambda s: s.adjoint_release(), lambda s: s.close()):
    with s.adjoint_buffers_kept():
        forward(s)
        drops[0](s)
        assert used() == base + held
        give_back(s)
        assert used() <= base
        if not s._h: break
""")


def test_the_harness_asks_for_it(fake_hip):  # noqa: F811
    fake_hip("""
sys.modules["torch"] = None
""" + SETUP + """
from nekcem_amd import adjoint
from nekcem_amd.adjoint import DrudeProbeProblem, ProbeProblem
common = dict(solver=s, H0=np.zeros((3, n)), E0=np.zeros((3, n)), dt=1e-3, nsteps=8, every=4, probes=np.arange(3))
for run in (lambda: adjoint._run_forward(ProbeProblem(**common), np.ones(n), np.ones(n)),
            lambda: adjoint._run_forward_drude(DrudeProbeProblem(dindex=np.arange(216), owner=np.zeros(216, int),
                                                                 **common), np.ones(1), np.ones(1))):
    run()
    held = used()
    free = s._L.nkc_set_materials
    log()
    run()
    assert used() == held
    drops[0](s)
    assert used() == base
""")


def test_waiting_buffers_do_not_count_against_another_handle(fake_hip):  # noqa: F811
    fake_hip("""
def solver(): return MaxwellSolver.from_box((3, 3, 3), 5, (0.,) * 3, (1.,) * 3, ("PEC",) * 3)
a, b = solver(), solver()
n = a.npts
a.set_materials(np.ones(n)); b.set_materials(np.ones(n))
# the memory decides how many segments keep their stages
fake.fake_set_capacity(0, fake.fake_used(0) + 8 * 6 * n * 400)
def plan(s):
    s.adjoint_forward(1e-3, 20, 4)
    i = s.adjoint_info()
    return i["window"], i["kept"]
alone = plan(a)
assert alone[0] == 4 and 1 < alone[1] < 5
a.adjoint_release()
b.adjoint_set_grads(False)
b.adjoint_forward(1e-3, 16, 16)
held = b.adjoint_info()["bytes"]
assert held > 8 * 6 * n * 80        # half of it: a segment's stages
with b.adjoint_buffers_kept():
    b.set_materials(np.ones(n))
    assert b.adjoint_info()["bytes"] == held      # waits
    assert plan(a) == alone
""")
