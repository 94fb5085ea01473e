"""What ProbeFields and DrudeProbeFields hand the library for a list of
probes, on the CPU: a stand-in library reads the node lists and the seeds from
the addresses it is given, after filling memory that was freed by then.  Lists
that are contiguous, strided (a slice, a column of a table), repeated, and
edited in place between passes must give the fields and seeds that indexing by
the list gives."""
import contextlib
import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from nekcem_amd.adjoint import DrudeProbeFields, DrudeProbeProblem, ProbeFields, ProbeProblem  # noqa: E402

NPTS = 5000
FIELDS = np.random.default_rng(0).standard_normal((6, NPTS))


def _read(p, n, dtype):
    # whatever was freed before this call is taken and overwritten first
    scrap = [torch.full((n,), -1, dtype=torch.long) for _ in range(64)]
    a = np.ctypeslib.as_array(C.cast(p, C.POINTER(C.c_int64 if dtype is np.int64 else C.c_double)), (n,)).copy()
    del scrap
    return a


class _Library:
    """Every call returns 0; the two that take a node list keep what they read."""

    def __init__(self):
        self.seeds = None

    def __getattr__(self, name):
        return lambda *a: 0

    def nkc_get_state_at(self, h, n, nodes, out):
        listed = _read(nodes, n, np.int64)
        if listed.min() < 0 or listed.max() >= NPTS:
            return 1
        np.ctypeslib.as_array(out, (6 * n,))[:] = FIELDS[:, listed].reshape(-1)
        return 0

    def nkc_adjoint_backward_at(self, h, n, nodes, seeds, geps, gmu):
        listed, s = _read(nodes, n, np.int64), _read(seeds, 6 * n, np.float64).reshape(6, n)
        self.seeds = np.zeros((6, NPTS))
        np.add.at(self.seeds, (slice(None), listed), s)
        return 0


class _Solver:
    npts, _h = NPTS, None

    def __init__(self):
        self._L = _Library()

    def adjoint_buffers_kept(self):
        return contextlib.nullcontext()

    def __getattr__(self, name):
        return lambda *a, **k: None


RNG = np.random.default_rng(1)
LISTS = {
    "contiguous": lambda: RNG.choice(NPTS, 64, replace=False),
    "slice": lambda: RNG.choice(NPTS, 2000, replace=False)[::2],
    "column": lambda: RNG.choice(NPTS, (64, 3))[:, 1],
    "repeated": lambda: np.repeat(RNG.choice(NPTS, 40), 3)[::2],
    "one": lambda: RNG.choice(NPTS, (4, 2))[:1, 1],
}


def _pass(kind, problem, s):
    if kind == "material":
        x = [torch.ones(NPTS, dtype=torch.float64, requires_grad=True) for _ in range(2)]
        out = ProbeFields.apply(*x, problem)
    else:
        x = [torch.ones(2, dtype=torch.float64, requires_grad=True) for _ in range(2)]
        out = DrudeProbeFields.apply(*x, problem)
    g = torch.randn(out.shape, dtype=torch.float64)
    torch.autograd.grad(out, x, g)
    want = np.zeros((6, NPTS))
    np.add.at(want, (slice(None), problem.probes), g.numpy())
    assert np.array_equal(out.detach().numpy(), FIELDS[:, problem.probes])
    assert np.allclose(s._L.seeds, want, rtol=0, atol=1e-14 * np.abs(want).max())


def _problem(kind, s, probes):
    common = dict(solver=s, H0=np.zeros((3, NPTS)), E0=np.zeros((3, NPTS)), dt=0.1, nsteps=2, every=1, probes=probes)
    if kind == "material":
        return ProbeProblem(**common)
    return DrudeProbeProblem(dindex=np.arange(6), owner=np.array([0, 0, 0, 1, 1, 1]), **common)


@pytest.mark.parametrize("kind", ["material", "drude"])
@pytest.mark.parametrize("name", LISTS)
def test_fields_and_seeds_of_a_list(name, kind):
    s = _Solver()
    problem = _problem(kind, s, LISTS[name]())
    for _ in range(2):
        _pass(kind, problem, s)


@pytest.mark.parametrize("name", ["contiguous", "column"])
def test_a_list_edited_in_place(name):
    s = _Solver()
    problem = _problem("material", s, LISTS[name]())
    _pass("material", problem, s)
    problem.probes[:] = RNG.choice(NPTS, len(problem.probes), replace=False)
    _pass("material", problem, s)
