"""Graphene sheets at the orders test_gpu_graphene does not take, against the
oracle: the face nodes are dealt to lanes differently at N = 3, and elements go
to the XCDs in ranges of equal work; with a mesh of many rounds of workgroups
for the latter.

Tolerance: that of test_gpu_graphene (1e-11 relative, the sums differ in their
order only).
"""
import pytest

from tests.test_gpu_graphene import _planes, _rel
from tests.test_gpu_parity import parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,nel", [(3, (4, 3, 4)), (3, (14, 12, 14)), (5, (4, 3, 4)), (6, (4, 3, 4)), (8, (4, 3, 4)),
                                   (9, (4, 3, 4))])
def test_sheet_planes(oracle, N, nel):
    s, ref, H, E, G0, _ = _planes(oracle, N=N, nel=nel)
    s.step(0.002, 10)
    gH, gE = s.get_state()
    out = ref.run(H, E, 0.002, 10, G=G0)
    assert parity(gH, gE, out["H"], out["E"], ref.bm1) <= 1e-11
    assert _rel(s.get_graphene("state"), out["G"]) <= 1e-11
    assert _rel(s.get_graphene("register"), out["kG"]) <= 1e-11
    s.close()
