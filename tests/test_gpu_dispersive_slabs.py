"""Slabs of more elements than CUs: N = 9 with a dispersive region, three and
two slabs at the ends of their ranges, against whole elements (the tolerance
and its reasons are test_gpu_stage_slabs')."""
import pytest

from tests.test_gpu_stage_slabs import test_slabs_equal_whole_elements as _slabs_equal_whole_elements

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("small", [(3, 1, 43), (5, 5, 8), (3, 1, 67), (8, 4, 11), (353, 1, 1)])
def test_many_slabs_equal_whole_elements(small):
    _slabs_equal_whole_elements(9, small, "dispersive")
