"""The longest column that the workgroup solve takes and the first that goes to
the sweeps."""
import pytest

from test_gpu_solve_segments import test_segment_edges as check_column

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ny", [269, 270])
def test_longest_column(ny):
    check_column(ny, 1)
