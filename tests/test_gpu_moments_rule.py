"""The plane moments on both sides of the line between the fused kernel and the
points in memory for rows below 16 pairs, and at many planes, against the
oracle."""
import pytest

from test_gpu_diag_shapes import test_diagnostics as check_diagnostics

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz", [
    (16, 127, 32),    # 128 planes of two row groups: 256 workgroups, fused
    (16, 128, 32),    # 258: through memory
    (12, 300, 16),    # one row group a plane, 301 workgroups
    (24, 60, 96)])    # 8 row groups a plane
def test_moments(nx, ny, nz):
    check_diagnostics(nx, ny, nz, 3 * nx // 2, 3 * nz // 2)
