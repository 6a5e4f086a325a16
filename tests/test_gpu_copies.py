"""State copies of sizes around the one above which the two halves of a
transfer overlap in pieces (8 MB, pieces of 2 MB, threads from 16 MB on): what
was set comes back, bit for bit."""
import numpy as np
import pytest

from helpers import make_channel
from oracle import chan_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz", [(64, 81, 64), (64, 82, 64), (64, 83, 64), (96, 110, 72), (128, 99, 54)])
def test_state_round_trip(nx, ny, nz):
    g = O.make_grid(nx, ny, nz, 3 * nx // 2, 3 * nz // 2, 2.0, 2.0, 1000.0, stretch=1.5)
    rng = np.random.default_rng(ny)
    U = rng.standard_normal((3, ny + 1, g.nxh, nz)) + 1j * rng.standard_normal((3, ny + 1, g.nxh, nz))
    ch = make_channel(g)
    for k in (1.0, 2.0):
        ch.set_state(data1=k * U)
        assert np.array_equal(ch.get_data1(), k * U)
    ch.close()
