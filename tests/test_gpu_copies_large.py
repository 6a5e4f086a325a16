"""State copies that take all four copying threads (48 MB and more) and pieces
above 2 MB (beyond 64 of them, 128 MB), the last one short: what was set comes
back, bit for bit."""
import numpy as np
import pytest

from helpers import make_channel
from oracle import chan_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz", [(192, 129, 108), (216, 160, 162)])
def test_state_round_trip(nx, ny, nz):
    g = O.make_grid(nx, ny, nz, 3 * nx // 2, 3 * nz // 2, 2.0, 2.0, 1000.0, stretch=1.5)
    U = np.empty((3, ny + 1, g.nxh, nz), np.complex128)
    assert U.nbytes > 48 << 20 and U.nbytes % (4 << 20)
    U.view(np.float64)[:] = np.random.default_rng(ny).random(U.view(np.float64).shape)
    ch = make_channel(g)
    for k in (1.0, 2.0):
        ch.set_state(data1=k * U)
        assert np.array_equal(ch.get_data1(), k * U)
    ch.close()
