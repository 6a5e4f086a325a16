"""What a batched ensemble and the subgrid closure refuse, and that the message
says what they take; the diagnostics of a grid that no transform fits."""
import pytest

from helpers import chanflow, make_channel
from oracle import chan_oracle as O

pytestmark = pytest.mark.gpu

LENGTHS = "16, 24, 32, 36, 48, 64, 72, 96, 144, 192"


def _channel(nx=32, ny=33, nz=32):
    return make_channel(O.make_grid(nx, ny, nz, 3 * nx // 2, 3 * nz // 2, 2.0, 2.0, 2500.0, stretch=1.5, fix_mass=1))


@pytest.mark.parametrize("size,message", [
    (dict(nx=36), "nx2/2 is none of " + LENGTHS),
    (dict(nz=36), "nz2 is none of " + LENGTHS + ", 288"),
    (dict(ny=150), "ny.1 rows do not make 5 to 9 in each of at most 16 segments, 3 or more in the last")])
def test_ensemble(size, message):
    ch = _channel(**size)
    with pytest.raises(chanflow().ChanError, match=message):
        chanflow().Ensemble([ch])
    ch.close()


def test_closure():
    ch = _channel(nx=36)
    with pytest.raises(chanflow().ChanError, match="needs the wavefront x-pass and nx2/2 one of " + LENGTHS):
        ch.les_configure("dynamic")
    ch.close()


@pytest.mark.parametrize("nz", [512, 486])
def test_norm_of_a_grid_without_transforms(nz):
    """The l2 norm needs no transform, but nothing else works on these grids."""
    ch = _channel(ny=9, nz=nz)
    for call in (ch.l2_norm, ch.initialize_flow, lambda: ch.step(1)):
        with pytest.raises(chanflow().ChanError, match="FFT batch too large for workgroup"):
            call()
    ch.close()
