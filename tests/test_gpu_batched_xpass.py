"""The batched x-pass at lengths and row counts where nothing but its own
counted wait stands between the prefetch of a plane's rows and their use,
bit for bit against each member stepped alone."""
import numpy as np
import pytest

from helpers import chanflow, make_channel, synth
from oracle import chan_oracle as O

pytestmark = pytest.mark.gpu


def _member(nx, nx2, seed, rows):
    g = O.make_grid(nx, 21, 24, nx2, 36, 2.0, 2.0, 2500.0, stretch=1.5, fix_mass=1)
    ch = make_channel(g)
    ch.set_tuning("xpass_rows", rows)
    ch.set_state(data1=synth().laminar_perturbed(nx, 21, 24, g.yh, g.y, seed=seed, amp=1e-2, kmax=4.0))
    ch.set_scalars(dt=0.005, t_total=0.0, p_grad=-2.0 / g.re)
    ch.initialize_flow()
    return ch


@pytest.mark.parametrize("nx,nx2,rows", [
    (24, 32, 4),     # 16 pairs, four rows
    (48, 64, 2),     # 32 pairs, two rows
    (64, 64, 2),     # the same, undealiased in x: 33 columns a row
    (96, 128, 1),    # 64 pairs, one row
    (128, 192, 2),   # 96 pairs, whose two rows only a single channel has
    (128, 192, 4),   # and whose four rows none has
])
def test_batched_against_single(nx, nx2, rows):
    mem = [_member(nx, nx2, s, rows) for s in (1, 2)]
    twins = [_member(nx, nx2, s, rows) for s in (1, 2)]
    ens = chanflow().Ensemble(mem)
    for step in (1, 2):
        ens.step(1)
        for a, b in zip(mem, twins):
            b.step(1, step0=step)
            for x, y in zip(a.get_state(), b.get_state()):
                assert np.array_equal(x, y)
    ens.close()
    for ch in mem + twins:
        ch.close()
