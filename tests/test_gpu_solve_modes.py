"""Columns of more than 129 rows, whose workgroups take four modes in an order
that pairs them on one XCD: mode counts that leave a partial workgroup and
partial groups of sixteen workgroups, two steps against the sweep-based solve
(the same arithmetic up to round-off, which grows with the condition of the y
operators, as ny^2)."""
import numpy as np
import pytest

from helpers import make_channel, rel_l2, synth
from oracle import chan_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz", [(8, 130, 24), (4, 150, 6), (16, 200, 18), (12, 241, 54), (32, 242, 16)])
def test_modes_per_workgroup(nx, ny, nz):
    g = O.make_grid(nx, ny, nz, 3 * nx // 2, 3 * nz // 2, 2.0, 2.0, 2500.0, stretch=1.5, fix_mass=1)
    U0 = synth().laminar_perturbed(g.nx, g.ny, g.nz, g.yh, g.y, seed=ny, amp=1e-2, kmax=4.0)
    out = []
    for key in (1, 0):
        ch = make_channel(g)
        ch.set_tuning("solve_seg", key)
        ch.set_state(data1=U0)
        ch.set_scalars(dt=1e-3, t_total=0.0, p_grad=-2.0 / g.re)
        ch.initialize_flow()
        ch.step(2)
        out.append(ch.get_data1())
        assert ch.get_scalars()["t_total"] == 2e-3
        ch.close()
    assert np.isfinite(out[0]).all()
    assert rel_l2(out[0], out[1]) <= 1e-12 * (ny / 129.0) ** 2
