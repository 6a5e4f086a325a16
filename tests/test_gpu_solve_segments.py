"""The workgroup form of the segmented column solve at the edges of its shapes
(rows per segment, padding rows, mode counts that do not fill the last
workgroup) against the oracle's rhs_solve."""
import numpy as np
import pytest

from helpers import make_channel, rel_l2, synth
from oracle import chan_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ny,key", [
    (8, 1),      # 3 segments of 3 rows
    (9, 1),      # 10 rows: 4 per segment, padding in the first and in the last
    (10, 1),     # 11 rows: 4 per segment, padding in the last only
    (10, 2),     # 3 segments of 5, 4 padding rows: 2 in each of the outer segments
    (12, 1),     # 13 rows: 5 per segment, 2 padding rows in the last
    (81, 1),     # 82 rows in 21 segments of 4
    (98, 1),     # 99 rows in 25 segments of 4 (33 of 3 would take more than 256 threads)
    (128, 2),    # 129 rows, 1 padding row
    (130, 1),    # 131 rows, 4 padding rows
    (200, 1),    # 201 rows: six wavefronts
    (279, 1),    # the longest column that fits a workgroup's LDS
    (280, 1),    # one row more: the sweep-based solve
])
def test_segment_edges(ny, key):
    """7 x 18 = 126 modes (15 full workgroups and one of 6), three substeps
    with wall data on both walls, a perturbed register and a pressure whose
    mean mode is not zero (it must not matter).  The bound grows with the
    condition of the y operators, as ny^2."""
    g = O.make_grid(12, ny, 18, 18, 27, 2.0, 2.0, 2500.0, stretch=1.5, fix_mass=1, dt_flag=0)
    grow = max(1.0, (ny / 129.0) ** 2)
    rng = np.random.default_rng(1000 + ny)
    U0 = synth().laminar_perturbed(g.nx, g.ny, g.nz, g.yh, g.y, seed=ny, amp=1e-2, kmax=4.0)
    st = O.initial_state(g, U0, dt=0.01)

    def noise(shape):
        return 1e-3 * (rng.standard_normal(shape) + 1j * rng.standard_normal(shape))
    cbc_top, cbc_bot = noise((3, g.nxh, g.nz)), noise((3, g.nxh, g.nz))
    cbc_top[:, 0, 0] = cbc_top[:, 0, 0].real
    cbc_bot[:, 0, 0] = cbc_bot[:, 0, 0].real
    for rk in (1, 2, 3):
        print(f"ny {ny} key {key} substep {rk}", flush=True)
        s0 = st.copy()
        s0.U, _ = O.nonlinear(g, st.U, step=1, rk_step=rk, dt=0.01)
        s0.R = s0.R + noise(s0.R.shape)
        s0.R[1, g.ny] = 0.0
        s0.P = s0.P.copy()
        s0.P[:, 0, 0] = 0.3 + rng.standard_normal(g.ny + 1)
        s0.cbc_top, s0.cbc_bot = cbc_top, cbc_bot
        ch = make_channel(g)
        ch.set_tuning("solve_seg", key)
        ch.set_state(data1=s0.U, data2=O.to_fortran_data2(s0.R), data4=O.to_fortran_data4(s0.P))
        ch.set_scalars(dt=s0.dt, p_grad=s0.p_grad, d_um_dy=s0.d_um_dy)
        ch.set_wall_bc(cbc_top, cbc_bot)
        ch.rhs_solve(1, rk)
        (d1, d2, d4), sc = ch.get_state(), ch.get_scalars()
        ch.close()
        ref = O.rhs_solve(g, s0.copy(), rk)
        assert rel_l2(d1, ref.U) <= 1e-12 * grow
        assert rel_l2(d2, O.to_fortran_data2(ref.R)) <= 1e-12 * grow
        assert rel_l2(d4, O.to_fortran_data4(ref.P)) <= 1e-11 * grow
        assert rel_l2(sc["d_um_dy"], ref.d_um_dy) <= 1e-12 * grow
        assert abs(sc["p_grad"] - ref.p_grad) <= 1e-12 * abs(ref.p_grad)
