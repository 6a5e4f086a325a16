"""Rounding of the kernels that took the place of others, measured against
extended precision: no larger than the others'."""
import numpy as np
import pytest

from extended import X, error, wide, wide_grid
from helpers import make_channel, synth
from oracle import chan_oracle as O

pytestmark = pytest.mark.gpu


def test_solve_rounds_no_more_than_the_sweeps():
    """One substep of each kind at column lengths of every segment form: the
    errors of the workgroup solve over those of the sweep-based solve, in the
    geometric mean over the cases (468 modes each), at most 1 for u, v, w, the
    register and the pressure."""
    logs = []
    for ny in (33, 56, 81, 110, 129, 200):
        g = O.make_grid(24, ny, 36, 36, 54, 2.0, 2.0, 2500.0 + 10 * ny, stretch=1.5 + 0.005 * ny, fix_mass=1)
        st = O.initial_state(g, synth().laminar_perturbed(g.nx, g.ny, g.nz, g.yh, g.y, seed=ny, amp=1e-2, kmax=20.0),
                             dt=0.004)
        O.rk3_step(g, st, 1)
        wave = np.ones((g.nxh, g.nz), bool)
        wave[0, 0] = False               # all but the mean mode, whose single profile says little
        for rk in (1, 2, 3):
            st.U, _ = O.nonlinear(g, st.U, step=2, rk_step=rk, dt=st.dt)
            ref = X.State(U=wide(st.U), R=wide(st.R), P=wide(st.P), dt=wide(st.dt), p_grad=wide(st.p_grad),
                          d_um_dy=wide(st.d_um_dy))
            X.rhs_solve(wide_grid(g), ref, rk)
            assert ref.U.dtype == ref.P.dtype == np.clongdouble
            e = []
            for seg in (1, 0):
                ch = make_channel(g)
                ch.set_tuning("solve_seg", seg)
                ch.set_state(data1=st.U, data2=O.to_fortran_data2(st.R), data4=O.to_fortran_data4(st.P))
                ch.set_scalars(dt=st.dt, p_grad=st.p_grad, d_um_dy=st.d_um_dy)
                ch.rhs_solve(1, rk)
                d1, d2, d4 = ch.get_state()
                ch.close()
                R, P = O.from_fortran_data2(d2), O.from_fortran_data4(d4)
                e.append([error(d1[c][:, wave], ref.U[c][:, wave]) for c in range(3)] +
                         [error(R[:, :, wave], ref.R[:, :, wave]), error(P[:, wave], ref.P[:, wave])])
            logs.append(np.log(np.array(e[0]) / np.array(e[1])))
            O.rhs_solve(g, st, rk)
    ratio = np.exp(np.mean(logs, axis=0))
    assert (ratio <= 1.0).all(), ratio


@pytest.mark.parametrize("nx2,nz2", [(48, 18), (48, 27), (48, 54), (48, 81), (48, 108), (48, 128), (48, 162), (48, 216),
                                     (48, 243), (36, 48), (54, 48), (108, 48), (162, 48), (216, 48), (256, 48),
                                     (324, 48), (432, 48), (486, 48)])
def test_transforms_round_alike_both_ways(nx2, nz2):
    """At the lengths with two or more factors of 3 the transform to physical
    space passes the stages, sums and twiddles of the one back, and one packing
    like it: its relative error is at most a quarter more."""
    nx, nz = (2 * n // 3 if n % 3 == 0 else 3 * n // 4 for n in (nx2, nz2))
    g = O.make_grid(nx, 17, nz, nx2, nz2, 2.0, 2.0, 1000.0, stretch=2.0)
    wg = wide_grid(g)
    rng = np.random.default_rng(nx2 * 1000 + nz2)
    C = rng.standard_normal((16, g.nxh, g.nz)) + 1j * rng.standard_normal((16, g.nxh, g.nz))
    f = rng.standard_normal((16, g.nz2, g.nx2))
    ch = make_channel(g)
    back = error(ch.xz_c2r(C), X.xz_c2r(wg, wide(C)))
    forth = error(ch.xz_r2c(f), X.xz_r2c(wg, wide(f)))
    ch.close()
    assert back <= 1.25 * forth, (back, forth)
