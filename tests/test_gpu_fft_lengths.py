"""Transforms and nonlinear passes at the compile-time transform lengths with
two or more factors of 3 (odd ones among them) against the oracle, and two
z-rows per wavefront where their raw rows follow each other unpadded.

Bound: single calls agree to round-off as in test_gpu_parity.py (1e-12)."""
import numpy as np
import pytest

from helpers import make_channel, rel_l2
from oracle import chan_oracle as O

pytestmark = pytest.mark.gpu

TOL = 1e-12


# x lengths nx2/2 and nx/2, z lengths nz2 and nz: every new one in each place,
# dealiased by 3/2 and not at all, plane counts that leave partial workgroups
@pytest.mark.parametrize("nx,nx2,nz,nz2", [
    (24, 36, 18, 27), (36, 54, 36, 54), (54, 108, 54, 81), (72, 108, 72, 108), (108, 162, 108, 162),
    (144, 216, 144, 216), (162, 324, 162, 243), (256, 256, 128, 128), (54, 54, 18, 18), (288, 432, 8, 12),
    (324, 486, 8, 12)])
def test_transforms(nx, nx2, nz, nz2):
    g = O.make_grid(nx, 9, nz, nx2, nz2, 2.0, 2.0, 1000.0, stretch=2.0)
    ch = make_channel(g)
    rng = np.random.default_rng(nx * 1000 + nz)

    def spec(n):
        return rng.standard_normal((n, g.nxh, g.nz)) + 1j * rng.standard_normal((n, g.nxh, g.nz))
    C = spec(3)
    assert rel_l2(ch.xz_c2r(C), O.xz_c2r(g, C)) < TOL
    f = rng.standard_normal((3, g.nz2, g.nx2))
    assert rel_l2(ch.xz_r2c(f), O.xz_r2c(g, f)) < TOL
    fl = rng.standard_normal((3, 2, g.nz2, g.nx2))
    assert rel_l2(ch.div_fluxes(*fl), O.div_fluxes(g, *fl)) < TOL
    Cs = spec(3)
    assert rel_l2(ch.small_c2r(Cs), O.small_c2r(g, Cs)) < TOL
    fs = rng.standard_normal((3, g.nz, g.nx))
    assert rel_l2(ch.small_r2c(fs), O.small_r2c(g, fs)) < TOL
    ch.close()


@pytest.mark.parametrize("lin", [False, True])
@pytest.mark.parametrize("nx,nx2,nz,nz2,rows", [
    (24, 36, 18, 27, 0), (36, 54, 36, 54, 0), (36, 54, 36, 54, 1), (72, 108, 54, 81, 0), (72, 108, 36, 54, 2),
    (108, 162, 16, 24, 0), (144, 216, 108, 162, 0), (128, 256, 16, 16, 0), (216, 324, 16, 24, 0),
    (54, 54, 18, 18, 0), (288, 432, 16, 24, 0), (324, 486, 16, 24, 0),
    (128, 192, 16, 24, 2), (192, 192, 16, 16, 2), (96, 144, 18, 24, 2), (144, 144, 18, 18, 2)])
def test_nonlinear(nx, nx2, nz, nz2, rows, lin):
    g = O.make_grid(nx, 12, nz, nx2, nz2, 4.0, 2.0, 2000.0, stretch=1.5)
    rng = np.random.default_rng(nx * 1000 + nz + lin)
    U = 0.01 * (rng.standard_normal((3, g.ny + 1, g.nxh, g.nz)) + 1j * rng.standard_normal((3, g.ny + 1, g.nxh, g.nz)))
    U[1, g.ny] = 0.0
    ch = make_channel(g)
    ch.set_tuning("xpass_rows", rows)
    ch.set_state(data1=U)
    ch.set_scalars(dt=1e-5)
    if lin:
        base = O.laminar_baseflow(g)
        ch.set_baseflow(base)
        ref, _, cflr = O.nonlinear_linearized(g, U, base, step=1, rk_step=1, dt=1e-5, return_cfl=True)
    else:
        ref, _, cflr = O.nonlinear(g, U, step=1, rk_step=1, dt=1e-5, return_cfl=True)
    _, cfl = ch.nonlinear(1, 1, linearized=lin)
    got = ch.get_data1()
    ch.close()
    assert rel_l2(got, ref) < TOL
    assert abs(cfl - cflr) < TOL * cflr
