"""The diagnostics of a field without symmetries (a kx = 0 column that is not
Hermitian, Nyquist modes, an imaginary mean) on grids dealiased in both, one
and no direction, with plane and mode counts that leave partial workgroups,
against the oracle.  Bounds: 1e-12 for l2, energies and the flux, for the
moments 1e-10 and 1e-12 of their kind's scale (reductions in another order)."""
import numpy as np
import pytest

from helpers import make_channel, rel_l2
from oracle import chan_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz,nx2,nz2", [
    (8, 7, 12, 12, 18), (32, 33, 32, 48, 48), (36, 12, 54, 54, 81), (24, 9, 16, 24, 24), (24, 9, 16, 36, 16),
    (16, 18, 18, 16, 18), (256, 6, 48, 384, 72), (12, 40, 6, 18, 9), (324, 7, 8, 486, 12),
    (2048, 6, 4, 3072, 6), (4608, 6, 4, 4608, 4)])
def test_diagnostics(nx, ny, nz, nx2, nz2):
    g = O.make_grid(nx, ny, nz, nx2, nz2, 2.0, 2.0, 1000.0, stretch=1.5)
    rng = np.random.default_rng(nx * ny * nz)
    U = rng.standard_normal((3, ny + 1, g.nxh, nz)) + 1j * rng.standard_normal((3, ny + 1, g.nxh, nz))
    U[0, :, 0, 0] += 3.0
    ch = make_channel(g)
    ch.set_state(data1=U)
    l2, _ = ch.l2_norm()
    assert abs(l2 - O.l2_norm(g, U)) <= 1e-12 * O.l2_norm(g, U)
    assert rel_l2(ch.mode_energy(), O.mode_energy(g, U)) <= 1e-12
    q = O.mass_flux(g, U)
    assert abs(ch.mass_flux() - q) <= 1e-12 * np.abs(U[0, :, 0, 0].real * g.dyh).sum()
    M, R = ch.plane_moments(), O.plane_moments(g, U)
    for k0 in range(0, 15, 3):
        scale = np.abs(R[k0:k0 + 3]).max()
        np.testing.assert_allclose(M[k0:k0 + 3], R[k0:k0 + 3], rtol=1e-10, atol=1e-12 * scale)
    ch.close()
