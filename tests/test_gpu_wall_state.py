"""The wall data that steps, substeps and replays leave for each other: a jet
without forcing keeps its profile from substep to substep and a step without
jet and feedback clears nothing that is zero already, so every order of the
calls that write the wall data is compared, bit for bit, with one that writes
them anew each time (a jet whose forcing is too small to change it)."""
import numpy as np
import pytest

from helpers import chanflow, grid_cfg0, init_cfg0, make_channel
from oracle import chan_oracle as O

pytestmark = pytest.mark.gpu


def _channel(g, forcing=None):
    ch = make_channel(g)
    ch.set_state(data1=init_cfg0(O, g))
    ch.set_scalars(dt=0.004, t_total=0.0, p_grad=-2.0 / g.re)
    if forcing is not None:
        ch.jet_configure(0, 0.1, 0.3, 0.25 * g.lx, 0.5 * g.lz, forcing, 1.0)
    ch.initialize_flow()
    return ch


def _same(a, b):
    for x, y in zip(a.get_state(), b.get_state()):
        assert np.array_equal(x, y)
    assert a.get_scalars()["t_total"] == b.get_scalars()["t_total"]


@pytest.mark.parametrize("gain", [0.0, 0.5])
def test_steady_jet(gain):
    g = grid_cfg0(O, ctrlu=gain)
    a, b = _channel(g, 0.0), _channel(g, 1e-300)
    rng = np.random.default_rng(4)
    w = 1e-3 * rng.standard_normal((3, g.nxh, g.nz)) + 0j
    for order in ("step", "walls rhs step", "boundary off rhs", "step on step", "boundary walls off rhs", "step"):
        for op in order.split():
            print(order, op, flush=True)
            for ch, f in ((a, 0.0), (b, 1e-300)):
                if op == "step":
                    ch.step(2)
                elif op == "walls":
                    ch.set_wall_bc(w, None)
                elif op == "rhs":
                    ch.nonlinear(1, 2)
                    ch.rhs_solve(1, 2)
                elif op == "boundary":
                    ch.boundary()
                else:
                    ch.jet_configure(0, 0.1 if op == "on" else 0.0, 0.3, 0.25 * g.lx, 0.5 * g.lz, f, 1.0)
            _same(a, b)
    a.close(); b.close()


@pytest.mark.parametrize("nstreams", [0, 1])
def test_replays_clear_the_walls(nstreams):
    """Wall data set, or left by a direct step with a jet configured after the
    capture, do not reach a replay; no replay at all leaves a direct step right."""
    cf = chanflow()
    g = grid_cfg0(O)
    a, b = _channel(g), _channel(g)
    ens = cf.Ensemble([a], nstreams=nstreams)
    ens.step(0)
    rng = np.random.default_rng(5)
    w = 1e-3 * rng.standard_normal((3, g.nxh, g.nz)) + 0j
    for jet in (False, True):
        a.set_wall_bc(w, w)
        ens.step(2); b.step(2)
        _same(a, b)
        if not jet:
            a.set_wall_bc(w, w)
            a.step(1); b.step(1)
            _same(a, b)
            for ch in (a, b):
                ch.jet_configure(0, 0.1, 0.3, 0.25 * g.lx, 0.5 * g.lz, 0.0, 1.0)
                ch.step(1)
            b.jet_configure(0, 0.0, 0.3, 0.0, 0.0, 0.0, 1.0)
    ens.close(); a.close(); b.close()


def test_replayed_jet():
    cf = chanflow()
    g = grid_cfg0(O)
    a, b = _channel(g, 0.0), _channel(g, 0.0)
    ens = cf.Ensemble([a], nstreams=1)
    ens.step(0)
    a.step(1); b.step(1)
    _same(a, b)
    for _ in range(2):
        a.set_wall_bc(np.full((3, g.nxh, g.nz), 1e-3 + 0j), None)
        ens.step(2); b.step(2)
        _same(a, b)
        a.step(1); b.step(1)
        _same(a, b)
    ens.close(); a.close(); b.close()
