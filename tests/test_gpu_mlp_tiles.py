"""The training kernels of the closure network at the edges of their 16-point
tiles and of the 256 workgroups that share them, against the float64
restatement."""
import numpy as np
import pytest

from helpers import chanflow
from oracle import les_oracle as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 4096, 4097, 8200])
def test_tile_edges(n):
    """One point, a tile less one, whole and plus one, every workgroup with one
    tile, one of them with two, and three rounds with a ragged end.  Float32
    sums of at most a few hundred terms: relative errors of some 1e-6."""
    rng = np.random.default_rng(n)
    W, b = L.init_params(n)
    X = rng.standard_normal((n, 10)).astype(np.float32)
    T = rng.standard_normal((n, 6)).astype(np.float32)
    net = chanflow().Mlp(chanflow().Mlp.flatten(W, b))
    ref = L.forward(W, b, X)
    assert np.abs(net.forward(X) - ref).max() <= 1e-5 * np.abs(ref).max()
    g, loss = net.gradient(X, T)
    gref = chanflow().Mlp.flatten(*L.backward(W, b, X, T)).astype(np.float64)
    assert np.linalg.norm(g - gref) <= 1e-5 * np.linalg.norm(gref)
    assert abs(loss - L.mse(ref, T)) <= 1e-5 * L.mse(ref, T)
    # one Adam step moves every parameter with a gradient by lr (its first
    # step is lr g / (|g| + eps)); a second call continues from the first
    p0 = net.get_params()
    assert net.train(X, T, epochs=1, batch=n, lr=1e-3) == pytest.approx(loss, rel=1e-6)
    moved = net.get_params() - p0
    big = np.abs(gref) > 1e-3 * np.abs(gref).max()
    assert np.allclose(moved[big], -1e-3 * np.sign(gref[big]), rtol=1e-3, atol=1e-7)
    net.close()
