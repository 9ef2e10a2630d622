"""Warm-start MLP training at the edges of its tiles: batches around one
16-sample tile, a workgroup's four tiles and the reduction's sixteen partials,
and the packed weights and data buffers that a network keeps between calls.
Tolerances as in test_gpu_mlp.py."""
import numpy as np
import pytest

from oracle import mlp_ref as M
from tests.test_gpu_mlp import TENSORS, random_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 17, 63, 64, 65, 1023, 1025, 1089])
def test_gradients_at_tile_edges(bbx, n):
    rng = np.random.default_rng(100 + n)
    p = random_params(1)
    net = bbx.Mlp(1)
    net.set_params(p)
    x = rng.normal(size=(n, M.F)).astype(np.float32)
    t = rng.normal(size=n).astype(np.float32)
    g, loss = net.gradients(x, t)
    lref, gref = M.loss_and_grad(p, x, t, emulate=True)
    assert loss == pytest.approx(lref, rel=1e-4)
    for name, (a, b) in TENSORS.items():
        scale = np.abs(gref[a:b]).max()
        assert np.abs(g[a:b] - gref[a:b]).max() <= 2e-3 * scale + 1e-9, name


def test_packed_weights_follow_the_parameters(bbx):
    """After training, gradients are those of a new network with the same
    parameters, bit for bit; a second, smaller training set in the kept
    buffers trains as it does in new ones."""
    rng = np.random.default_rng(3)
    x = rng.normal(size=(5000, M.F)).astype(np.float32)
    t = np.tanh(x[:, 0]).astype(np.float32)
    a = bbx.Mlp(0)
    a.set_params(random_params(4))
    a.train(x, t, steps=7, batch=333)
    b = bbx.Mlp(0)
    b.set_params(a.get_params())
    ga, la = a.gradients(x[:500], t[:500])
    gb, lb = b.gradients(x[:500], t[:500])
    assert np.array_equal(ga, gb) and la == lb
    a.set_params(random_params(5))
    b.set_params(random_params(5))
    assert a.train(x[:77], t[:77], steps=5, batch=100) == b.train(x[:77], t[:77], steps=5, batch=100)
    assert np.array_equal(a.get_params(), b.get_params())
