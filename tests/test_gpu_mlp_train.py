"""The training kernels at their edges: batches of less than one workgroup's
64 samples, one, and a few with remainders, and workgroup counts around the
partials the reduction loads at once (32), against the numpy oracle; Adam
steps in one call against the same steps in two; more steps than the loss
buffer of a new network holds."""
import numpy as np
import pytest

from bookleaf_f90_amd import abi
from oracle import mlp as M
from tests.test_gpu_mlp import _random_norm, _random_weights

pytestmark = pytest.mark.gpu


def _net(n, seed=4):
    from bookleaf_f90_amd.device import RelaxNet
    rng = np.random.default_rng(seed)
    x = rng.normal(0, 1, (n, abi.MLP_NIN)).astype(np.float32)
    t = (x[:, 24:] + rng.normal(0, 0.1, (n, abi.MLP_NOUT))).astype(np.float32)
    net = RelaxNet(seed=0, capacity=n)
    net.add_pairs(x, t)
    return net, x, t


@pytest.mark.parametrize("n", [1, 63, 64, 65, 2047, 2048, 2049, 2113])
def test_gradient_at_the_edges_of_the_blocks(n):
    print("gradient of", n, flush=True)
    net, x, t = _net(n)
    w, norm = _random_weights(n), _random_norm(n)
    net.set_weights(w)
    net.set_norm(*norm)
    g, loss = net.gradient(n)
    ln, gn = M.loss_and_gradient(w, x, t, norm=norm)
    # a hidden activation may round to the next BF16 value (2^-8 relative) in
    # some samples: the bar of the network's other gradient tests
    assert np.max(np.abs(g - gn)) <= 2.0e-3 * np.max(np.abs(gn))
    assert abs(loss - ln) <= 1.0e-3 * abs(ln)


def test_steps_in_one_call_are_the_steps_of_two():
    """Adam's step count and moments carry over; every step draws by its
    place in its own call, so the second call's seed differs."""
    one, _, _ = _net(500)
    two, _, _ = _net(500)
    w = _random_weights(9)
    for net in (one, two):
        net.set_weights(w)
    a = one.train(5, batch=100, lr=1e-3, seed=3)
    b = two.train(5, batch=100, lr=1e-3, seed=3)
    assert np.array_equal(a, b) and np.array_equal(one.weights(), two.weights())
    assert np.array_equal(one.train(0, batch=100), np.empty(0, np.float32))
    assert np.array_equal(one.train(3, batch=65, seed=4), two.train(3, batch=65, seed=4))
    assert np.array_equal(one.weights(), two.weights())


def test_more_steps_than_the_first_loss_buffer():
    net, _, _ = _net(300)
    h = net.train(4100, batch=64, lr=1e-4, seed=1)
    assert h.shape == (4100,) and np.all(np.isfinite(h)) and np.all(h > 0.0)
    assert np.mean(h[-200:]) < np.mean(h[:200])
