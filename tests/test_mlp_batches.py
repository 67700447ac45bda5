"""Training steps on both sides of the largest batch that goes through the rows in
one launch (8,192): each follows the loss gradient, graph replay and eager steps
give the same weights, and a large batch takes no longer than with a network too
wide for one launch."""
import time

import numpy as np
import pytest

from tests.helpers import dev
from tests.test_mlp import bingham_truth
from tests.test_mlp_inference import _net, test_one_launch_training_step_follows_the_loss_gradient as _step

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,depth", [(256, 3), (32, 1)])
@pytest.mark.parametrize("batch", [8160, 8192, 8224, 16384])
def test_step_follows_the_loss_gradient(batch, width, depth):
    _step(99, width, depth, batch)


@pytest.mark.parametrize("batch", [8192, 8224])
def test_graph_replay_equals_eager_steps(batch):
    rng = np.random.default_rng(batch)
    x, t = dev(rng.uniform(0.1, 1.5, size=(2 * batch + 77, 40))), dev(bingham_truth(2 * batch + 77, 4))
    got = []
    for graph in (True, False):
        net = _net(40, 64, 2)
        net.set_train_graph(graph)
        net.train(x, None, t, epochs=3, batch=batch, lr=2e-3, seed=5)
        got.append(net.get_weights())
    np.testing.assert_array_equal(got[0], got[1])


def test_large_batch_takes_no_longer_than_a_wider_network():
    import torch
    n = 65536
    t = dev(bingham_truth(n, 4))
    rng = np.random.default_rng(1)

    def ms(n_in):
        x, net = dev(rng.uniform(0.1, 1.5, size=(n, n_in))), _net(n_in, 32, 3)
        best = float("inf")
        for _ in range(5):
            torch.cuda.synchronize()
            a = time.perf_counter()
            net.train(x, None, t, epochs=20, batch=n, lr=1e-3, seed=5)
            best = min(best, time.perf_counter() - a)
        return 1000 * best

    one, wider = ms(256), ms(260)  # 260 inputs: layer by layer at any batch
    assert one < 1.15 * wider, (one, wider)
