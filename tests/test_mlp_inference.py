"""Network inference in one launch (layers of at most 256 inputs and units)
against the layer-by-layer form, at the edges of its blocks of 64 rows, of the
64-column input runs and of the 32-unit tiles.  The layer-by-layer form is
reached by the same network with its inputs padded to 260 columns of zero
weight: the same products in the same order, so equal bits; and against the
oracle."""
import numpy as np
import pytest

from oracle import mlp_ref as R
from tests.helpers import dev, host
from tests.test_mlp import BINGHAM_HEAD


def _net(n_in, width, depth):
    from cudimot_amd import capi
    head = [capi.head_entry(e["kind"], e["param"], e["param2"], e["lo"], e["hi"], e["weight"], e["vmin"], e["vmax"])
            for e in BINGHAM_HEAD]
    return capi.Mlp(n_in, head, width=width, depth=depth, seed=3)


@pytest.mark.gpu
@pytest.mark.parametrize("n,n_in,width,depth", [(1, 99, 256, 3), (32, 64, 128, 2), (33, 65, 32, 1), (63, 256, 96, 7),
                                                (65, 1, 160, 2), (1000, 129, 256, 1), (70001, 99, 224, 3)])
def test_one_launch_equals_layer_by_layer(n, n_in, width, depth):
    import torch
    from cudimot_amd import capi
    net, wide = _net(n_in, width, depth), _net(260, width, depth)
    w = net.get_weights()
    first = np.zeros((width, 260), dtype=np.float32)
    first[:, :n_in] = w[:width * n_in].reshape(width, n_in)
    wide.set_weights(np.concatenate([first.ravel(), w[width * n_in:]]))
    rng = np.random.default_rng(n)
    x = rng.uniform(50.0, 1500.0, size=(n, n_in)).astype(np.float32)
    xw = np.zeros((n, 260), dtype=np.float32)
    xw[:, :n_in] = x
    scale = rng.uniform(800.0, 1200.0, size=n).astype(np.float32)
    res = []
    for m, inp in ((net, x), (wide, xw)):
        out, params = torch.empty((n, m.n_out), device="cuda"), dev(np.full((n, 7), 1.5))
        m.forward(dev(inp), dev(scale), out)
        m.init_params(dev(inp), dev(scale), params)
        capi.sync()
        res.append((host(out), host(params)))
    np.testing.assert_array_equal(res[0][0], res[1][0])
    np.testing.assert_array_equal(res[0][1], res[1][1])
    ref, _ = R.forward(R.unflatten(w, net.layer_shapes()), x[-200:] / scale[-200:, None], bf16=True)
    assert np.abs(res[0][0][-200:] - ref).max() / np.abs(ref).max() < 1e-2


@pytest.mark.gpu
@pytest.mark.parametrize("n_in,width,depth,batch", [(99, 256, 3, 2048), (64, 32, 1, 32), (256, 96, 7, 96),
                                                    (33, 160, 2, 64)])
def test_one_launch_training_step_follows_the_loss_gradient(n_in, width, depth, batch):
    """One step (one batch, hardly any noise) against the loss and gradient of
    the layer-by-layer launches at the same weights: Adam's first step is
    -lr g / (|g| + 1e-8), so -lr sign(g) to 0.1% where |g| > 1e-5.  An input
    that the residual noise moves over a BF16 rounding boundary (2^-9 of it)
    can turn the sign of a gradient near zero only."""
    from cudimot_amd import capi
    from tests.test_mlp import bingham_truth
    net = _net(n_in, width, depth)
    rng = np.random.default_rng(batch)
    x = rng.uniform(0.1, 1.5, size=(batch, n_in)).astype(np.float32)
    t = dev(bingham_truth(batch, 4))
    w0 = net.get_weights()
    loss, g = net.loss_grad(dev(x), None, t)
    lr = 1e-3
    losses = net.train(dev(x), None, t, epochs=1, batch=batch, lr=lr, seed=1, snr=(1e9, 1e9))
    step = (net.get_weights().astype(np.float64) - w0) / lr
    assert abs(losses[0] - loss) <= 1e-4 * abs(loss), (losses, loss)
    big = np.abs(g) > 1e-5
    assert big.any()
    close = np.abs(step[big] + np.sign(g[big])) < 2e-3 + 2.0 ** -22 * np.abs(w0[big]) / lr
    assert close.mean() > 0.999, close.mean()
