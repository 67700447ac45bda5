"""The sum of squares behind MCMC and BIC/AIC at the edges of its blocks of four
measurements per lane: BIC of a Gaussian fit at measurement counts around the
multiples of 4 L against FP64 sums over the predicted signal (a float, whose
rounding of 6e-8 moves a residual of its own size by as much)."""
import numpy as np
import pytest

from cudimot_amd import synth
from tests.helpers import dev, host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lanes", [1, 4, 16, 64])
@pytest.mark.parametrize("nmeas", [1, 3, 4, 5, 15, 16, 17, 31, 63, 64, 65, 127, 128, 255, 256, 257, 271, 511, 512, 515])
def test_bic_at_block_edges(nmeas, lanes):
    import torch
    from cudimot_amd import capi
    n = 70
    rng = np.random.default_rng(nmeas)
    cfp = np.concatenate([synth.unit_sphere(rng, nmeas), rng.uniform(200.0, 3000.0, (nmeas, 1))], 1)
    t = synth.truth_ball_1_stick(n, 7)
    m = capi.Model("Ball_1_Stick")
    m.set_group(capi.BIC_AIC, lanes)
    s = dev(t).reshape(n, -1, 1)
    sig = torch.empty((n, nmeas), device="cuda")
    m.predicted_signal(s, dev(cfp), None, sig)
    meas = sig + 30.0 * torch.randn(sig.shape, device="cuda", generator=torch.Generator(device="cuda").manual_seed(3))
    bic, aic = torch.full((n,), -1.0, device="cuda"), torch.full((n,), -1.0, device="cuda")
    m.bic_aic(meas, s, dev(cfp), None, bic, aic)
    capi.sync()
    sse = ((host(sig) - host(meas)) ** 2).sum(1)
    nll = 0.5 * nmeas * np.log(0.5 * sse)
    np.testing.assert_allclose(host(bic), 2 * nll + 5 * np.log(nmeas), rtol=2e-6, atol=1e-3)
    np.testing.assert_allclose(host(aic), 2 * nll + 10, rtol=2e-6, atol=1e-3)
