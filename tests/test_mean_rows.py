"""Predicted signal and BIC/AIC of a set of samples against the same call on their
mean, on both sides of the sample counts at which a row of samples goes from a
thread to 16 lanes (16, with a voxel cache 18), at every lane count of the two
calls themselves (the mean is formed in FP64, the parameters are then floats: a
last-bit difference of a parameter moves the signal by a few 1e-7 of it, the cost
by as much of its size)."""
import numpy as np
import pytest

from cudimot_amd import synth
from tests.helpers import ACQ, MODEL_ACQ, dev, host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lanes", [1, 4, 16, 64])
@pytest.mark.parametrize("S", [1, 2, 15, 16, 17, 18, 19, 33])
@pytest.mark.parametrize("model,n", [("NODDI_Bingham", 261), ("Ball_2_Sticks", 67)])
def test_signal_and_scores_of_samples_equal_those_of_their_mean(model, n, S, lanes):
    import torch
    from cudimot_amd import capi
    rng = np.random.default_rng(100 * S + lanes)
    t = synth.truth_for(model, n, 20 + S)
    x = (t[:, :, None] * (1.0 + 0.01 * rng.normal(size=(n, t.shape[1], S)))).astype(np.float32)
    tau = np.abs(1e-3 * (1.0 + 0.05 * rng.normal(size=(n, 1, S)))).astype(np.float32)
    cfp = dev(ACQ[MODEL_ACQ[model]]())
    m = capi.Model(model)
    for method in (capi.PREDICTED, capi.BIC_AIC):
        m.set_group(method, lanes)
    s0 = torch.full((n, 1), 1000.0, device="cuda") if m.fixp_tsize else None
    out = []
    for p, u in ((x, tau), (x.astype(np.float64).mean(2, keepdims=True), tau.astype(np.float64).mean(2, keepdims=True))):
        sig = torch.empty((n, cfp.shape[0]), device="cuda")
        m.predicted_signal(dev(p), cfp, s0, sig)
        res = [sig]
        meas = (out[0][0] if out else sig) + 20.0
        for rician in (False, True):
            bic, aic = torch.empty(n, device="cuda"), torch.empty(n, device="cuda")
            m.bic_aic(meas, dev(p), cfp, s0, bic, aic, rician=rician, tau_samples=dev(u) if rician else None)
            res += [bic, aic]
        capi.sync()
        out.append(res)
    for a, b in zip(*out):
        np.testing.assert_allclose(host(a), host(b), rtol=2e-5, atol=1e-3)
