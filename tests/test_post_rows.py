"""Sample-row kernels at the edges of their tiling (16 lanes per row of
samples, 16 rows or 64 voxels per block): means, orientations and NODDI maps
against the oracle; predicted signal and BIC/AIC of a set of samples against
the same call on their mean alone (the mean is formed in FP64, the parameters
are then floats: a last-bit difference of a parameter moves the signal by a few
1e-7 of it, the cost by as much of its size)."""
import numpy as np
import pytest

from cudimot_amd import synth
from oracle import finish_ref as fr
from tests.helpers import ACQ, dev, host

EDGES = [(1, 1), (63, 15), (64, 16), (65, 17), (257, 33)]


def _samples(n, S, seed):
    rng = np.random.default_rng(seed)
    t = synth.truth_noddi_bingham(n, seed)
    return (t[:, :, None] * (1.0 + 0.01 * rng.normal(size=(n, t.shape[1], S)))).astype(np.float32)


@pytest.mark.gpu
@pytest.mark.parametrize("n,S", EDGES)
def test_sample_rows_match_oracle(n, S):
    import torch
    from cudimot_amd import capi
    x = _samples(n, S, 40 + S)
    d = dev(x)
    mean, dy, disp = torch.empty((n, 7), device="cuda"), torch.empty((n, 3), device="cuda"), torch.empty(n, device="cuda")
    maps = torch.empty((n, 5), device="cuda")
    capi.sample_mean(d, mean)
    capi.dyads(d, 4, 5, dy, disp, psi=6)
    capi.noddi_maps(d, 2, maps, beta=3)
    capi.sync()
    np.testing.assert_allclose(host(mean), fr.sample_mean(x), rtol=1e-6, atol=1e-7)
    wd, wdisp = fr.dyads(x, 4, 5, 6)
    np.testing.assert_allclose(np.abs(np.sum(host(dy) * wd, axis=1)), 1.0, atol=2e-5)
    np.testing.assert_allclose(host(disp), wdisp, atol=2e-6)
    np.testing.assert_allclose(host(maps), fr.noddi_maps(x, 2, 3), rtol=2e-6, atol=1e-7)


@pytest.mark.gpu
@pytest.mark.parametrize("lanes", [1, 16, 64])
@pytest.mark.parametrize("n,S", EDGES)
def test_signal_and_scores_of_samples_equal_those_of_their_mean(n, S, lanes):
    import torch
    from cudimot_amd import capi
    x = _samples(n, S, 60 + S)
    mean = x.astype(np.float64).mean(axis=2, keepdims=True).astype(np.float32)
    cfp = dev(ACQ["M99"]())
    m = capi.Model("NODDI_Bingham")
    for method in (capi.MCMC, capi.LEVMAR, capi.GRIDSEARCH):
        m.set_group(method, lanes)
    s0 = torch.full((n, 1), 1000.0, device="cuda")
    rng = np.random.default_rng(S)
    tau = np.abs(1e-3 * (1.0 + 0.05 * rng.normal(size=(n, 1, S)))).astype(np.float32)
    mtau = tau.astype(np.float64).mean(axis=2, keepdims=True).astype(np.float32)
    out = {}
    for key, p, t in (("samples", x, tau), ("mean", mean, mtau)):
        sig = torch.empty((n, 99), device="cuda")
        m.predicted_signal(dev(p), cfp, s0, sig)
        res = [sig]
        meas = out["samples"][0] + 20.0 if key == "mean" else sig + 20.0
        for rician in (False, True):
            bic, aic = torch.empty(n, device="cuda"), torch.empty(n, device="cuda")
            m.bic_aic(meas, dev(p), cfp, s0, bic, aic, rician=rician, tau_samples=dev(t) if rician else None)
            res += [bic, aic]
        capi.sync()
        out[key] = res
    for a, b in zip(out["samples"], out["mean"]):
        np.testing.assert_allclose(host(a), host(b), rtol=2e-5, atol=1e-3)
