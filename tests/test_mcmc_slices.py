"""MCMC over volumes of more blocks than the GPU holds at once, which run in
time slices from a queue: each voxel's chain is the one it has in a smaller
volume (its draws are addressed by its index), so the whole call equals calls
over parts of it, bit for bit."""
import pytest

from tests import helpers as H


@pytest.mark.gpu
@pytest.mark.parametrize("model,n,lanes,rician,chain", [("Ball_1_Stick", 20001, 64, False, (7, 33, 3)),
                                                        ("Ball_1_Stick", 20001, 64, False, (1, 16, 1)),
                                                        ("Ball_1_Stick", 20001, 64, True, (10, 30, 5)),
                                                        ("NODDI_Bingham", 9002, 64, False, (10, 30, 5))])
def test_whole_volume_equals_its_parts(model, n, lanes, rician, chain):
    import torch
    from cudimot_amd import capi, synth
    nb, nj, se = chain
    cfp = H.dev(H.ACQ[H.MODEL_ACQ[model]]())
    t = H.dev(synth.clip_to_bounds(model, H.truth(model, 500, 9))).repeat(n // 500 + 1, 1)[:n].contiguous()
    m = capi.Model(model)
    m.set_group(capi.MCMC, lanes)
    fixp = torch.full((n, 1), 1000.0, device="cuda") if m.fixp_tsize else None
    meas = torch.empty((n, cfp.shape[0]), device="cuda")
    m.predicted_signal(t.float().reshape(n, -1, 1).contiguous(), cfp, fixp, meas)
    g = torch.Generator(device="cuda").manual_seed(2)
    meas = (meas + 0.04 * meas.mean() * torch.randn(meas.shape, device="cuda", generator=g)).abs().contiguous()

    def run(a, b):
        p = t[a:b].clone()
        s = torch.full((b - a, m.nparams, nj // se), -1.0, device="cuda")
        tau = torch.full((b - a, nj // se), -1.0, device="cuda") if rician else None
        m.mcmc(meas[a:b], p, cfp, None if fixp is None else fixp[a:b], s, tau, nburn=nb, njumps=nj, sampleevery=se,
               rician=rician, seed=99, voxel_offset=a)
        capi.sync()
        return p, s, tau

    whole = run(0, n)
    step = 500
    for a in range(0, n, step):
        b = min(n, a + step)
        for x, y in zip(whole, run(a, b)):
            if x is not None:
                assert torch.equal(x[a:b], y), (model, a)
