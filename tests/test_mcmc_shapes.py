"""Launch shapes that MCMC takes by itself on volumes that do not fill the GPU:
no slower than the shapes set by hand, with the same samples."""
import pytest

from tests.test_mcmc_time_slices import _volume

pytestmark = pytest.mark.gpu


def _ms(f):
    import torch
    best = float("inf")
    for _ in range(6):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        f()
        b.record()
        torch.cuda.synchronize()
        best = min(best, a.elapsed_time(b))
    return best


def _calls(model, n, rician, jumps):
    import torch
    m, t, cfp, fixp, meas = _volume(model, n)
    s = torch.empty((n, m.nparams, 1), device="cuda")
    tau = torch.empty((n, 1), device="cuda") if rician else None
    p = t.clone()

    def go():
        p.copy_(t)
        m.mcmc(meas, p, cfp, fixp, s, tau, nburn=jumps, njumps=jumps, sampleevery=jumps, rician=rician, seed=3,
               stream=torch.cuda.current_stream())
    return m, go, s


@pytest.mark.parametrize("model,n", [("NODDI_Watson", 1), ("NODDI_Watson", 300), ("DiffusionTensor", 32000), ("Ball_1_Stick", 300)])
def test_small_volumes_take_the_registers_they_can_have(model, n):
    from cudimot_amd import capi
    m, go, s = _calls(model, n, False, 48)
    own = _ms(go)
    first = s.clone()
    by_hand = []
    for budget in (1, 2, 4):
        m.set_occupancy(capi.MCMC, budget)
        by_hand.append(_ms(go))
        assert (s == first).all()
    assert own < 1.12 * min(by_hand) + 0.03, (own, by_hand)


@pytest.mark.parametrize("n", [21000, 26000])
def test_rician_chains_of_mid_size_volumes_take_the_better_lanes(n):
    from cudimot_amd import capi
    m, go, _ = _calls("Ball_2_Sticks", n, True, 15)
    own = _ms(go)
    by_hand = []
    for lanes in (4, 16):
        m.set_group(capi.MCMC, lanes)
        by_hand.append(_ms(go))
    assert own < 1.08 * min(by_hand), (own, by_hand)


@pytest.mark.parametrize("model", ["NODDI_Watson", "Ball_1_Stick"])
@pytest.mark.parametrize("n", [5600, 7000])
def test_rician_chains_of_small_volumes_keep_16_lanes(model, n):
    from cudimot_amd import capi
    m, go, _ = _calls(model, n, True, 48)
    own = _ms(go)
    by_hand = []
    for lanes in (16, 64):
        m.set_group(capi.MCMC, lanes)
        by_hand.append(_ms(go))
    assert own < 1.08 * min(by_hand), (own, by_hand)
