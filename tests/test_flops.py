"""FLOP model (cudimot_amd/flops.py over the operation-counting build of the
plug-ins): every shipped plug-in evaluates through each of its cache hooks,
with the engine's measurement cache handed in where the plug-in declares
one, and gives finite counts."""
import numpy as np
import pytest


@pytest.mark.parametrize("model", ["Ball_1_Stick", "Ball_2_Sticks", "Ball_3_Sticks", "DiffusionTensor",
                                   "NODDI_Watson", "NODDI_Bingham", "NODDI_Bingham_2Fans", "toymodel"])
def test_per_eval_counts_every_plugin(model):
    from cudimot_amd import flops, synth
    cfp = synth.model_acquisition(model)
    t = synth.truth_for(model, 6, 2)
    ev = flops.per_eval(model, t, cfp, np.full((6, 1), 1000.0))
    vals = [v for v in ev.values() if isinstance(v, (float, np.floating))]
    assert all(np.isfinite(v) and v >= 0 for v in vals), ev
    assert ev["fwd32"] + ev["fwd64"] > 0


def test_bingham_mcmc_flops_use_the_per_measurement_cache():
    """The intra-axonal cache is recomputed only in steps of the parameters
    it depends on (kappa, beta, th, ph, psi)."""
    from cudimot_amd import flops, synth
    cfp = synth.model_acquisition("NODDI_Bingham")
    ev = flops.per_eval("NODDI_Bingham", synth.truth_for("NODDI_Bingham", 6, 2), cfp, np.full((6, 1), 1000.0))
    assert ev["mvc"] and ev["mvc_dep"] == 0x7C
    assert ev["mv64"] > 0 and ev["pmv64"] == 0


@pytest.mark.parametrize("model", ["Ball_1_Stick", "Ball_2_Sticks", "Ball_3_Sticks", "NODDI_Watson", "NODDI_Bingham"])
def test_kept_frames_leave_no_sines_in_a_measurement(model):
    """A chain takes the sine and cosine of an angle once per step that moves it,
    not at every measurement."""
    from cudimot_amd import flops, synth
    cfp = synth.model_acquisition(model)
    ev = flops.per_eval(model, synth.truth_for(model, 6, 2), cfp, np.full((6, 1), 1000.0))
    angles = bin(ev["fr_dep"]).count("1")
    assert angles >= 2 and ev["fr32"] + ev["fr64"] == 2
    whole = ev["pmv32"] + ev["mv32"] if ev["mvc"] else ev["meas32"]
    assert ev["moved32"] <= whole - 2 * angles and ev["kept32"] <= ev["moved32"]
    f32, f64 = flops.mcmc_flops(ev, 1, 10, 3)
    vc = bin(ev["vc_dep"]).count("1")
    assert f32 == pytest.approx(3 * (vc * ev["vc32"] + angles * ev["fr32"] + 10 * (ev["kept32"] + 3)))
    assert f64 == pytest.approx(3 * (vc * ev["vc64"] + angles * ev["fr64"] + 10 * (ev["kept64"] + 1)))
