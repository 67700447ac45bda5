"""GridSearch of plug-ins without the hooks of the search over basis signals: the
general scan in slices and whole."""
import numpy as np
import pytest

from tests.helpers import dev, host

pytestmark = pytest.mark.gpu

# 243 combinations each.  The last two values of one parameter differ by less than
# a single-precision screen can tell, so that every voxel has several candidates
# and some more than a slice lists.
GRIDS = {
    "DiffusionTensor": "search[1]=(0.0005,0.0015,0.0025)\nsearch[2]=(-0.0003,0,1e-11)\nsearch[4]=(0.0005,0.0015,0.0025)\n"
                       "search[5]=(0,1e-11,2e-11)\nsearch[6]=(0.0005,0.0015,0.0025)\n",
    "NODDI_Bingham_2Fans": "search[0]=(0.0,0.1,0.1000001)\nsearch[1]=(0.2,0.4,0.4000001)\nsearch[2]=(0.4,0.6,0.8)\n"
                           "search[3]=(5,15,40)\nsearch[8]=(0.4,0.6,0.8)\n",
}


@pytest.mark.parametrize("model", sorted(GRIDS))
@pytest.mark.parametrize("lanes", [1, 4, 64])
@pytest.mark.parametrize("n", [1, 37])
def test_slices_keep_what_the_whole_scan_keeps(model, lanes, n):
    """The same voxels in a call that fills the GPU, whose groups scan the grid alone."""
    import torch
    from cudimot_amd import capi, synth
    m = capi.Model(model)
    m.load_grid(GRIDS[model], is_text=True)
    m.set_group(capi.GRIDSEARCH, lanes)
    cfp = dev(synth.model_acquisition(model)[::4])
    t = np.ascontiguousarray(synth.truth_for(model, n, 41), dtype=np.float32)
    copies = 8 * 256 * 256 // lanes // n + 1

    def search(k):
        fixp = torch.full((k * n, 1), 1000.0, device="cuda") if m.fixp_tsize else None
        clean = torch.empty((n, cfp.shape[0]), device="cuda")
        m.predicted_signal(dev(t.reshape(n, -1, 1)), cfp, None if fixp is None else fixp[:n], clean)
        noise = torch.randn(clean.shape, device="cuda", generator=torch.Generator(device="cuda").manual_seed(6))
        meas = (clean + 0.03 * clean.mean() * noise).abs().repeat(k, 1).contiguous()
        p = dev(np.tile(t, (k, 1)))
        kept = torch.full((k * n,), -7, dtype=torch.int32, device="cuda")
        m.gridsearch(meas, p, cfp, fixp, kept=kept)
        capi.sync()
        return host(p), kept.cpu().numpy()

    (p, k), (big_p, big_k) = search(1), search(copies)
    assert (k >= 0).all()
    for c in (0, copies // 2, copies - 1):
        np.testing.assert_array_equal(k, big_k[c * n:(c + 1) * n])
        np.testing.assert_array_equal(p, big_p[c * n:(c + 1) * n])
