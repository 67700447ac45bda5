"""GridSearch over basis signals (plug-ins that declare CDM_GRID_LINEAR)
against the general scan of every combination, which a call under stream
capture takes when the volume fills the GPU: both keep the FP64 argmin, the
earliest combination on ties, so the kept combination and the parameters are
the same for every voxel."""
import numpy as np
import pytest

from cudimot_amd import synth

pytestmark = pytest.mark.gpu

N = 8192 + 5  # at 64 lanes: past 8 blocks of four voxels per CU

# model, grid, lanes of the basis search (0: automatic), shells of the acquisition
CASES = [
    # the recipes' grids
    ("NODDI_Watson", "search[0]=(0.0,0.1,0.5,0.9,1.0)\nsearch[1]=(0,0.3,0.6,1.0)\nsearch[2]=(0.000001,0.3,2,8,40)\n", 0, (30, 60)),
    ("NODDI_Watson_refnum", "search[0]=(0.0,0.2,0.4)\nsearch[1]=(0.3,0.6,0.9)\nsearch[2]=(1,5,20)\n", 0, (30, 60)),
    ("NODDI_Bingham", "search[0]=(0,0.1,0.3)\nsearch[1]=(0.3,0.6,0.9)\nsearch[2]=(0.5,2,10,40)\nsearch[3]=(0.2,3,20)\n", 0, (30, 60)),
    ("Ball_2_Sticks", "search[2]=(0.2,0.4,0.6)\nsearch[3]=(0.3,1.2,2.1)\nsearch[4]=(-2,0,2)\n"
                      "search[5]=(0.0,0.1)\nsearch[6]=(0.6,1.5)\nsearch[7]=(-1,1)\n", 0, (70, 71)),
    ("Ball_3_Sticks", "search[1]=(0.001,0.002)\nsearch[2]=(0.4,0.6)\nsearch[5]=(0,0.2)\nsearch[8]=(0.1,0.15)\n"
                      "search[6]=(0.6,1.5)\nsearch[9]=(0.5,1.5,2.4)\nsearch[10]=(-1,1)\n", 16, (40, 41)),
    # one level only: weights, shared, other basis parameters; one combination
    ("NODDI_Bingham", "search[0]=(0,0.05,0.1,0.2,0.3,0.4,0.5)\n", 4, (7, 8)),
    ("NODDI_Bingham", "search[6]=(0,0.5,1,1.5,2,2.5)\n", 64, (30, 60)),
    ("NODDI_Bingham", "search[1]=(0.1,0.5,0.9)\n", 16, (11, 6)),
    ("Ball_1_Stick", "search[4]=(-2.5,-0.5,1.5)\nsearch[0]=(900,1100)\nsearch[3]=(0.2,0.8,1.4)\n", 1, (9, 10)),
    ("Ball_2_Sticks", "search[5]=(0.1)\n", 0, (31, 30)),
    # values outside the bounds drop out
    ("Ball_2_Sticks", "search[2]=(0.2,1.5,0.6)\nsearch[1]=(0.001,0.5)\nsearch[6]=(0.6,1.5)\n", 4, (20, 21)),
]


def _volume(model, n, shells, torch):
    from cudimot_amd import capi
    cfp = synth.acquisition(5, [(1000, shells[0]), (2500, shells[1])], seed=3)
    t = synth.truth_for(model, 200, 17)
    t = np.tile(t, (n // 200 + 1, 1))[:n].astype(np.float32)
    m = capi.Model(model)
    d_t, d_cfp = torch.as_tensor(t).cuda(), torch.as_tensor(cfp, dtype=torch.float32).cuda()
    s0 = torch.full((n, 1), 1000.0, device="cuda")
    clean = torch.empty((n, cfp.shape[0]), device="cuda")
    m.predicted_signal(d_t.reshape(n, -1, 1), d_cfp, s0, clean)
    g = torch.Generator(device="cuda").manual_seed(5)
    meas = (clean + 40.0 * torch.randn(clean.shape, device="cuda", generator=g)).abs()
    return d_t, d_cfp, s0, meas.contiguous()


@pytest.mark.parametrize("model,grid,lanes,shells", CASES)
def test_basis_search_equals_general_scan(model, grid, lanes, shells):
    import torch
    from cudimot_amd import capi
    start, cfp, s0, meas = _volume(model, N, shells, torch)
    start[3, 1] = -5.0  # outside the bounds (sticks: d; NODDI: fintra)
    meas[7, 2] = float("nan")
    meas[8, 4] = float("inf")
    meas[9] = 0.0
    meas[10] = 3e30  # costs past the float range
    m = capi.Model(model)
    m.load_grid(grid, is_text=True)
    if lanes:
        m.set_group(capi.GRIDSEARCH, lanes)
    out = {}
    for name, n in (("whole", N), ("slab", 300)):  # one scan per voxel, and slices
        p = start[:n].clone()
        kept = torch.full((n,), -7, dtype=torch.int32, device="cuda")
        m.gridsearch(meas[:n], p, cfp, s0[:n], kept=kept)
        out[name] = (p, kept)
    torch.cuda.synchronize()
    # the general scan, recorded into a graph (the 64-lane groups fill the GPU)
    m.set_group(capi.GRIDSEARCH, 64)
    p = start.clone()
    kept = torch.full((N,), -7, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        m.gridsearch(meas, p, cfp, s0, kept=kept, stream=torch.cuda.current_stream())
    g.replay()
    torch.cuda.synchronize()
    want_p, want_k = p.cpu().numpy(), kept.cpu().numpy()
    assert (want_k >= 0).mean() > 0.99
    for name, (p, kept) in out.items():
        k = kept.cpu().numpy()
        n = len(k)
        bad = np.nonzero(k != want_k[:n])[0]
        assert bad.size == 0, (name, bad[:10], k[bad[:10]], want_k[bad[:10]])
        np.testing.assert_array_equal(p.cpu().numpy(), want_p[:n])
