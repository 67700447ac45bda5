"""GridSearch under stream capture: a call over a small volume, whose scan is
split into slices, records after the same call outside capture has run (the
slices' scratch is there), its replays keep the eager call's combinations, and
searches between the replays, over volumes that need more scratch, leave the
recorded one alone."""
import pytest

from cudimot_amd import synth

pytestmark = pytest.mark.gpu

WATSON = ("search[0]=(0.0,0.1,0.2,0.3,0.4,0.5,0.6,0.7,0.8,0.9,1.0)\n"
          "search[1]=(0.0,0.1,0.2,0.3,0.4,0.5,0.6,0.7,0.8,0.9,1.0)\nsearch[2]=(1,2,3,4,5,6,7,8)\n")
STICKS = ("search[2]=(0.2,0.4,0.6)\nsearch[3]=(0.3,1.2,2.1)\nsearch[4]=(-2,0,2)\n"
          "search[5]=(0.0,0.1,0.2)\nsearch[6]=(0.6,1.5,2.4)\nsearch[7]=(-1,1,3)\n")


def _volume(model, n):
    import torch
    from cudimot_amd import capi
    cfp = torch.as_tensor(synth.model_acquisition(model), dtype=torch.float32).cuda()
    t = torch.as_tensor(synth.truth_for(model, 250, 17), dtype=torch.float32).cuda().repeat(n // 250 + 1, 1)[:n].contiguous()
    s0 = torch.full((n, 1), 1000.0, device="cuda")
    clean = torch.empty((n, cfp.shape[0]), device="cuda")
    capi.Model(model).predicted_signal(t.reshape(n, -1, 1), cfp, s0, clean)
    g = torch.Generator(device="cuda").manual_seed(5)
    meas = (clean + 40.0 * torch.randn(clean.shape, device="cuda", generator=g)).abs().contiguous()
    return t, cfp, s0, meas


@pytest.mark.parametrize("warm", [True, False])
@pytest.mark.parametrize("model,grid,n", [("NODDI_Watson", WATSON, 300), ("NODDI_Watson", WATSON, 1000),
                                          ("Ball_2_Sticks", STICKS, 300)])
def test_captured_small_volume_equals_eager(model, grid, n, warm):
    import torch
    from cudimot_amd import capi
    start, cfp, s0, meas = _volume(model, 20 * n)
    want_p, want_k = start[:n].clone(), torch.full((n,), -7, dtype=torch.int32, device="cuda")
    m = capi.Model(model)
    m.load_grid(grid, is_text=True)
    m.gridsearch(meas[:n], want_p, cfp, s0[:n], kept=want_k)
    torch.cuda.synchronize()
    assert (want_k >= 0).all()
    if not warm:  # a handle that has searched one voxel only: the grid is there, no scratch is
        m = capi.Model(model)
        m.load_grid(grid, is_text=True)
        m.gridsearch(meas[:1], start[:1].clone(), cfp, s0[:1])
        torch.cuda.synchronize()
    p, k = start[:n].clone(), torch.full((n,), -7, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        m.gridsearch(meas[:n], p, cfp, s0[:n], kept=k, stream=torch.cuda.current_stream())
    for between in (n, 4 * n, 20 * n):
        p.copy_(start[:n])
        k.fill_(-7)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(k, want_k) and torch.equal(p, want_p), (model, n, between)
        q = start[:between].clone()
        m.gridsearch(meas[:between], q, cfp, s0[:between])
        torch.cuda.synchronize()
        assert torch.equal(q[:n], want_p)
