"""Which GridSearch a call takes where a grid that moves no weight gives the
search over basis signals little to share: the call keeps the combinations of
the scan (which a captured call takes), and takes no longer."""
import numpy as np
import pytest

from cudimot_amd import synth

pytestmark = pytest.mark.gpu


def _list(lo, hi, n):
    return ",".join("%.6g" % v for v in np.linspace(lo, hi, n))


ANGLES = "search[%d]=(%s)\nsearch[%d]=(%s)\n"
CASES = [
    # nothing shared between combinations: the scan on a volume that fills the GPU, the search on a small one
    ("Ball_3_Sticks", ANGLES % (3, _list(0.1, 3, 8), 4, _list(-3, 3, 8)), 20000, (140, 130)),
    ("Ball_3_Sticks", ANGLES % (3, _list(0.1, 3, 8), 4, _list(-3, 3, 8)), 500, (140, 130)),
    # one shared signal, two, and a weight that moves
    ("Ball_1_Stick", "search[1]=(0.0005,0.001,0.002)\n" + ANGLES % (3, _list(0.1, 3, 8), 4, _list(-3, 3, 8)), 20000, (300, 300)),
    ("Ball_2_Sticks", ANGLES % (6, _list(0.1, 3, 8), 7, _list(-3, 3, 8)), 20000, (300, 300)),
    ("Ball_2_Sticks", "search[2]=(0.3,0.5,0.7)\nsearch[3]=(0.5,1.5,2.5)\n", 20000, (300, 300)),
    # rows that leave one block per CU
    ("NODDI_Watson", "search[2]=(1,4,8)\n" + ANGLES % (3, _list(0.1, 3, 6), 4, _list(-3, 3, 6)), 20000, (300, 300)),
    # few combinations, other row lengths
    ("Ball_3_Sticks", ANGLES % (3, _list(0.1, 3, 4), 4, _list(-3, 3, 4)), 20000, (95, 91)),
    ("Ball_3_Sticks", ANGLES % (3, _list(0.1, 3, 4), 4, _list(-3, 3, 4)), 20000, (96, 91)),
    # at the lines: measurements in all (262,144), a voxel (80), voxels (8,192 and 81,920)
    ("Ball_2_Sticks", ANGLES % (3, _list(0.1, 3, 8), 4, _list(-3, 3, 8)), 2750, (50, 36)),
    ("Ball_2_Sticks", ANGLES % (3, _list(0.1, 3, 8), 4, _list(-3, 3, 8)), 3000, (50, 36)),
    ("Ball_3_Sticks", ANGLES % (9, _list(0.1, 3, 8), 10, _list(-3, 3, 8)), 8000, (50, 45)),
    ("Ball_3_Sticks", ANGLES % (9, _list(0.1, 3, 8), 10, _list(-3, 3, 8)), 8250, (50, 45)),
    ("Ball_1_Stick", "search[1]=(0.0005,0.002)\n" + ANGLES % (3, _list(0.1, 3, 8), 4, _list(-3, 3, 8)), 81750, (30, 30)),
    ("Ball_1_Stick", "search[1]=(0.0005,0.002)\n" + ANGLES % (3, _list(0.1, 3, 8), 4, _list(-3, 3, 8)), 82000, (30, 30)),
    ("Ball_2_Sticks", ANGLES % (3, _list(0.1, 3, 8), 4, _list(-3, 3, 8)), 14250, (50, 36)),
    ("Ball_2_Sticks", ANGLES % (3, _list(0.1, 3, 8), 4, _list(-3, 3, 8)), 14750, (50, 36)),
    ("Ball_1_Stick", "search[1]=(0.0005,0.001,0.0015,0.002,0.0025)\n", 20000, (37, 37)),
    ("Ball_1_Stick", "search[1]=(0.0005,0.001,0.0015,0.002,0.0025)\n", 20000, (38, 37)),
    ("Ball_1_Stick", "search[1]=(0.0005,0.002)\n" + ANGLES % (3, _list(0.1, 3, 8), 4, _list(-3, 3, 8)), 20000, (240, 234)),
    ("Ball_1_Stick", "search[1]=(0.0005,0.002)\n" + ANGLES % (3, _list(0.1, 3, 8), 4, _list(-3, 3, 8)), 20000, (240, 235)),
]


@pytest.mark.parametrize("model,grid,n,shells", CASES, ids=["%s-%d-%d-%d" % (c[0], i, c[2], 5 + sum(c[3])) for i, c in enumerate(CASES)])
def test_same_combinations_and_no_slower_than_the_scan(model, grid, n, shells):
    import torch
    from cudimot_amd import capi
    cfp = torch.as_tensor(synth.acquisition(5, [(1000, shells[0]), (2500, shells[1])], seed=3), dtype=torch.float32).cuda()
    start = torch.as_tensor(synth.truth_for(model, 250, 17), dtype=torch.float32).cuda().repeat(n // 250, 1).contiguous()
    s0 = torch.full((n, 1), 1000.0, device="cuda")
    meas = torch.empty((n, cfp.shape[0]), device="cuda")
    m = capi.Model(model)
    m.predicted_signal(start.reshape(n, -1, 1), cfp, s0, meas)
    g = torch.Generator(device="cuda").manual_seed(5)
    meas = (meas + 40.0 * torch.randn(meas.shape, device="cuda", generator=g)).abs().contiguous()
    m.load_grid(grid, is_text=True)
    p = [start.clone() for _ in range(2)]
    k = [torch.full((n,), -7, dtype=torch.int32, device="cuda") for _ in range(2)]
    m.gridsearch(meas, p[0], cfp, s0, kept=k[0])
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        m.gridsearch(meas, p[1], cfp, s0, kept=k[1], stream=torch.cuda.current_stream())
    graph.replay()
    torch.cuda.synchronize()
    assert (k[0] >= 0).all() and torch.equal(k[0], k[1]) and torch.equal(p[0], p[1])

    def ms(f):
        best = float("inf")
        for _ in range(5):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            f()
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b))
        return best

    stream = torch.cuda.current_stream()
    call = ms(lambda: m.gridsearch(meas, p[0], cfp, s0, kept=k[0], stream=stream))
    scan = ms(graph.replay)
    assert call < 1.25 * scan + 0.05, (call, scan)
