"""A newly loaded grid: its set-up on the host, which the first search after a
load pays for, costs less than parsing its text; values listed twice or out of
order keep the earliest best combination."""
import ctypes
import time

import numpy as np
import pytest

from tests.test_gridsearch_capture import _volume

pytestmark = pytest.mark.gpu


def _list(lo, hi, n):
    return ",".join("%.6g" % v for v in np.linspace(lo, hi, n))


def test_first_search_after_a_load_costs_less_than_the_load():
    """262,144 combinations of one voxel: what the first call takes beyond the
    second is the set-up (the device part is the same)."""
    import torch
    from cudimot_amd import capi
    start, cfp, s0, meas = _volume("NODDI_Watson", 1)
    text = "search[0]=(%s)\nsearch[1]=(%s)\nsearch[2]=(%s)\n" % (_list(0.01, 0.95, 64), _list(0.01, 0.95, 64),
                                                               _list(0.5, 20, 64))
    m = capi.Model("NODDI_Watson")
    nc, ng = ctypes.c_int(), ctypes.c_int()

    def timed(f):
        torch.cuda.synchronize()
        t = time.perf_counter()
        f()
        torch.cuda.synchronize()
        return time.perf_counter() - t

    def search():
        m.gridsearch(meas, start.clone(), cfp, s0)

    load, first, second = [], [], []
    for _ in range(5):
        load.append(timed(lambda: capi.check(capi.lib().cdm_model_load_grid(m.h, text.encode(), 1, ctypes.byref(nc),
                                                                           ctypes.byref(ng)))))
        first.append(timed(search))
        second.append(timed(search))
    assert nc.value == 64 ** 3
    assert min(first) - min(second) < min(load), (load, first, second)


@pytest.mark.parametrize("model,plain,listed", [
    # the same values, some of them twice, out of order or outside the bounds
    ("NODDI_Watson", "search[0]=(0.1,0.3)\nsearch[1]=(0.3,0.6,0.9)\nsearch[2]=(1,4,16)\n",
     "search[0]=(0.3,0.1,0.3)\nsearch[1]=(0.9,0.3,0.6)\nsearch[2]=(16,1,4,1)\n"),
    ("NODDI_Watson", "search[0]=(0.1,0.3)\nsearch[1]=(0.3,0.6,0.9)\nsearch[2]=(1,4,16)\n",
     "search[0]=(1.5,0.3,0.1)\nsearch[1]=(0.9,-1,0.3,0.6)\nsearch[2]=(16,1,100,4)\n"),
    # (no fraction of zero: the angles of a stick without weight tie)
    ("Ball_2_Sticks", "search[2]=(0.3,0.6)\nsearch[3]=(0.3,1.2)\nsearch[5]=(0.1,0.2)\nsearch[7]=(-1,1,3)\n",
     "search[2]=(0.6,0.3)\nsearch[3]=(1.2,0.3,0.3)\nsearch[5]=(0.2,0.1)\nsearch[7]=(3,-1,1)\n"),
])
def test_order_and_repeats_keep_the_parameters(model, plain, listed):
    import torch
    from cudimot_amd import capi
    n = 700
    start, cfp, s0, meas = _volume(model, n)
    got = []
    for text in (plain, listed):
        m = capi.Model(model)
        gp, grid = m.load_grid(text, is_text=True)
        p, k = start.clone(), torch.full((n,), -7, dtype=torch.int32, device="cuda")
        m.gridsearch(meas, p, cfp, s0, kept=k)
        torch.cuda.synchronize()
        k = k.cpu().numpy()
        assert (k >= 0).all()
        vals = np.asarray(grid)[k]
        np.testing.assert_array_equal(p.cpu().numpy()[:, gp], vals.astype(np.float32))
        # the earliest of equal combinations
        first = {}
        for i, row in enumerate(map(tuple, grid)):
            first.setdefault(row, i)
        assert all(first[tuple(grid[i])] == i for i in set(k.tolist()))
        got.append(vals)
    np.testing.assert_array_equal(got[0], got[1])
