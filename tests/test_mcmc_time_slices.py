"""MCMC in time slices, with the launches looked at: a captured call's kernel nodes
tell how many blocks it launched, so a case that does not run in slices fails.
Each sliced chain equals the chain of cdm_mcmc_noalloc, which has none, over parts
of the volume, bit for bit: burn-in and recording in four slices and more, uneven
last slices, tau handed from block to block, cache rows in LDS and in memory,
partial caches, jump blocks and graph replay.  Light models stay in one launch of
a block per tile, which is the faster one there."""
import ctypes

import pytest

from tests import helpers as H

pytestmark = pytest.mark.gpu


class _Dim3(ctypes.Structure):
    _fields_ = [("x", ctypes.c_uint), ("y", ctypes.c_uint), ("z", ctypes.c_uint)]


class _KernelParams(ctypes.Structure):  # hipKernelNodeParams
    _fields_ = [("block", _Dim3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p), ("grid", _Dim3),
                ("params", ctypes.c_void_p), ("shared", ctypes.c_uint)]


def _grids(call):
    """Blocks of each kernel with dynamic LDS that call(stream) launches (recorded,
    not run): the MCMC kernels, no fill."""
    import torch
    from cudimot_amd import capi
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        call(torch.cuda.current_stream())
    hip = capi.lib()  # the runtime that the library itself is bound to
    raw = ctypes.c_void_p(graph.raw_cuda_graph())
    n = ctypes.c_size_t()
    assert hip.hipGraphGetNodes(raw, None, ctypes.byref(n)) == 0
    nodes = (ctypes.c_void_p * n.value)()
    assert hip.hipGraphGetNodes(raw, nodes, ctypes.byref(n)) == 0
    out = []
    for node in nodes:
        kind, p = ctypes.c_int(-1), _KernelParams()
        assert hip.hipGraphNodeGetType(ctypes.c_void_p(node), ctypes.byref(kind)) == 0
        if kind.value == 0:  # a kernel
            assert hip.hipGraphKernelNodeGetParams(ctypes.c_void_p(node), ctypes.byref(p)) == 0
            if p.shared:
                out.append(p.grid.x)
    return out


def _volume(model, n):
    import torch
    from cudimot_amd import capi, synth
    cfp = H.dev(H.ACQ[H.MODEL_ACQ[model]]())
    t = H.dev(synth.clip_to_bounds(model, H.truth(model, 500, 9))).repeat(n // 500 + 1, 1)[:n].contiguous()
    m = capi.Model(model)
    fixp = torch.full((n, 1), 1000.0, device="cuda") if m.fixp_tsize else None
    meas = torch.empty((n, cfp.shape[0]), device="cuda")
    m.predicted_signal(t.reshape(n, -1, 1).contiguous(), cfp, fixp, meas)
    g = torch.Generator(device="cuda").manual_seed(2)
    meas = (meas + 0.04 * meas.mean() * torch.randn(meas.shape, device="cuda", generator=g)).abs().contiguous()
    return m, t, cfp, fixp, meas


CASES = [
    # model, voxels, lanes, register budget, Rician, (burn-in, jumps, every), least slices of a phase, jump blocks
    ("Ball_2_Sticks", 18001, 16, 2, False, (70, 99, 3), 2, 0),
    ("Ball_2_Sticks", 70003, 4, 2, False, (200, 330, 10), 4, 0),
    ("Ball_1_Stick", 18003, 16, 4, False, (400, 630, 21), 4, 0),
    ("Ball_2_Sticks", 18001, 16, 1, True, (130, 150, 10), 4, 0),
    ("NODDI_Bingham", 34005, 4, 1, False, (100, 130, 10), 4, 0),   # cache rows in LDS
    ("NODDI_Bingham", 66001, 4, 4, False, (70, 90, 9), 2, 0),      # and in memory
    ("NODDI_Bingham", 9003, 16, 1, True, (100, 130, 10), 4, 0),
    ("NODDI_Bingham_2Fans", 9002, 16, 2, False, (100, 130, 10), 4, 0),  # a partial cache
    ("NODDI_Watson", 18002, 16, 4, False, (100, 130, 10), 4, 0),
    ("Ball_2_Sticks", 70003, 4, 2, False, (190, 320, 10), 2, 128),
]


@pytest.mark.parametrize("case", CASES, ids=["%s-%d-%d-%s-%d" % (c[0], c[1], c[2], "rician" if c[4] else "gauss", c[7]) for c in CASES])
def test_sliced_chains_equal_unsliced_parts(case):
    import torch
    from cudimot_amd import capi
    model, n, lanes, budget, rician, (nb, nj, se), least, block = case
    m, t, cfp, fixp, meas = _volume(model, n)
    m.set_group(capi.MCMC, lanes)
    m.set_occupancy(capi.MCMC, budget)

    def buffers(k):
        return (torch.empty((k, m.nparams), device="cuda"), torch.empty((k, m.nparams, nj // se), device="cuda"),
                torch.empty((k, nj // se), device="cuda") if rician else None)

    def run(f, a, b, stream=None, into=None):
        p, s, tau = into or buffers(b - a)
        p.copy_(t[a:b])
        s.fill_(-1.0)
        f(meas[a:b], p, cfp, None if fixp is None else fixp[a:b], s, tau, nburn=nb, njumps=nj, sampleevery=se,
          rician=rician, seed=99, voxel_offset=a, stream=stream)
        return p, s, tau

    m.set_mcmc_blocks(block, False)
    whole = run(m.mcmc, 0, n)
    tiles = (n * lanes + 255) // 256
    grids = _grids(lambda s: run(m.mcmc, 0, n, s))
    launches = 2 if not block else -(-nb // block) + -(-nj // block)
    assert len(grids) == launches and all(x % tiles == 0 for x in grids), (grids, tiles)
    assert max(x // tiles for x in grids) >= least, (grids, tiles)
    if not block:
        assert min(x // tiles for x in grids) >= 2, (grids, tiles)
    if block:  # recorded by the handle, then replayed
        m.set_mcmc_blocks(block, True)
        into = buffers(n)
        for _ in range(3):
            again = run(m.mcmc, 0, n, into=into)
            torch.cuda.synchronize()
            assert all(x is None or torch.equal(x, y) for x, y in zip(whole, again))
        assert m.graph_stats() == (2, 4)
    torch.cuda.synchronize()
    m.set_mcmc_blocks(0, False)
    for a in range(0, n, 1500):
        b = min(n, a + 1500)
        for x, y in zip(whole, run(m.mcmc_noalloc, a, b)):
            if x is not None:
                assert torch.equal(x[a:b], y), (model, a)


@pytest.mark.parametrize("model,n,jumps", [("toymodel", 66000, 64), ("Ball_1_Stick", 140000, 32), ("DiffusionTensor", 140000, 32)])
def test_light_models_take_one_block_per_tile(model, n, jumps):
    import torch
    from cudimot_amd import capi
    m, t, cfp, fixp, meas = _volume(model, n)
    s = torch.empty((n, m.nparams, 1), device="cuda")
    go = lambda q: m.mcmc(meas, t.clone(), cfp, fixp, s, nburn=jumps, njumps=jumps, sampleevery=jumps, stream=q)  # noqa: E731
    go(None)
    tiles = (n * m.get_group(capi.MCMC, cfp.shape[0], n) + 255) // 256
    assert _grids(go) == [tiles, tiles]


@pytest.mark.parametrize("model,n,jumps", [("Ball_2_Sticks", 4000, 100), ("DiffusionTensor", 3300, 40)])
def test_rician_launches_of_few_rounds_take_slices(model, n, jumps):
    """No slower than the chains without slices, and the same."""
    import torch
    from cudimot_amd import capi
    m, t, cfp, fixp, meas = _volume(model, n)
    m.set_group(capi.MCMC, 64)
    s = torch.empty((n, m.nparams, 1), device="cuda")
    tau = torch.empty((n, 1), device="cuda")
    p = t.clone()

    def go(f, a, b, q=None):
        p.copy_(t)
        f(meas[a:b], p[a:b], cfp, None if fixp is None else fixp[a:b], s[a:b], tau[a:b], nburn=jumps, njumps=jumps,
          sampleevery=jumps, rician=True, seed=5, voxel_offset=a, stream=q or torch.cuda.current_stream())

    def ms(f):
        best = float("inf")
        for _ in range(6):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            f()
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b))
        return best
    go(m.mcmc, 0, n)
    assert min(_grids(lambda q: go(m.mcmc, 0, n, q))) >= 2 * n // 4
    sliced = ms(lambda: go(m.mcmc, 0, n))
    got = s.clone(), tau.clone()
    whole = ms(lambda: [go(m.mcmc_noalloc, a, min(n, a + 1500)) for a in range(0, n, 1500)])
    assert torch.equal(got[0], s) and torch.equal(got[1], tau)
    assert sliced < whole, (sliced, whole)


@pytest.mark.parametrize("model,n,jumps", [("DiffusionTensor", 4153, 70), ("NODDI_Watson", 4153, 32), ("Ball_1_Stick", 4313, 70)])
def test_short_chains_at_64_lanes_take_slices(model, n, jumps):
    """Launches of two rounds and a little more, whose last is nearly empty."""
    import torch
    from cudimot_amd import capi
    m, t, cfp, fixp, meas = _volume(model, n)
    m.set_group(capi.MCMC, 64)
    s = torch.empty((n, m.nparams, 1), device="cuda")
    p = t.clone()
    go = lambda q: m.mcmc(meas, p, cfp, fixp, s, nburn=jumps, njumps=jumps, sampleevery=jumps, stream=q)  # noqa: E731
    go(None)
    torch.cuda.synchronize()
    assert min(_grids(go)) >= 2 * ((n + 3) // 4)
