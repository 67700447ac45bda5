"""The build's check for vector instructions placed before a mask update, and
the Levenberg-Marquardt kernels at every launch shape against one another."""
import pytest

from cudimot_amd import build, execcheck

# Where lanes rejoin: the copy belongs after the mask update
JOIN = """
<kernel>:
	s_and_saveexec_b64 s[0:1], vcc
	s_xor_b64 s[22:23], exec, s[0:1]
	s_cbranch_execz L4                                         // 000000000010: BF880009
	v_add_f64 v[2:3], v[4:5], v[6:7]
<L4>:
	s_mov_b32 s34, 0x11122322
	s_waitcnt lgkmcnt(0)
	%s
	s_andn2_saveexec_b64 s[0:1], s[22:23]
	%s
	s_cbranch_execz L5
	v_mul_f64 v[2:3], v[4:5], v[6:7]
<L5>:
	v_readlane_b32 s0, v127, 14
	%s
	s_or_b64 exec, exec, s[0:1]
	%s
	s_endpgm
"""
COPY, SPILL = "v_mov_b64_e32 v[10:11], v[80:81]", "scratch_store_dwordx2 off, v[72:73], off offset:1236"
REGS = "v_readlane_b32 s1, v127, 15"


@pytest.mark.parametrize("lines,found", [
    ((COPY, REGS, REGS, REGS), [("L4", COPY, "s_andn2_saveexec_b64 s[0:1], s[22:23]")]),
    ((REGS, COPY, SPILL, SPILL), [("L5", SPILL, "s_or_b64 exec, exec, s[0:1]")]),
    ((REGS, COPY, REGS, SPILL), []),
    (("v_accvgpr_write_b32 a155, v117", REGS, COPY, REGS),
     [("L4", "v_accvgpr_write_b32 a155, v117", "s_andn2_saveexec_b64 s[0:1], s[22:23]"),
      ("L5", COPY, "s_or_b64 exec, exec, s[0:1]")]),
])
def test_instructions_before_a_mask_update_are_found(lines, found):
    text = (JOIN % lines).splitlines(True)
    assert execcheck.misplaced(text) == [("kernel",) + f for f in found]
    # not the head of a block that an empty mask reaches: the branch's own code
    assert execcheck.misplaced([l.replace("s_cbranch_execz", "s_cbranch_vccz") for l in text]) == []


@pytest.mark.parametrize("bad", [0, 1, 2])
def test_a_faulty_unit_is_compiled_again_and_refused_if_it_stays(tmp_path, monkeypatch, bad):
    src = tmp_path / "unit.hip"
    src.write_text("")
    cmds = []
    monkeypatch.setattr(build, "_run", cmds.append)
    monkeypatch.setattr(execcheck, "misplaced_in_object", lambda o, a: [("k", "L4", COPY, "s_or")] if len(cmds) <= bad
                        else [])
    if bad == 2:
        with pytest.raises(RuntimeError, match="k L4"):
            build._compile(str(src), str(tmp_path / "unit.o"), [])
        assert not (tmp_path / "unit.o.sha").exists()
    else:
        build._compile(str(src), str(tmp_path / "unit.o"), [])
    assert ["-sgpr-regalloc=basic" in c for c in cmds] == [False, True][:min(bad, 1) + 1]


def _fit(m, v, lanes, budget):
    import torch
    from cudimot_amd import capi
    from tests.helpers import dev
    m.set_group(capi.LEVMAR, lanes)
    m.set_occupancy(capi.LEVMAR, budget)
    p = dev(v["start"])
    cost = torch.empty(v["n"], device="cuda")
    iters = torch.empty(v["n"], dtype=torch.int32, device="cuda")
    m.levmar(v["meas"], p, v["cfp"], v["fixp"], max_iters=40, cost=cost, iters=iters)
    return p, cost, iters


@pytest.mark.gpu
@pytest.mark.parametrize("lanes", [1, 4, 16, 64])
def test_fits_do_not_depend_on_the_kernel_compiled_for_them(lanes):
    """Register budgets and the batched launch change registers and spills only."""
    import torch
    from cudimot_amd import capi
    from tests.helpers import dev
    from tests.test_batch import _volumes
    vols = _volumes(710)
    items, fits = [], []
    for v in vols:
        m = capi.Model(v["name"])
        fits.append([_fit(m, v, lanes, w) for w in (1, 2, 4)])
        mb = capi.Model(v["name"])
        mb.set_group(capi.LEVMAR, lanes)
        items.append(dict(model=mb, meas=v["meas"], params=dev(v["start"]), cfp=v["cfp"], fixp=v["fixp"],
                          cost=torch.empty(v["n"], device="cuda"),
                          iters=torch.empty(v["n"], dtype=torch.int32, device="cuda")))
    capi.batch_levmar(items, max_iters=40)
    capi.sync()
    for v, f, it in zip(vols, fits, items):
        assert (f[0][2] > 0).float().mean() > 0.9, v["name"]
        for other in f[1:] + [(it["params"], it["cost"], it["iters"])]:
            assert all(torch.equal(a, b) for a, b in zip(f[0], other)), v["name"]


@pytest.mark.gpu
@pytest.mark.parametrize("model", ["Ball_1_Stick", "Ball_2_Sticks", "NODDI_Watson", "NODDI_Watson_refnum", "NODDI_Bingham"])
def test_fits_of_the_other_plug_ins_do_not_depend_on_the_register_budget(model):
    import torch
    from cudimot_amd import capi
    from tests.test_mcmc_time_slices import _volume
    n = 150
    m, t, cfp, fixp, meas = _volume(model, n)
    rng = torch.Generator(device="cuda").manual_seed(3)
    start = (t * (1 + 0.02 * torch.randn(t.shape, device="cuda", generator=rng))).contiguous()
    v = dict(meas=meas, cfp=cfp, fixp=fixp, n=n, start=start.cpu().numpy())
    for lanes in (1, 4, 16, 64):
        f = [_fit(m, v, lanes, w) for w in (1, 2, 4)]
        assert (f[0][2] > 0).float().mean() > 0.9, lanes
        assert all(torch.equal(a, b) for g in f[1:] for a, b in zip(f[0], g)), lanes
