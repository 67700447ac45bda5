"""Performance cases: the calls a user of the engine makes, over their sizes.

A voxelwise fit goes through the same few entry points whatever the model: a
starting point (tensor fit, GridSearch or the network), Levenberg-Marquardt,
MCMC, and the derived maps of the samples.  Each case is one of those calls on
a synthetic volume resident in device memory.  Volumes run from a few hundred
voxels (a slice, or the voxels a fallback refits) to a whole brain, and the
acquisitions are the measured workloads' (64, 99 and 280 measurements) or, in
drawn cases, other counts of directions.

Signals come from physical forward models written here in torch (sticks and
tensors in closed form, the NODDI orientation distributions by quadrature over
the sphere), with Rician noise, so they do not depend on the engine.

LM on a NODDI model is called with a few iterations: near the optimum its
surface is so flat that long runs end in different places of the same valley
after any change of rounding.
"""
import math

import numpy as np
import torch

from cudimot_amd import capi, learned, pipelines, synth

DPAR, DISO = 1.7e-3, 3.0e-3  # NODDI diffusivities (mm^2/s)

# Grids: the three-level stick search of the tests, and the scan of 12 angles
# that completes the learned start.
STICKS_GRID = ("search[2]=(0.2,0.4,0.6)\nsearch[3]=(0.3,1.2,2.1)\nsearch[4]=(-2,0,2)\n"
               "search[5]=(0.0,0.1,0.2)\nsearch[6]=(0.6,1.5,2.4)\nsearch[7]=(-1,1,3)\n")
STICKS_AXES = {2: (0.2, 0.4, 0.6), 3: (0.3, 1.2, 2.1), 4: (-2., 0., 2.), 5: (0., 0.1, 0.2), 6: (0.6, 1.5, 2.4),
               7: (-1., 1., 3.)}
PSI_GRID = "search[6]=(%s)\n" % ",".join("%.9g" % (math.pi * k / 12) for k in range(12))

# b-values of the shells of each kind of signal
SHELLS = {"sticks1": (1000, 2000, 3000), "sticks2": (1000, 2000, 3000), "tensor": (1000, 2000, 3000),
          "watson": (700, 2000, 3000), "bingham": (700, 2000, 3000)}


def listed():
    return [
        # A region of interest fitted by itself: a few voxels per call, where launches and each
        # voxel's serial chain count.
        dict(name="lm_stick_roi", kind="lm", signal="sticks1", model="Ball_1_Stick", n=400, b0=4, d1=30, d2=30, d3=0,
             iters=100, fixed=""),
        # The tensor fit every orientation start begins with, whole volume.
        dict(name="lm_tensor", kind="lm", signal="tensor", model="DiffusionTensor", n=250000, b0=4, d1=30, d2=30, d3=0,
             iters=50, fixed=""),
        # LM of a few iterations on the two NODDI models, a slab of a volume.
        dict(name="lm_watson", kind="lm", signal="watson", model="NODDI_Watson", n=60000, b0=9, d1=30, d2=60, d3=0,
             iters=12, fixed=""),
        dict(name="lm_bingham", kind="lm", signal="bingham", model="NODDI_Bingham", n=50003, b0=9, d1=30, d2=60, d3=0,
             iters=8, fixed=""),
        # GridSearch: the reference pipelines' recipes.  The Bingham grid (11,050 combinations) is
        # searched for the few hundred voxels the learned start's fallback refits.
        dict(name="grid_bingham_fallback", kind="grid", signal="bingham", model="NODDI_Bingham", n=307, b0=9, d1=30,
             d2=60, d3=0, grid="recipe", fixed="4,5"),
        dict(name="grid_watson", kind="grid", signal="watson", model="NODDI_Watson", n=150000, b0=9, d1=30, d2=60, d3=0,
             grid="recipe", fixed="3,4"),
        dict(name="grid_sticks", kind="grid", signal="sticks2", model="Ball_2_Sticks", n=50000, b0=10, d1=90, d2=90,
             d3=90, grid="recipe", fixed=""),
        # MCMC, the bulk of a fit's time, in shorter chains than a user's (1000 + 1250 jumps): time is
        # proportional to the jumps.  One model is FP64-heavy, the other FP32 with many measurements.
        dict(name="mcmc_bingham", kind="mcmc", signal="bingham", model="NODDI_Bingham", n=40000, b0=9, d1=30, d2=60,
             d3=0, burn=100, jumps=250, every=25, rician=False),
        dict(name="mcmc_sticks", kind="mcmc", signal="sticks2", model="Ball_2_Sticks", n=30000, b0=10, d1=90, d2=90,
             d3=90, burn=100, jumps=250, every=25, rician=False),
        # What follows the chains on a whole volume: sample means, mean orientations, dispersion maps,
        # predicted signal and model-selection scores.
        dict(name="maps_bingham", kind="maps", signal="bingham", model="NODDI_Bingham", n=200000, b0=9, d1=30, d2=60,
             d3=0, samples=50),
        # The network's starting points for a whole volume (500,000 voxels), and its training.
        dict(name="net_init", kind="net", signal="bingham", model="NODDI_Bingham", n=500000, b0=9, d1=30, d2=60, d3=0),
        dict(name="net_train", kind="train", signal="bingham", model="NODDI_Bingham", n=32768, b0=9, d1=30, d2=60, d3=0,
             batch=2048, epochs=2),
    ]


def draw(rng):
    """A case of the same ranges: another size (log-uniform up to the listed
    one of its kind), another acquisition, other options."""
    base = dict(rng.choice(listed()))
    name, kind = base.pop("name"), base["kind"]
    lo = {"lm": 50, "grid": 40, "mcmc": 100, "maps": 100, "net": 64, "train": 2048}[kind]
    hi = 5000 if name == "lm_stick_roi" else base["n"]
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    base["n"] = min(hi, n + rng.randrange(7))
    # another protocol with no more measurements than the listed one
    base["b0"] = rng.randint(2, base["b0"])
    for k in ("d1", "d2", "d3"):
        if base[k]:
            base[k] = rng.randint(max(9, base[k] // 3), base[k])
    if kind == "lm":
        base["iters"] = rng.randint(3, base["iters"])
        if name == "lm_watson" and rng.random() < 0.3:
            base["fixed"] = "2,3,4"  # the recipe's fit of the fractions alone
    elif kind == "grid" and base["model"] == "NODDI_Bingham" and rng.random() < 0.5:
        base["grid"], base["fixed"] = "psi", ""  # the learned start's scan over psi alone
        base["n"] = min(120000, base["n"] * rng.randint(1, 390))
    elif kind == "mcmc":
        base["every"] = rng.choice([5, 10, 25])
        base["jumps"] = base["every"] * rng.randint(1, 250 // base["every"])
        base["burn"] = rng.randint(1, 100)
        base["rician"] = rng.random() < 0.25
        if base["rician"]:
            base["n"] = min(base["n"], 4000)
    elif kind == "maps":
        base["samples"] = rng.randint(5, 50)
    elif kind == "train":
        base["batch"] = rng.choice([512, 1024, 2048])
        base["n"] = max(base["n"], base["batch"])
    return base


# ------------------------------------------------------------------ volumes

def _cfp(case):
    shells = [(b, case[k]) for b, k in zip(SHELLS[case["signal"]], ("d1", "d2", "d3")) if case[k]]
    return synth.acquisition(case["b0"], shells, seed=12)


def _nmeas(case):
    return case["b0"] + case["d1"] + case["d2"] + case["d3"]


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _uniform(g, n, lo, hi):
    return lo + (hi - lo) * torch.rand(n, generator=g, device="cuda", dtype=torch.float64)


def _angles(g, n):
    return torch.acos(_uniform(g, n, -1, 1)), _uniform(g, n, -math.pi, math.pi)


def _unit(th, ph):
    return torch.stack([th.sin() * ph.cos(), th.sin() * ph.sin(), th.cos()], -1)


def _fanning(th, ph, psi):
    """The fanning direction across the fibre (the Bingham plug-in's frame)."""
    a = torch.stack([-ph.sin(), ph.cos(), torch.zeros_like(ph)], -1)
    b = torch.stack([-th.cos() * ph.cos(), -th.cos() * ph.sin(), th.sin()], -1)
    return psi.cos()[:, None] * a + psi.sin()[:, None] * b


def _truth(kind, n, g):
    """Ground truths [n][P] (float64, the plug-in's parameter order)."""
    if kind == "sticks1":
        th, ph = _angles(g, n)
        return torch.stack([_uniform(g, n, 800, 1200), _uniform(g, n, 5e-4, 3e-3), _uniform(g, n, 0.1, 0.8), th, ph], 1)
    if kind == "sticks2":
        f1 = _uniform(g, n, 0.3, 0.6)
        f2 = f1 * _uniform(g, n, 0.2, 0.6)
        a, b = _angles(g, n), _angles(g, n)
        return torch.stack([_uniform(g, n, 800, 1200), _uniform(g, n, 5e-4, 3e-3), f1, a[0], a[1], f2, b[0], b[1]], 1)
    if kind == "tensor":
        th, ph = _angles(g, n)
        e1, psi = _unit(th, ph), _uniform(g, n, 0, math.pi)
        e2 = _fanning(th, ph, psi)
        e3 = torch.linalg.cross(e1, e2)
        t = 0
        for e in (e1, e2, e3):
            t = t + _uniform(g, n, 2e-4, 3e-3)[:, None, None] * e[:, :, None] * e[:, None, :]
        return torch.stack([_uniform(g, n, 800, 1200), t[:, 0, 0], t[:, 0, 1], t[:, 0, 2], t[:, 1, 1], t[:, 1, 2],
                            t[:, 2, 2]], 1)
    fiso, fin = _uniform(g, n, 0.02, 0.3), _uniform(g, n, 0.1, 0.9)
    th, ph = _angles(g, n)
    if kind == "watson":
        kappa = 1.0 / torch.tan(_uniform(g, n, 0.02, 0.9) * (math.pi / 2))
        return torch.stack([fiso, fin, kappa, th, ph], 1)
    kappa = _uniform(g, n, 1, 63)
    beta = torch.minimum(kappa * _uniform(g, n, 0.02, 0.95), kappa - 0.2).clamp(0.02, 31.0)
    return torch.stack([fiso, fin, kappa, beta, th, ph, _uniform(g, n, 0, math.pi)], 1)


def _sphere(count=3000):
    """Half of a Fibonacci lattice: the quadrature points of the orientation
    distributions (antipodally symmetric)."""
    k = torch.arange(count, device="cuda", dtype=torch.float64) + 0.5
    z = 1 - k / count
    r, a = (1 - z * z).sqrt(), k * (math.pi * (3 - math.sqrt(5)))
    return torch.stack([r * a.cos(), r * a.sin(), z], 1)


def _signal(kind, t, cfp, s0=None):
    """Noise-free signals [n][M] (float64)."""
    c = torch.as_tensor(cfp, device="cuda", dtype=torch.float64)
    grad, b = c[:, :3], c[:, 3]
    if kind in ("sticks1", "sticks2"):
        bd = b * t[:, 1:2]
        out = (1 - t[:, 2:3] - (t[:, 5:6] if kind == "sticks2" else 0)) * torch.exp(-bd)
        for k in ((2, 5) if kind == "sticks2" else (2,)):
            out = out + t[:, k:k + 1] * torch.exp(-bd * (_unit(t[:, k + 1], t[:, k + 2]) @ grad.T) ** 2)
        return t[:, :1] * out
    if kind == "tensor":
        q = torch.stack([grad[:, 0] ** 2, 2 * grad[:, 0] * grad[:, 1], 2 * grad[:, 0] * grad[:, 2], grad[:, 1] ** 2,
                         2 * grad[:, 1] * grad[:, 2], grad[:, 2] ** 2], 0)
        return t[:, :1] * torch.exp(-b * (t[:, 1:] @ q))
    pts = _sphere()
    sticks = torch.exp(-b * DPAR * (pts @ grad.T) ** 2).float()
    pairs = (pts[:, :, None] * pts[:, None, :]).reshape(-1, 9).float()
    out = torch.empty((t.shape[0], len(b)), device="cuda", dtype=torch.float64)
    for a in range(0, t.shape[0], 32768):
        u = t[a:a + 32768]
        th, ph = (u[:, 3], u[:, 4]) if kind == "watson" else (u[:, 4], u[:, 5])
        w = u[:, 2:3].float() * (_unit(th, ph).float() @ pts.T.float()) ** 2
        if kind == "bingham":
            w = w + u[:, 3:4].float() * (_fanning(th, ph, u[:, 6]).float() @ pts.T.float()) ** 2
        w = torch.softmax(w, 1)
        tens = (w @ pairs).double().reshape(-1, 3, 3)
        dperp = DPAR * (1 - u[:, 1:2])
        gtg = ((tens @ grad.T) * grad.T).sum(1)
        extra = torch.exp(-b * (dperp + (DPAR - dperp) * gtg))
        fan = (1 - u[:, 1:2]) * extra + u[:, 1:2] * (w @ sticks).double()
        out[a:a + 32768] = (1 - u[:, :1]) * fan + u[:, :1] * torch.exp(-b * DISO)
    return out * s0


def _volume(case, seed):
    """(truth, cfp, s0 [n][1] or None, noisy measurements [n][M])."""
    g, n, kind = _gen(seed), case["n"], case["signal"]
    cfp = _cfp(case)
    t = _truth(kind, n, g)
    s0 = _uniform(g, n, 800, 1200)[:, None] if kind in ("watson", "bingham") else None
    meas = _signal(kind, t, cfp, s0).float()
    sigma = (t[:, :1] if s0 is None else s0).float() / 25.0
    for k in (0, 1):
        noise = torch.randn(meas.shape, generator=g, device="cuda") * sigma
        meas = meas + noise if k == 0 else torch.sqrt(meas * meas + noise * noise)
    return t, cfp, None if s0 is None else s0.float().contiguous(), meas.contiguous()


def _near(t, kind, seed, rel):
    """Starting points a few per cent off the truth, inside the bounds."""
    g = _gen(seed + 1000003)
    p = t * (1 + rel * torch.randn(t.shape, generator=g, device="cuda", dtype=torch.float64))
    if kind in ("watson", "bingham"):
        p[:, 0:2] = p[:, 0:2].clamp(0.01, 0.99)
        p[:, 2] = p[:, 2].clamp(0.2, 63)
        if kind == "bingham":
            p[:, 3] = torch.minimum(p[:, 3], p[:, 2] - 0.2).clamp(0.02, 31)
    elif kind == "sticks2":
        p[:, 5] = torch.minimum(p[:, 5], 0.95 * p[:, 2])
    return p.float().contiguous()


# -------------------------------------------------------------------- cases

def prepare(case, seed):
    kind = case["kind"]
    if kind == "maps":
        # samples of converged chains: scattered about the truth
        g = _gen(seed)
        t = _truth("bingham", case["n"], g)
        s0 = _uniform(g, case["n"], 800, 1200)[:, None]
        cfp = _cfp(case)
        meas = _signal("bingham", t, cfp, s0).float()
        meas = meas + torch.randn(meas.shape, generator=g, device="cuda") * (s0.float() / 25)
        x = t.float()[:, :, None] * (1 + 0.03 * torch.randn((case["n"], 7, case["samples"]), generator=g, device="cuda"))
        x[:, 3] = torch.minimum(x[:, 3], x[:, 2] - 0.1)
        return dict(kind=kind, model=capi.Model(case["model"]), samples=x.contiguous(), meas=meas,
                    cfp=torch.as_tensor(cfp, dtype=torch.float32).cuda(), s0=s0.float().contiguous())
    if kind in ("net", "train"):
        t, cfp, s0, meas = _volume(case, seed)
        st = dict(kind=kind, scale=s0[:, 0].contiguous(), meas=meas)
        if kind == "net":
            st["net"] = capi.Mlp(cfp.shape[0], learned.head("NODDI_Bingham"), learned.WIDTH, learned.DEPTH, seed=7)
            st["p_init"] = torch.tensor([0.2, 0.7, 5, 2, 1.5, 1.5, 1.5], device="cuda").repeat(case["n"], 1)
        else:
            st.update(truth=t.float().contiguous(), clean=_signal("bingham", t, cfp, 1.0).float().contiguous(),
                      batch=case["batch"], epochs=case["epochs"], seed=seed % 1000)
        return st
    t, cfp, s0, meas = _volume(case, seed)
    m = capi.Model(case["model"])
    st = dict(kind=kind, model=m, meas=meas, cfp=torch.as_tensor(cfp, dtype=torch.float32).cuda(), s0=s0)
    if case.get("fixed"):
        m.set_fixed(case["fixed"])
    if kind == "lm":
        if case["signal"] == "tensor":  # the tensor frame's start: S0 from b = 0, D = 1e-3 I
            p = torch.zeros((case["n"], 7), device="cuda")
            p[:, 0] = meas[:, :case["b0"]].mean(1)
            p[:, 1] = p[:, 4] = p[:, 6] = 1e-3
        else:
            p = _near(t, case["signal"], seed, 0.05)
        st.update(start=p, iters=case["iters"])
    elif kind == "grid":
        if case["grid"] == "psi":
            m.load_grid(PSI_GRID, is_text=True)
            p = _near(t, "bingham", seed, 0.05)
        elif case["signal"] == "sticks2":
            m.load_grid(STICKS_GRID, is_text=True)
            p = t.float()
            p[:, 0] = meas[:, :case["b0"]].mean(1)
            p[:, 1] = 2e-3
        else:
            m.load_grid(pipelines.WATSON_GRID if case["signal"] == "watson" else pipelines.BINGHAM_GRID, is_text=True)
            p = t.float()
        st["start"] = p.contiguous()
    else:
        st.update(start=_near(t, case["signal"], seed, 0.02), burn=case["burn"], jumps=case["jumps"],
                  every=case["every"], rician=case["rician"], seed=seed % 100000)
    return st


def run(st):
    kind = st["kind"]
    if kind == "lm":
        p = st["start"].clone()
        cost = torch.empty(p.shape[0], device="cuda")
        st["model"].levmar(st["meas"], p, st["cfp"], st["s0"], max_iters=st["iters"], cost=cost)
        return {"params": p, "cost": cost}
    if kind == "grid":
        p = st["start"].clone()
        kept = torch.empty(p.shape[0], dtype=torch.int32, device="cuda")
        st["model"].gridsearch(st["meas"], p, st["cfp"], st["s0"], kept=kept)
        return {"params": p, "kept": kept}
    if kind == "mcmc":
        p = st["start"].clone()
        ns = st["jumps"] // st["every"]
        x = torch.empty((p.shape[0], p.shape[1], ns), device="cuda")
        tau = torch.empty((p.shape[0], ns), device="cuda") if st["rician"] else None
        st["model"].mcmc(st["meas"], p, st["cfp"], st["s0"], x, tau, nburn=st["burn"], njumps=st["jumps"],
                         sampleevery=st["every"], rician=st["rician"], seed=st["seed"])
        return {"params": p, "samples": x} if tau is None else {"params": p, "samples": x, "tau": tau}
    if kind == "maps":
        x, m = st["samples"], st["model"]
        n = x.shape[0]
        new = lambda *s: torch.empty(s, device="cuda")  # noqa: E731
        out = dict(mean=new(n, 7), fibre=new(n, 3), spread=new(n), fan=new(n, 3), maps=new(n, 5),
                   predicted=new(n, st["meas"].shape[1]), bic=new(n), aic=new(n))
        capi.sample_mean(x, out["mean"])
        capi.dyads(x, 4, 5, out["fibre"], out["spread"])
        capi.dyads(x, 4, 5, out["fan"], None, psi=6)
        capi.noddi_maps(x, 2, out["maps"], beta=3)
        m.predicted_signal(x, st["cfp"], st["s0"], out["predicted"])
        m.bic_aic(st["meas"], x, st["cfp"], st["s0"], out["bic"], out["aic"])
        return out
    if kind == "net":
        p = st["p_init"].clone()
        out = torch.empty((p.shape[0], st["net"].n_out), device="cuda")
        st["net"].forward(st["meas"], st["scale"], out)
        st["net"].init_params(st["meas"], st["scale"], p)
        return {"outputs": out, "params": p}
    net = capi.Mlp(st["clean"].shape[1], learned.head("NODDI_Bingham"), learned.WIDTH, learned.DEPTH, seed=7)
    losses = net.train(st["clean"], None, st["truth"], epochs=st["epochs"], batch=st["batch"], lr=2e-3, seed=st["seed"])
    return {"weights": net.get_weights(), "losses": losses}


def work(case):
    """Inputs read once, outputs written once; operations of the forward
    models where they are distinct (per voxel and measurement: about 40 for a
    stick or tensor signal, 180 for a NODDI one of which a change of the
    fractions alone needs 10)."""
    n, m = case["n"], _nmeas(case)
    kind, model = case["kind"], case.get("model")
    P = {"Ball_1_Stick": 5, "Ball_2_Sticks": 8, "DiffusionTensor": 7, "NODDI_Watson": 5, "NODDI_Bingham": 7}[model]
    one = {"Ball_1_Stick": 30, "Ball_2_Sticks": 50, "DiffusionTensor": 30, "NODDI_Watson": 110, "NODDI_Bingham": 180}[model]
    if kind == "lm":
        # a Jacobian row and its products, and one cost evaluation, per iteration
        row = 2 * one + P * (P + 3) if not model.startswith("NODDI") else 2 * (P - 2) * one + P * (P + 3)
        return {"bytes": 4.0 * n * (m + 2 * P + 1), "flops": float(n) * min(case["iters"], 15) * m * (row + one)}
    if kind == "grid":
        # distinct forward models, then three sums per combination of the parameters they are linear in
        basis = {"psi": 12 * one}.get(case["grid"]) or {"Ball_2_Sticks": 2 * 9 * 15 + 81 * 12, "NODDI_Watson": 88 * 15 + 8 * 60,
                                                        "NODDI_Bingham": 170 * 10 * 15 + 170 * 150}[model]
        return {"bytes": 4.0 * n * (m + 2 * P + 1), "flops": float(n) * m * basis}
    if kind == "mcmc":
        deep = {"Ball_2_Sticks": 3 * 8 + 4 * 25 + 50, "NODDI_Bingham": 5 * 180 + 2 * 40}[model]
        return {"bytes": 4.0 * n * (m + 2 * P + P * (case["jumps"] // case["every"])),
                "flops": float(n) * (case["burn"] + case["jumps"]) * m * deep * (2 if case["rician"] else 1)}
    if kind == "maps":
        return {"bytes": 4.0 * n * (7 * case["samples"] + 2 * m + 22), "flops": float(n) * (150 * case["samples"] + 2 * 180 * m)}
    layers = m * 256 + 2 * 256 * 256 + 256 * 7
    if kind == "net":
        return {"bytes": 4.0 * n * (m + 7 + 14), "flops": 2.0 * 2 * n * layers}
    steps = case["epochs"] * (n // case["batch"])
    return {"bytes": 4.0 * steps * case["batch"] * (m + 7) + 4.0 * layers, "flops": 6.0 * steps * case["batch"] * layers}


# -------------------------------------------------------------------- exact

def _principal(d):
    """Principal axis of the mean dyadic of directions [n][S][3], z >= 0."""
    m = (d[:, :, :, None] * d[:, :, None, :]).mean(1)
    w, v = torch.linalg.eigh(m.cpu())
    e = v[:, :, 2]
    key = torch.where(e[:, 2] != 0, e[:, 2], torch.where(e[:, 1] != 0, e[:, 1], e[:, 0]))
    return e * torch.where(key < 0, -1.0, 1.0)[:, None], 1.0 - w[:, 2]


def _exact_sticks_grid(case, seed):
    st = prepare(case, seed)
    y, p = st["meas"].double(), st["start"].double()
    cfp = st["cfp"].double()
    grad, b = cfp[:, :3], cfp[:, 3]
    f32 = lambda v: float(np.float32(v))  # noqa: E731
    ax = {k: [f32(x) for x in v] for k, v in STICKS_AXES.items()}
    bd = b * p[:, 1:2]
    ball = torch.exp(-bd)

    def stick(th, ph):
        n = torch.tensor([math.sin(th) * math.cos(ph), math.sin(th) * math.sin(ph), math.cos(th)], device="cuda",
                         dtype=torch.float64)
        return torch.exp(-bd * (grad @ n) ** 2)
    first = [(a, c, stick(a, c)) for a in ax[3] for c in ax[4]]
    second = [(a, c, stick(a, c)) for a in ax[6] for c in ax[7]]
    best = torch.full((case["n"],), math.inf, device="cuda", dtype=torch.float64)
    out = p.clone()
    for f1 in ax[2]:
        for t1, h1, s1 in first:
            for f2 in ax[5]:
                for t2, h2, s2 in second:
                    s = p[:, :1] * ((1 - f1 - f2) * ball + f1 * s1 + f2 * s2)
                    c = ((s - y) ** 2).sum(1)
                    better = c < best
                    best = torch.where(better, c, best)
                    out[better, 2:] = torch.tensor([f1, t1, h1, f2, t2, h2], device="cuda", dtype=torch.float64)
    return {"params": out, "kept": None}


def exact(case, seed):
    kind = case["kind"]
    if kind == "grid" and case["signal"] == "sticks2":
        return _exact_sticks_grid(case, seed)
    if kind == "maps":
        x = prepare(case, seed)["samples"].double()
        th, ph, psi = x[:, 4], x[:, 5], x[:, 6]
        fibre, spread = _principal(_unit(th, ph))
        n, S = th.shape
        fan, _ = _principal(_fanning(th.reshape(-1), ph.reshape(-1), psi.reshape(-1)).reshape(n, S, 3))
        k, bt = x[:, 2].mean(1), x[:, 3].mean(1)
        k2 = (x[:, 2] - x[:, 3]).mean(1)
        at = lambda v: torch.atan(v) * (2 / math.pi)  # noqa: E731
        maps = torch.stack([k2, at(1 / k2), at(1 / k), at(torch.sqrt(1 / (k * k2))), at(bt / k2)], 1)
        return dict(mean=x.mean(2), fibre=fibre, spread=spread, fan=fan, maps=maps, predicted=None, bic=None, aic=None)
    if kind == "net":
        st = prepare(case, seed)
        net, w, at = st["net"], st["net"].get_weights(), 0
        h = st["meas"].double() / st["scale"].double()[:, None]
        shapes = net.layer_shapes()
        for k, (rows, cols) in enumerate(shapes):
            wk = torch.as_tensor(w[at:at + rows * cols].reshape(rows, cols)).cuda().double()
            bk = torch.as_tensor(w[at + rows * cols:at + rows * cols + rows]).cuda().double()
            at += rows * cols + rows
            h = h @ wk.T + bk
            if k + 1 < len(shapes):
                h = torch.nn.functional.gelu(h)
        return {"outputs": h, "params": None}
    return None
