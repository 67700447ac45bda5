"""Benchmark of the fitting path: NODDI-Bingham LM + MCMC, learned start.

One step over one synthetic NODDI-Bingham volume of 500,000 voxels already
resident in HBM.  The acquisition has 9 b=0 + 30 directions at b=700 + 60 at
b=2000 (99 measurements). The truths are kappa1 U[1,64], kappa2/kappa1 U[0,1],
psi U[0,pi), fiso U[0,0.3], fintra U[0.1,0.9], S0 = 1000, Rician noise at
SNR 25. One step is:
  learned start    the network's fiso, fintra, kappa, beta, theta, phi plus a
                   12-point psi scan (cudimot_amd.pipelines)
  LM               --iterLevMar 200, all parameters, with the GridSearch + LM
                   fallback for voxels whose residual exceeds the noise bound
  MCMC             the reference's defaults: 1000 burn-in jumps, 1250 jumps,
                   a sample every 25
The network is trained before timing, on 2M signals generated by the
plug-in's forward model with Rician noise at SNR U[10,50]. Its training
time is reported but is not part of the step.

Prints one JSON line: voxels/s (whole job), with
  roofline              the MCMC kernel (dominant; bound by vector-ALU issue).
                        Counted FP32/FP64 flops per launch over the launch's
                        average HIP-event duration, as a fraction of MI355X's
                        vector peaks (FP64 78.6, FP32 157.3 TFLOP/s):
                        frac = F64/(78.6e12 t) + F32/(157.3e12 t). achieved is
                        the FP64-equivalent rate.
  cpu_baseline          the FP64 CPU oracle (OpenMP, one voxel per iteration)
                        on a seeded 384-voxel sample, LM + MCMC from the same
                        starts; cores = the OpenMP team that ran
  fit_rmse              parameter RMSE vs the truth of the chains' last
                        states and of the MCMC posterior means, also split
                        into truths inside the reference's bounds
                        (beta <= 32, kappa - beta > 0.05) and outside them
  learned_vs_gridsearch learned start + LM against the reference pipeline's
                        tensor fit + GridSearch + LM on a held-out volume of
                        500,000 voxels: throughput, parameter RMSE, and which
                        start reaches the lower final sum of squares
  learned_init          the network's training

With --other-configs it measures the remaining configurations of the set
instead, one JSON line each (GPU voxels/s with the inputs resident in HBM,
beside the FP64 CPU oracle on a sample of the same volume):
  Ball_1_Stick   M=64,  10,000 voxels: LM (100 iterations) from P_init
  Ball_2_Sticks  M=280, 500,000 voxels: GridSearch (729 combinations) -> LM
                 (200) -> MCMC (1000 / 1250 / 25)
  NODDI_Watson   M=99,  500,000 voxels: tensor frame -> GridSearch (968
                 combinations, orientation fixed) -> LM (orientation fixed)
                 -> LM, the reference pipeline's recipe
  DiffusionTensor M=64, NODDI_Bingham_2Fans M=99, Ball_3_Sticks M=280,
                 400,000 voxels each: LM (200) -> MCMC (500 / 1250 / 25), one
                 batched call per method, from starts 5% off the truth
"""
import argparse
import json
import os
import sys
import time

import numpy as np

REPO = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, REPO)

PEAK_F64 = 78.6e12
PEAK_F32 = 157.3e12
# HBM bytes of the MCMC kernel at its tuned launch shape (per-measurement cache
# rows in LDS), from the rocprofv3 --pmc FETCH_SIZE and WRITE_SIZE passes over
# cudimot_amd/profile_workload.py (131,072 voxels, a 100-jump burn-in launch
# and a 100-jump launch recording 10 samples), scaled by the same counters'
# readings for a 512 MiB copy (fetch x2.0, write x1.0):
# - per voxel and launch: the measurements read, the chain state and
#   parameters written (721 B);
# - per voxel and jump: what reaches HBM of the 32 bytes of scratch per lane that
#   each step in an angle writes (4 lanes and 3 angles a voxel, 384 B at most;
#   burn-in launch: 309,283 + 3,003,687 KiB / 131,072 voxels, less the 721 B,
#   over 100 jumps);
# - per stored sample value: one 32-byte sector and more, since a launch stores
#   one sample of each parameter per recording and a parameter's samples lie
#   contiguous per voxel ((30,659 + 331,689) KiB / 9,175,040 stores).
MCMC_BYTES_PER_VOXEL_LAUNCH = 721.0
MCMC_BYTES_PER_VOXEL_JUMP = 251.6
MCMC_BYTES_PER_SAMPLE_STORE = 40.4
SNR = 25.0
S0 = 1000.0


def log(msg):
    print("bench: " + msg, file=sys.stderr, flush=True)


def make_volume(m, n, seed, torch):
    """Truth (host), cfp (host), d_cfp, s0 [n][1], noisy measurements (device).
    The truths follow the configuration's distribution as drawn (kappa1
    U[1,64], kappa2/kappa1 U[0,1]), so beta = kappa1 - kappa2 exceeds the
    reference's bound of 32 for some voxels; those are reported apart."""
    from cudimot_amd import synth
    cfp = synth.model_acquisition("NODDI_Bingham")
    t = synth.truth_noddi_bingham(n, seed)
    d_cfp = torch.as_tensor(cfp, dtype=torch.float32).cuda()
    d_s0 = torch.full((n, 1), S0, device="cuda")
    clean = torch.empty((n, cfp.shape[0]), device="cuda")
    m.predicted_signal(torch.as_tensor(t, dtype=torch.float32).cuda().reshape(n, 7, 1), d_cfp, d_s0, clean)
    g = torch.Generator(device="cuda").manual_seed(seed)
    sigma = S0 / SNR
    n1 = torch.randn(clean.shape, device="cuda", generator=g) * sigma
    n2 = torch.randn(clean.shape, device="cuda", generator=g) * sigma
    meas = torch.sqrt((clean + n1) ** 2 + n2 ** 2).contiguous()
    return t, cfp, d_cfp, d_s0, meas


def _axis(a):
    return np.stack([np.sin(a[:, 4]) * np.cos(a[:, 5]), np.sin(a[:, 4]) * np.sin(a[:, 5]), np.cos(a[:, 4])], 1)


def reachable(t):
    """Truths the reference's NODDI_Bingham can represent: beta <= 32 (its
    bounds[3], modelpriors:9) and kappa - beta > 0.05 (ConstraintsMCMC)."""
    return (t[:, 3] <= 32.0) & (t[:, 2] - t[:, 3] > 0.05)


def _rmse(p, t, axis_p=None):
    axis_p = _axis(p) if axis_p is None else axis_p
    ang = np.degrees(np.arccos(np.clip(np.abs(np.sum(axis_p * _axis(t), 1)), 0, 1)))
    r = {k: float(np.sqrt(np.mean((p[:, i] - t[:, i]) ** 2))) for i, k in enumerate(("fiso", "fintra", "kappa", "beta"))}
    r["axis_deg_mean"] = float(ang.mean())
    r["axis_deg_median"] = float(np.median(ang))
    return {k: round(v, 5) for k, v in r.items()}


def rmse_report(p, t, axis_p=None):
    """Parameter RMSE against the truth, over all voxels and split into the
    truths inside the reference's bounds and constraints and those outside
    (which no fit within them can reach)."""
    p = p.detach().cpu().numpy().astype(np.float64) if hasattr(p, "detach") else np.asarray(p, dtype=np.float64)
    ok = reachable(t)
    out = _rmse(p, t, axis_p)
    out["inside_bounds"] = dict(_rmse(p[ok], t[ok], None if axis_p is None else axis_p[ok]), voxels=int(ok.sum()))
    out["outside_bounds"] = dict(_rmse(p[~ok], t[~ok], None if axis_p is None else axis_p[~ok]),
                                 voxels=int((~ok).sum()))
    return out


def posterior_mean(samples, torch):
    """Posterior means of the chains: the sample mean of each scalar
    parameter, and the fibre axis as the principal eigenvector of the mean
    dyadic tensor of the sampled axes (the finish step's dyads)."""
    s = samples.double()
    mean = s.mean(2)
    th, ph = s[:, 4, :], s[:, 5, :]
    v = torch.stack([torch.sin(th) * torch.cos(ph), torch.sin(th) * torch.sin(ph), torch.cos(th)], 2)
    dyad = torch.einsum("nsi,nsj->nij", v, v) / v.shape[1]
    _, vecs = torch.linalg.eigh(dyad)
    return mean.cpu().numpy(), vecs[:, :, 2].cpu().numpy()


def host_cpu():
    """CPU model name and the CPUs this process may run on."""
    model = "unknown"
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                model = line.split(":", 1)[1].strip()
                break
    except OSError:
        pass
    try:
        avail = len(os.sched_getaffinity(0))
    except AttributeError:
        avail = os.cpu_count() or 1
    return model, avail


def dispersion(sec):
    """Per-voxel wall-clock seconds: median, 10th and 90th percentiles, max."""
    q = np.percentile(sec, [10, 50, 90])
    return {"p10": round(float(q[0]), 4), "median": round(float(q[1]), 4), "p90": round(float(q[2]), 4),
            "max": round(float(sec.max()), 4)}


def cpu_baseline(args, cfp, meas_np, p0_np, idx):
    """FP64 CPU oracle (OpenMP, one voxel per iteration) on a seeded voxel
    sample of the volume, LM + MCMC from the GPU pipeline's learned starts."""
    from oracle import bind
    from cudimot_amd import capi
    o = bind.OracleModel("NODDI_Bingham")
    spec = {k: np.asarray(v) for k, v in capi.Model("NODDI_Bingham").spec().items() if k != "init_provided"}
    ns = len(idx)
    fx = np.full((ns, 1), S0)
    s_lm, s_mc = np.zeros(ns), np.zeros(ns)
    t0 = time.time()
    p, _, _ = o.levmar(spec, meas_np, p0_np, cfp, fx, max_iters=args.lm_iters, seconds=s_lm)
    o.mcmc(spec, meas_np, p, cfp, fx, nburn=args.burnin, njumps=args.jumps, sampleevery=args.sampleevery,
           seed=args.seed, voxel_offset=0, seconds=s_mc)
    dt = time.time() - t0
    model, avail = host_cpu()
    threads = bind.omp_threads()
    return {"value": round(ns / dt, 3), "unit": "voxels/s", "cores": threads, "kind": "port",
            "sample": "%d voxels drawn (seed 0) from the same volume, the GPU pipeline's learned starts, full LM "
                      "(%d it.) + MCMC (%d+%d jumps, 1 sample/%d) in %.1f s on %d OpenMP threads" %
                      (ns, args.lm_iters, args.burnin, args.jumps, args.sampleevery, dt, threads),
            "cpu": model, "cpus_available": avail, "omp_threads": threads,
            "per_voxel_s": dispersion(s_lm + s_mc)}


BALL2_GRID = ("search[2]=(0.2,0.4,0.6)\nsearch[3]=(0.3,1.2,2.1)\nsearch[4]=(-2,0,2)\n"
              "search[5]=(0.0,0.1,0.2)\nsearch[6]=(0.6,1.5,2.4)\nsearch[7]=(-1,1,3)\n")


def _config_volume(model, n, seed, snr, torch):
    """Truth (host), cfp (host), d_cfp, fixp (S0 = 1000 where the model has
    one), Rician-noisy measurements (device)."""
    from cudimot_amd import capi, synth
    cfp = synth.model_acquisition(model)
    t = synth.truth_for(model, n, seed)
    m = capi.Model(model)
    d_cfp = torch.as_tensor(cfp, dtype=torch.float32).cuda()
    fx = torch.full((n, 1), S0, device="cuda") if m.fixp_tsize else None
    clean = torch.empty((n, cfp.shape[0]), device="cuda")
    m.predicted_signal(torch.as_tensor(t, dtype=torch.float32).cuda().reshape(n, -1, 1), d_cfp, fx, clean)
    scale = torch.as_tensor(t[:, :1], dtype=torch.float32).cuda() if fx is None else fx
    g = torch.Generator(device="cuda").manual_seed(seed)
    sig = scale / snr
    n1 = torch.randn(clean.shape, device="cuda", generator=g)
    n2 = torch.randn(clean.shape, device="cuda", generator=g)
    meas = torch.sqrt((clean + sig * n1) ** 2 + (sig * n2) ** 2).contiguous()
    return t, cfp, d_cfp, fx, meas


def _spec(model, fixed=None):
    from cudimot_amd import capi
    m = capi.Model(model)
    if fixed:
        m.set_fixed(fixed)
    return {k: np.asarray(v) for k, v in m.spec().items() if k != "init_provided"}


def other_configs(args):
    """The remaining configurations: one JSON line each on stdout.  Each CPU
    leg runs the FP64 oracle on a seeded random voxel sample of the same
    volume (one voxel per OpenMP iteration) and reports the per-voxel
    wall-clock dispersion; voxels are independent, so voxels/s scales."""
    import torch
    from oracle import bind
    from cudimot_amd import capi, pipelines, synth
    threads = bind.omp_threads()
    cpu_model, avail = host_cpu()
    f64 = lambda a: np.asarray(a, dtype=np.float32).astype(np.float64)
    host = lambda x: x.detach().cpu().numpy().astype(np.float64)

    def timed(fn):
        torch.cuda.synchronize()
        t0 = time.time()
        out = fn()
        torch.cuda.synchronize()
        return out, time.time() - t0

    def sample(n, k, seed):
        return np.sort(np.random.default_rng(seed).choice(n, min(k, n), replace=False))

    def report(name, n, method, gpu_s, cpu_vps, sec, note):
        line = {"config": name, "voxels": n, "method": method,
                "gpu": {"voxels_per_s": round(n / gpu_s, 1), "seconds": round(gpu_s, 3)},
                "cpu_baseline": {"voxels_per_s": round(cpu_vps, 3), "cores": threads, "kind": "port",
                                 "sample": note, "cpu": cpu_model, "cpus_available": avail,
                                 "per_voxel_s": dispersion(sec)},
                "ratio": round((n / gpu_s) / cpu_vps, 1)}
        print(json.dumps(line), flush=True)

    # Ball_1_Stick: LM x 100 from P_init (the CPU leg fits the whole volume)
    model, n = "Ball_1_Stick", 10000
    t, cfp, d_cfp, fx, meas = _config_volume(model, n, 11, 30.0, torch)
    m = capi.Model(model)
    sp = _spec(model)
    p0 = np.tile(np.asarray(sp["p_init"], dtype=np.float32), (n, 1))
    m.levmar(meas[:64].contiguous(), torch.as_tensor(p0[:64]).cuda(), d_cfp, None, max_iters=100)  # warm-up
    p = torch.as_tensor(p0).cuda()
    _, gs = timed(lambda: m.levmar(meas, p, d_cfp, None, max_iters=100))
    sec = np.zeros(n)
    t0 = time.time()
    bind.OracleModel(model).levmar(sp, host(meas), f64(p0), f64(cfp), None, max_iters=100, seconds=sec)
    dt = time.time() - t0
    report(model, n, "LM (100 it.) from P_init", gs, n / dt, sec,
           "LM from P_init on all %d voxels in %.1f s on %d OpenMP threads" % (n, dt, threads))
    log("Ball_1_Stick done")

    # Ball_2_Sticks: GridSearch -> LM -> MCMC
    model, n = "Ball_2_Sticks", 500000
    t, cfp, d_cfp, fx, meas = _config_volume(model, n, 12, 20.0, torch)
    m = capi.Model(model)
    sp = _spec(model)
    b0 = torch.as_tensor(cfp[:, 3] == 0).cuda()
    p0 = torch.as_tensor(np.tile(np.asarray(sp["p_init"], dtype=np.float32), (n, 1))).cuda()
    p0[:, 0] = meas[:, b0].mean(1)
    gp, grid = m.load_grid(BALL2_GRID, is_text=True)
    samples = torch.empty((n, 8, args.jumps // args.sampleevery), device="cuda")
    w = 4096
    m.gridsearch(meas[:w].contiguous(), p0[:w].clone(), d_cfp, None)  # warm-up
    m.levmar(meas[:w].contiguous(), p0[:w].clone(), d_cfp, None, max_iters=5)
    m.mcmc(meas[:w].contiguous(), p0[:w].clone(), d_cfp, None, samples[:w], None, nburn=2, njumps=2, sampleevery=1)
    p = p0.clone()

    def fit2():
        m.gridsearch(meas, p, d_cfp, None)
        m.levmar(meas, p, d_cfp, None, max_iters=args.lm_iters)
        m.mcmc(meas, p, d_cfp, None, samples, None, nburn=args.burnin, njumps=args.jumps,
               sampleevery=args.sampleevery, seed=args.seed)
    _, gs = timed(fit2)
    idx = sample(n, 512, 12)
    k = len(idx)
    o = bind.OracleModel(model)
    meas_k, p_k = host(meas)[idx], host(p0)[idx]
    s1, s2, s3 = np.zeros(k), np.zeros(k), np.zeros(k)
    t0 = time.time()
    pg, _ = o.gridsearch(sp, meas_k, p_k, f64(cfp), None, np.asarray(gp), np.asarray(grid), seconds=s1)
    pl, _, _ = o.levmar(sp, meas_k, pg, f64(cfp), None, max_iters=args.lm_iters, seconds=s2)
    o.mcmc(sp, meas_k, pl, f64(cfp), None, nburn=args.burnin, njumps=args.jumps, sampleevery=args.sampleevery,
           seed=args.seed, seconds=s3)
    dt = time.time() - t0
    report(model, n, "GridSearch (729) -> LM (%d) -> MCMC (%d/%d/%d)" % (args.lm_iters, args.burnin, args.jumps,
                                                                        args.sampleevery),
           gs, k / dt, s1 + s2 + s3,
           "the same three steps on %d voxels drawn from the volume in %.1f s on %d OpenMP threads" %
           (k, dt, threads))
    del samples
    log("Ball_2_Sticks done")

    # NODDI_Watson: the reference pipeline's recipe
    model, n = "NODDI_Watson", 500000
    t, cfp, d_cfp, fx, meas = _config_volume(model, n, 13, 25.0, torch)
    b0 = torch.as_tensor(pipelines.b0_mask(cfp)).cuda()
    s0 = meas[:, b0].mean(1, keepdim=True).contiguous()
    pipelines.watson_gridsearch_lm(meas[:w].contiguous(), cfp, s0[:w].contiguous(), lm_iters=5)  # warm-up

    def fit3():
        frame = pipelines.tensor_frame(meas, cfp)
        return pipelines.watson_gridsearch_lm(meas, cfp, s0, lm_iters=args.lm_iters, frame=frame), frame
    (_, frame), gs = timed(fit3)
    idx = sample(n, 1024, 13)
    k = len(idx)
    o = bind.OracleModel(model)
    gsm = capi.Model(model)
    gsm.set_fixed("3,4")
    gp, grid = gsm.load_grid(pipelines.WATSON_GRID, is_text=True)
    spg, spf, spa = _spec(model, "3,4"), _spec(model, "2,3,4"), _spec(model)
    meas_k, s0_k = host(meas)[idx], host(s0)[idx]
    pk = np.tile(np.asarray(spa["p_init"], dtype=np.float32), (k, 1)).astype(np.float64)
    pk[:, 3:5] = host(frame)[idx, 0:2]
    s1, s2, s3 = np.zeros(k), np.zeros(k), np.zeros(k)
    t0 = time.time()
    pg, _ = o.gridsearch(spg, meas_k, pk, f64(cfp), s0_k, np.asarray(gp), np.asarray(grid), seconds=s1)
    p1, _, _ = o.levmar(spf, meas_k, pg, f64(cfp), s0_k, max_iters=args.lm_iters, seconds=s2)
    o.levmar(spa, meas_k, p1, f64(cfp), s0_k, max_iters=args.lm_iters, seconds=s3)
    dt = time.time() - t0
    report(model, n, "tensor frame -> GridSearch (968) -> LM (orientation fixed) -> LM", gs, k / dt, s1 + s2 + s3,
           "GridSearch + LM + LM on %d voxels drawn from the volume, from the GPU's tensor-frame orientations, "
           "in %.1f s on %d OpenMP threads" % (k, dt, threads))
    log("NODDI_Watson done")

    # batched LM -> MCMC over three models
    models = [("DiffusionTensor", 51, 512), ("NODDI_Bingham_2Fans", 52, 48), ("Ball_3_Sticks", 53, 128)]
    n = 400000
    items, cpu = [], []
    offset = 0
    for name, seed, kc in models:
        t, cfp, d_cfp, fx, meas = _config_volume(name, n, seed, 20.0, torch)
        rng = np.random.default_rng(seed)
        start = t.copy()
        start[:, 1:] *= 1.0 + 0.05 * rng.normal(size=start[:, 1:].shape)
        start = synth.clip_to_bounds(name, start).astype(np.float32)
        h = capi.Model(name)
        P = h.nparams
        items.append(dict(model=h, meas=meas, params=torch.as_tensor(start).cuda(), cfp=d_cfp, fixp=fx,
                          samples=torch.empty((n, P, args.jumps // args.sampleevery), device="cuda"),
                          voxel_offset=offset))
        idx = sample(n, kc, seed)
        cpu.append((name, cfp, host(meas)[idx], start[idx].astype(np.float64),
                    None if fx is None else np.full((len(idx), 1), S0)))
        offset += n
    capi.batch_levmar([dict(it, meas=it["meas"][:w].contiguous(), params=it["params"][:w].clone(),
                            fixp=None if it["fixp"] is None else it["fixp"][:w].contiguous(),
                            samples=it["samples"][:w]) for it in items], max_iters=5)  # warm-up

    def fit5():
        capi.batch_levmar(items, max_iters=args.lm_iters)
        capi.batch_mcmc(items, nburn=500, njumps=args.jumps, sampleevery=args.sampleevery, seed=args.seed)
    _, gs = timed(fit5)
    # CPU time of the whole job: each model's seconds per voxel (its sample's
    # wall clock over its size) times its voxels
    total_s, secs, parts = 0.0, [], []
    for name, cfp, meas_k, p_k, fx_k in cpu:
        o = bind.OracleModel(name)
        sp = _spec(name)
        k = len(meas_k)
        s1, s2 = np.zeros(k), np.zeros(k)
        t0 = time.time()
        pl, _, _ = o.levmar(sp, meas_k, p_k, f64(cfp), fx_k, max_iters=args.lm_iters, seconds=s1)
        o.mcmc(sp, meas_k, pl, f64(cfp), fx_k, nburn=500, njumps=args.jumps, sampleevery=args.sampleevery,
               seed=args.seed, seconds=s2)
        dt = time.time() - t0
        total_s += n * dt / k
        secs.append(s1 + s2)
        parts.append("%s %d voxels in %.1f s" % (name, k, dt))
    report("DiffusionTensor + NODDI_Bingham_2Fans + Ball_3_Sticks", 3 * n,
           "LM (%d) -> MCMC (500/%d/%d), one batched call per method" % (args.lm_iters, args.jumps,
                                                                        args.sampleevery),
           gs, 3 * n / total_s, np.concatenate(secs),
           "LM + MCMC per model on voxels drawn from its volume (%s) on %d OpenMP threads; the job's CPU time is "
           "each model's seconds per voxel times its 400,000 voxels" % ("; ".join(parts), threads))
    log("batched configuration done")


def main():
    ap = argparse.ArgumentParser(description=__doc__, formatter_class=argparse.RawDescriptionHelpFormatter)
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=2)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--voxels", type=int, default=500000)
    ap.add_argument("--warmup-voxels", type=int, default=8192, help="voxels of each (untimed) warm-up step")
    ap.add_argument("--lm-iters", type=int, default=200)
    ap.add_argument("--burnin", type=int, default=1000)
    ap.add_argument("--jumps", type=int, default=1250)
    ap.add_argument("--sampleevery", type=int, default=25)
    ap.add_argument("--seed", type=int, default=8219)
    ap.add_argument("--train-samples", type=int, default=2000000)
    ap.add_argument("--train-epochs", type=int, default=30)
    ap.add_argument("--compare-voxels", type=int, default=500000,
                    help="held-out voxels of the learned vs GridSearch comparison (0: skip)")
    ap.add_argument("--lanes", type=int, default=0, help="voxel-group size for LM and MCMC (0: automatic)")
    ap.add_argument("--cpu-sample", type=int, default=384,
                    help="voxels of the CPU-oracle baseline, a seeded random sample of the volume (0: skip)")
    ap.add_argument("--other-configs", action="store_true",
                    help="measure the other configurations of the set instead (one JSON line each)")
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py measures one GPU: this build fits one GPU's voxel shard and has no multi-GPU path "
              "(voxels shard with no exchange; see the design notes).", file=sys.stderr)
        sys.exit(2)
    if args.other_configs:
        other_configs(args)
        return

    import torch
    from cudimot_amd import capi, flops, learned, pipelines

    assert torch.cuda.is_available(), "bench.py needs a HIP device"
    m = capi.Model("NODDI_Bingham")
    if args.lanes:
        m.set_group(capi.LEVMAR, args.lanes)
        m.set_group(capi.MCMC, args.lanes)
    stream = torch.cuda.current_stream()
    P = m.nparams
    nsamp = args.jumps // args.sampleevery

    # learned initialiser: trained on generated signals (not timed)
    t0 = time.time()
    net, losses = learned.train("NODDI_Bingham", n=args.train_samples, epochs=args.train_epochs, seed=args.seed)
    torch.cuda.synchronize()
    train_s = time.time() - t0
    log("network trained on %d signals x %d epochs in %.1f s (loss %.4f -> %.4f)" %
        (args.train_samples, args.train_epochs, train_s, losses[0], losses[-1]))

    def step(meas, d_cfp, d_s0, cfp, n, ev_mcmc=None):
        p, _, flagged = pipelines.bingham_learned_lm(meas, cfp, d_s0, net, lm_iters=args.lm_iters, stream=stream)
        samples = torch.empty((n, P, nsamp), device="cuda")
        if ev_mcmc:
            ev_mcmc[0].record(stream)
        m.mcmc(meas, p, d_cfp, d_s0, samples, None, nburn=args.burnin, njumps=args.jumps,
               sampleevery=args.sampleevery, seed=args.seed, stream=stream)
        if ev_mcmc:
            ev_mcmc[1].record(stream)
        return p, samples, flagged

    # warm-up on a small volume (module load, first launches)
    wt, wcfp, wd_cfp, wd_s0, wmeas = make_volume(m, args.warmup_voxels, args.seed + 7, torch)
    for _ in range(args.warmup):
        step(wmeas, wd_cfp, wd_s0, wcfp, args.warmup_voxels)
    torch.cuda.synchronize()

    truth, cfp, d_cfp, d_s0, meas = make_volume(m, args.voxels, args.seed, torch)
    torch.cuda.synchronize()
    log("warm-up done, timing %d step(s) of %d voxels" % (args.steps, args.voxels))
    mcmc_ev = []
    t0 = time.time()
    for k in range(args.steps):
        ev = (torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True))
        p_fit, samples, flagged = step(meas, d_cfp, d_s0, cfp, args.voxels, ev)
        mcmc_ev.append(ev)
        if k + 1 < args.steps:
            torch.cuda.synchronize()
            log("step %d done at %.1f s" % (k + 1, time.time() - t0))
    torch.cuda.synchronize()
    elapsed = time.time() - t0
    mcmc_s = np.mean([a.elapsed_time(b) for a, b in mcmc_ev]) / 1000.0
    value = args.voxels * args.steps / elapsed
    log("timed steps: %.1f s (%.1f voxels/s)" % (elapsed, value))

    # counted work of the MCMC call (burn-in + recording launches)
    sub = np.random.default_rng(0).choice(args.voxels, 256, replace=False)
    ev = flops.per_eval("NODDI_Bingham", truth[sub], cfp, np.full((256, 1), S0))
    f32, f64 = flops.mcmc_flops(ev, P, cfp.shape[0], args.burnin + args.jumps)
    f32 *= args.voxels
    f64 *= args.voxels
    frac = f64 / (PEAK_F64 * mcmc_s) + f32 / (PEAK_F32 * mcmc_s)
    roofline = {"bound": "valu", "pipe": "vector ALU (FP64 + FP32), no matrix cores", "kernel": "cdm_mcmc_kernel",
                "achieved": round(frac * PEAK_F64 / 1e12, 3), "peak": PEAK_F64 / 1e12, "unit": "TFLOP/s",
                "frac": round(frac, 4),
                "traffic": args.voxels * (2 * MCMC_BYTES_PER_VOXEL_LAUNCH +
                                          (args.burnin + args.jumps) * MCMC_BYTES_PER_VOXEL_JUMP +
                                          P * nsamp * MCMC_BYTES_PER_SAMPLE_STORE) / 2,
                "traffic_note": "HBM bytes per launch (mean of the burn-in and recording launches) from rocprofv3 "
                                "FETCH_SIZE/WRITE_SIZE, copy-calibrated: measurements and chain state per voxel, "
                                "scratch written by the steps in an angle (252 B per voxel and jump), a sector per "
                                "stored sample; the cache rows stay in LDS: 0.1 TB/s, so the kernel is bound by "
                                "vector-ALU issue, not HBM",
                "flops_per_launch_f32": f32 / 2, "flops_per_launch_f64": f64 / 2,
                "avg_launch_ms": mcmc_s * 1000 / 2,
                "per_eval": {k: round(float(v), 2) for k, v in ev.items()}}

    out = {"metric": "voxels/s NODDI-Bingham LM+MCMC", "value": round(value, 2), "unit": "voxels/s", "n_gpus": 1,
           "steps": args.steps, "warmup": args.warmup, "ms_per_step": round(elapsed * 1000 / args.steps, 1),
           "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "f32+f64", "data": "synthetic",
           "config": {"workload": "NODDI_Bingham learned start + LM(200) + MCMC(1000/1250/25), 99 meas, SNR 25",
                      "voxels": args.voxels, "lanes_lm": m.get_group(capi.LEVMAR, cfp.shape[0], args.voxels),
                      "lanes_mcmc": m.get_group(capi.MCMC, cfp.shape[0], args.voxels),
                      "fallback_voxels": int(flagged.sum())},
           "roofline": roofline,
           "learned_init": {"train_samples": args.train_samples, "epochs": args.train_epochs,
                            "train_s": round(train_s, 2), "loss_first": round(float(losses[0]), 5),
                            "loss_last": round(float(losses[-1]), 5),
                            "network": "99-256-256-256-7 GELU, BF16 MFMA, FP32 accumulate"},
           "fit_rmse": {"chain_last_state": rmse_report(p_fit, truth)}}
    pm, axis_pm = posterior_mean(samples, torch)
    out["fit_rmse"]["posterior_mean"] = rmse_report(pm, truth, axis_pm)

    if args.compare_voxels > 0:
        nc = args.compare_voxels
        tc, ccfp, cd_cfp, cd_s0, cmeas = make_volume(m, nc, args.seed + 99, torch)
        # warm both pipelines on a few voxels (grid upload, first launches)
        pipelines.bingham_gridsearch_lm(cmeas[:256].contiguous(), ccfp, cd_s0[:256].contiguous())
        torch.cuda.synchronize()
        t0 = time.time()
        pl, cl, fl = pipelines.bingham_learned_lm(cmeas, ccfp, cd_s0, net, lm_iters=args.lm_iters)
        torch.cuda.synchronize()
        tl = time.time() - t0
        t0 = time.time()
        pg, cg = pipelines.bingham_gridsearch_lm(cmeas, ccfp, cd_s0, lm_iters=args.lm_iters)
        torch.cuda.synchronize()
        tg = time.time() - t0
        log("learned + LM %.2f s, GridSearch + LM %.2f s on %d voxels" % (tl, tg, nc))
        # which start reaches the lower sum of squares (relative tolerance 1e-4)
        r = (cl.double() / cg.double()).cpu().numpy()
        out["learned_vs_gridsearch"] = {
            "voxels": nc, "speedup": round(tg / tl, 2),
            "final_cost": {"learned_lower": round(float(np.mean(r < 1 - 1e-4)), 4),
                           "equal": round(float(np.mean(np.abs(r - 1) <= 1e-4)), 4),
                           "gridsearch_lower": round(float(np.mean(r > 1 + 1e-4)), 4),
                           "median_ratio": round(float(np.median(r)), 6)},
            "learned_lm": {"voxels_per_s": round(nc / tl, 1), "fallback_voxels": int(fl.sum()),
                           "rmse": rmse_report(pl, tc)},
            "gridsearch_lm": {"voxels_per_s": round(nc / tg, 1), "grid": "5x10x17x13 (fiso, fintra, kappa, beta)",
                              "rmse": rmse_report(pg, tc)}}

    if args.cpu_sample > 0:
        ns = min(args.cpu_sample, args.voxels)
        log("CPU oracle on %d voxels" % ns)
        idx = np.sort(np.random.default_rng(0).choice(args.voxels, ns, replace=False))
        d_idx = torch.as_tensor(idx).cuda()
        meas_s = meas[d_idx].contiguous()
        # the same learned starts as the GPU fit
        p0, _, _ = pipelines.bingham_learned_lm(meas_s, cfp, d_s0[d_idx].contiguous(), net, lm_iters=0,
                                                fallback=False)
        out["cpu_baseline"] = cpu_baseline(args, cfp, meas_s.cpu().numpy().astype(np.float64),
                                           p0.cpu().numpy().astype(np.float64), idx)
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
