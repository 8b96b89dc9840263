"""The work that users of this framework have it do, one dict per case.

    listed()            the cases that are timed
    draw(rng)           one more case of the same ranges
    prepare(case, seed) what a program holds before the call: contexts with
                        their fields, networks with their weights, host arrays
    run(state)          one pass through the public entry points
    work(case)          bytes and flops that a pass cannot do without
    exact(case, seed)   what run() returns, in 64-bit torch / numpy

Kinds of case
  step         one Parker step of caller-supplied states (sp_step_once), as
               an integrator that keeps its own particles calls it
  interval     one MHD interval of a fresh population: inject, move, split,
               quick check, f(p) and the spatial map; with "host" the
               population comes from and returns to host arrays instead
  frames       one interval of a run over a series of snapshots with linear
               interpolation in time: the next frame is uploaded and prepared
  sweep        a batch of parameter variants on one snapshot, two intervals,
               f(p) of every variant after each
  diagnostics  quick check, f(p) and maps of a population with split weights
  fit          training of one f(p) surrogate network from its initial weights
  predict      spectra from an ensemble of two networks, host arrays
  predict_dev  the same with query rows and spectra in device memory
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "stochastic-parker_amd"))
from sp_hip import ParkerPusher, workloads  # noqa: E402
from sp_hip.surrogate import FLOOR, Mlp, Surrogate  # noqa: E402

KPARA0 = 1e-3
WHOLE_BOX = (0.0, 0.0, 0.0, 1.0, 1.0, 1.0)
SQRT3 = math.sqrt(3.0)


def listed():
    return [
        # smallest call: a thousand particles of a user's own integrator
        dict(name="step_2d_f64_1k", kind="step", grid=128, nptl=1000, prec="f64"),
        # a trial run at the default precision, population on the host
        dict(name="interval_2d_f64_2k", kind="interval", ndim=2, grid=64, nptl=2000, nsteps=200,
             prec="f64", host=True, opts=""),
        # the 512^2 configuration: 1e5 particles, 1000 diffusion-limited steps
        dict(name="interval_2d_f32_1e5", kind="interval", ndim=2, grid=512, nptl=100000,
             nsteps=1000, prec="f32", host=False, opts=""),
        # the 2048^2 configuration, its interval cut to a tenth
        dict(name="interval_2d_f32_2e7", kind="interval", ndim=2, grid=2048, nptl=20000000,
             nsteps=200, prec="f32", host=False, opts=""),
        # 3D turbulence on FP16 records, a grid that fills no whole bricks
        dict(name="interval_3d_f32h_5e6", kind="interval", ndim=3, grid=190, nptl=5000000,
             nsteps=100, prec="f32h", host=False, opts=""),
        # 3D at the reference's arithmetic, kappa depending on |B|
        dict(name="interval_3d_f64_3e5", kind="interval", ndim=3, grid=64, nptl=300000,
             nsteps=100, prec="f64", host=False, opts="mag"),
        # the time loop of a run over real snapshots
        dict(name="frames_2d_f32_1e6", kind="frames", grid=1024, nptl=1000000, nsteps=100,
             prec="f32"),
        # parameter sweep: 64 variants of 1e3 .. 1e5 particles in one launch
        dict(name="sweep_64", kind="sweep", grid=512, nvar=64, nmin=1000, nmax=100000),
        # diagnostics of 3e6 particles, 128 x 128 map with 16 momentum bins
        dict(name="diagnostics_3e6", kind="diagnostics", grid=512, nptl=3000000, map=128),
        # surrogate training at the batch size of Surrogate.fit
        dict(name="fit_4096", kind="fit", nhidden=256, nlayers=4, nout=64, batch=4096, nsteps=100),
        # one spectrum query: eight times, both members, host arrays
        dict(name="predict_8", kind="predict", nhidden=256, nlayers=4, nout=64, rows=8),
        # a sweep of 1e5 queries resident in device memory
        dict(name="predict_dev_8e5", kind="predict_dev", nhidden=256, nlayers=4, nout=64,
             rows=800000),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "interval", "interval", "interval", "frames", "sweep",
                       "diagnostics", "fit", "predict", "predict_dev"])
    if kind == "step":
        return dict(kind=kind, grid=_log(rng, 24, 512), nptl=_log(rng, 100, 60000),
                    prec=rng.choice(["f64", "f32"]))
    if kind == "interval":
        ndim = rng.choice([2, 2, 3])
        prec = rng.choice(["f64", "f32", "f32h"])
        nsteps = _log(rng, 100, 800)
        # as many particle-steps as the largest listed case at most
        most = {2: {"f64": 1e9, "f32": 3e9, "f32h": 3e9}, 3: {"f64": 1e8, "f32": 4e8, "f32h": 4e8}}
        nptl = _log(rng, 500, most[ndim][prec] / nsteps)
        return dict(kind=kind, ndim=ndim, grid=_log(rng, 40, 2048) if ndim == 2 else _log(rng, 24, 190),
                    nptl=nptl, nsteps=nsteps, prec=prec, host=nptl < 20000 and rng.random() < 0.5,
                    opts=rng.choice(["", "", "mag", "acc"] + ([] if prec == "f32h" else ["dpp"])))
    if kind == "frames":
        return dict(kind=kind, grid=_log(rng, 64, 1024), nptl=_log(rng, 2000, 2000000), nsteps=100,
                    prec=rng.choice(["f32", "f32h", "f64"]))
    if kind == "sweep":
        return dict(kind=kind, grid=rng.choice([128, 256, 500, 512]), nvar=_log(rng, 3, 100),
                    nmin=_log(rng, 300, 3000), nmax=_log(rng, 5000, 60000))
    if kind == "diagnostics":
        return dict(kind=kind, grid=512, nptl=_log(rng, 1000, 3000000), map=rng.choice([32, 64, 128]))
    net = dict(nhidden=rng.choice([128, 256]), nlayers=rng.randint(2, 5), nout=rng.choice([32, 64, 128]))
    if kind == "fit":
        return dict(kind=kind, batch=_log(rng, 200, 8192), nsteps=rng.randint(20, 80), **net)
    if kind == "predict":
        return dict(kind=kind, rows=_log(rng, 1, 60000), **net)
    return dict(kind=kind, rows=_log(rng, 100, 400000), **net)


# ---- inputs -----------------------------------------------------------------
def _snapshot_2d(n, seed):
    """Node fields (1, n+4, n+4, 8) of a snapshot like workloads.fields_2d:
    two current sheets with a perturbed guide field and compressive flow."""
    r = np.random.default_rng(seed)
    c = (torch.arange(n + 4, dtype=torch.float64, device="cuda") - 2.0) / n
    x, y = c[None, :], c[:, None]
    tau = 2.0 * math.pi

    def modes(m):
        k = r.integers(1, 5, (m, 2)) * r.choice([-1, 1], (m, 2))
        return [(float(a), float(b), float(p), float(q)) for (a, b), p, q in
                zip(k, r.uniform(0, tau, m), r.uniform(0.5, 1.0, m))]

    dax, day = torch.zeros(n + 4, n + 4, dtype=torch.float64, device="cuda"), 0.0
    for kx, ky, ph, a in modes(8):
        s = -torch.sin(tau * (kx * x + ky * y) + ph)
        dax = dax + a * kx * s
        day = day + a * ky * s
    scale = 0.01 / (dax * dax + day * day).mean().sqrt()
    bx = torch.tanh((y - 0.25) / 0.02) - torch.tanh((y - 0.75) / 0.02) - 1.0 + scale * day
    by = -scale * dax
    bz = torch.full_like(bx, 0.1)
    vx = vy = 0.0
    for (kx, ky, ph, a), th in zip(modes(16), r.uniform(0, tau, 16)):
        s = a * torch.sin(tau * (kx * x + ky * y) + ph)
        vx, vy = vx + math.cos(th) * s, vy + math.sin(th) * s
    sv = 0.1 / (vx * vx + vy * vy).mean().sqrt()
    f = torch.stack([vx * sv, vy * sv, 0.0 * vx, 1.0 + 0.0 * vx, bx, by, bz,
                     (bx * bx + by * by + bz * bz).sqrt()], dim=-1)
    return f.float().cpu().numpy()[None]


def _snapshot_3d(n, seed):
    """Node fields (n+4, n+4, n+4, 8) like workloads.fields_3d: k^-5/3
    turbulence in B (solenoidal) and V (compressive), a compressed slab."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    k = torch.fft.fftfreq(n, 1.0 / n, device="cuda", dtype=torch.float64)
    kv = torch.stack(torch.meshgrid(k, k, k[: n // 2 + 1].abs(), indexing="ij")[::-1])
    ka = kv.square().sum(0).sqrt()
    amp = torch.where((ka >= 2) & (ka <= min(64, n // 2 - 1)), ka.clamp(min=1) ** (-11.0 / 6.0), 0.0 * ka)
    kh = kv / ka.clamp(min=1)
    idx = (torch.arange(n + 4, device="cuda") - 2) % n

    def field(solenoidal, rms):
        s = torch.fft.rfftn(torch.randn(3, n, n, n, generator=g, device="cuda", dtype=torch.float64),
                            dim=(1, 2, 3))
        along = kh * (kh * s).sum(0)
        f = torch.fft.irfftn((s - along if solenoidal else along) * amp, s=(n, n, n), dim=(1, 2, 3))
        f = f * (rms / f.square().sum(0).mean().sqrt())
        return f[:, idx][:, :, idx][:, :, :, idx]

    b, v = field(True, 0.5), field(False, 0.05)
    b[0] += 1.0
    x = (torch.arange(n + 4, dtype=torch.float64, device="cuda") - 2.0) / n
    v[0] += 0.15 - 0.05 * (1.0 + torch.tanh((x - 0.5) / 0.02))
    out = torch.stack([v[0], v[1], v[2], torch.ones_like(v[0]), b[0], b[1], b[2],
                       b.square().sum(0).sqrt()], dim=-1)
    return out.float().cpu().numpy()


def _config(case, ndim, nsteps, nptl_max, **over):
    c = (workloads.config_2d if ndim == 2 else workloads.config_3d)(case["grid"])
    # at least 100 (1000) steps in an interval
    c.update(precision=case.get("prec", "f32"), nptl_max=nptl_max, kpara0=KPARA0,
             dt_max_rel=1e-3 if nsteps >= 1000 else 1e-2)
    opts = case.get("opts", "")
    if opts == "mag":
        c.update(mag_dependency=1)
    elif opts == "acc":
        c.update(acc_region_flag=1, acc_region=(0.1, 0.8, 0.2, 0.9, 0.0, 0.7))
    elif opts == "dpp":
        c.update(dpp_wave=1, dpp_shear=1, tau0=1e-4)
    c.update(over)
    return c


def _dists(pz, ndim, n, bins=None):
    if bins is None:
        bins = min(128 if ndim == 2 else 32, n)
    r = max(1, n // bins)
    pz.init_particle_distributions(npp_global=256, nmu_global=1, local_dist=1, local=[
        dict(enabled=1, npbins=16, nmu=1, rx=r, ry=r, rz=r if ndim == 3 else 1, pmin=1e-2, pmax=1e4)])


def _pusher(cfg, seed, *frames):
    pz = ParkerPusher(**dict(cfg, seed=seed & 0x7FFFFFFF))
    for slot, f in enumerate(frames):
        pz.upload_fields(f, slot)
        pz.calc_fields_gradients(slot)
    return pz


def _host_population(n, ndim, seed, splits=0):
    """Host particle arrays: uniform positions, momenta p0 with a power-law
    tail above it, split copies of weight 2^-k."""
    r = np.random.default_rng(seed)
    k = r.integers(0, splits + 1, n)
    p = np.where(r.random(n) < 0.7, np.exp(0.05 * r.standard_normal(n)),
                 r.pareto(3.0, n) + 1.0)
    return dict(x=r.random(n), y=r.random(n), z=r.random(n) if ndim == 3 else np.zeros(n),
                p=p, v=5.0 * p, mu=0.99 * (2.0 * r.random(n) - 1.0), weight=0.5 ** k,
                t=np.zeros(n), dt=np.full(n, 1e-7) * (1.0 + r.random(n)),
                split_times=k.astype(np.int8), count_flag=np.ones(n, np.int8),
                origin=np.zeros(n, np.int32), nsteps_tracked=np.zeros(n, np.int32),
                nsteps_pushed=np.zeros(n, np.int32), tag_injected=np.arange(n, dtype=np.int32),
                tag_splitted=np.ones(n, np.int32), rng_step=np.zeros(n, np.uint32))


def _no_particles():
    return {k: v[:0] for k, v in _host_population(1, 2, 0).items()}


def _weights(case, seed):
    """Parameters of one network as after training: U(-1/sqrt(K), 1/sqrt(K))
    layers, outputs around log10 f = -2."""
    r = np.random.default_rng(seed)
    dims = [6] + [case["nhidden"]] * case["nlayers"] + [case["nout"]]
    parts = []
    for k, n in zip(dims[:-1], dims[1:]):
        a = 1.7 / math.sqrt(k)
        parts += [r.uniform(-a, a, k * n), r.uniform(-a, a, n)]
    parts[-1] = parts[-1] - 2.0
    return np.concatenate(parts).astype(np.float32)


def _query_rows(rows, seed):
    return np.random.default_rng(seed + 5).uniform(-1.0, 1.0, (rows, 6)).astype(np.float32)


def _step_inputs(case, seed):
    r = np.random.default_rng(seed + 1)
    n = case["nptl"]
    dtf = workloads.interval_2d(case["grid"], 1000, KPARA0)
    st = np.stack([r.random(n), r.random(n), np.zeros(n), np.exp(0.3 * r.standard_normal(n)),
                   dtf * 0.9 * r.random(n), np.full(n, dtf * 1e-3)], axis=1)
    rands = (2.0 * r.random((n, 4)) - 1.0) * SQRT3
    return dtf, st, rands, (r.random(n) < 0.05).astype(np.int8)


class _DeviceRows:
    """A torch tensor as the device array that Surrogate.predict_device takes."""

    def __init__(self, t):
        self.t, self.shape, self.dtype, self.ptr = t, tuple(t.shape), np.dtype(np.float32), t.data_ptr()


def _surrogate(case, seed):
    s = Surrogate(members=2, nhidden=case["nhidden"], nlayers=case["nlayers"], nbins=case["nout"])
    for i, net in enumerate(s.nets):
        net.set_params(_weights(case, seed + i))
    return s


def _fit_data(case, seed):
    r = np.random.default_rng(seed + 9)
    x = r.uniform(-1.0, 1.0, (40000, 6)).astype(np.float32)
    c = np.linspace(-1.0, 1.0, case["nout"])
    w = 0.15 + 0.1 * x[:, :1] + 0.05 * x[:, 5:]
    y = np.log10(np.exp(-(((c - 0.3 * x[:, 1:2]) / w) ** 2)) / 20.0 + FLOOR)
    return x, y.astype(np.float32)


def prepare(case, seed):
    kind, s = case["kind"], dict(case=case)
    if kind == "step":
        dtf, st, rands, fixed = _step_inputs(case, seed)
        s.update(dtf=dtf, st=st, rands=rands, fixed=fixed,
                 pz=_pusher(_config(case, 2, 1000, 1024), seed, _snapshot_2d(case["grid"], seed)))
    elif kind in ("interval", "frames", "sweep"):
        ndim, n = case.get("ndim", 2), case["grid"]
        snap = _snapshot_2d if ndim == 2 else _snapshot_3d
        s["none"] = _no_particles()
        if kind == "sweep":
            v = workloads.sweep_variants(case["nvar"], case["nmin"], case["nmax"], seed=seed)
            # the settings of the surrogate's training runs (SweepSDE)
            cfg = _config(case, 2, 100, int(v["nptl"].sum()), pmin=0.5, pmax=2.0)
            s["v"] = v
            pz = _pusher(cfg, seed, snap(n, seed))
            pz.init_particle_distributions(npp_global=64, nmu_global=1)
            pz.set_variants(list(zip(v["kpara0"], v["kret"], v["gamma_turb"])))
        else:
            ti = kind == "frames"
            s["dtf"] = workloads.interval_2d(n, case["nsteps"], KPARA0)
            cfg = _config(case, ndim, case["nsteps"], int(1.2 * case["nptl"]) + 8, time_interp=int(ti))
            if case.get("host"):
                # a closed box: as many particles come back as went in
                cfg.update(pbcx=0, pbcy=0, pbcz=0)
            frames = [snap(n, seed + 100 * i) for i in range(2 if ti else 1)]
            s["frames"], s["at"] = (frames, 0) if ti else ([], 0)
            pz = _pusher(cfg, seed, *frames)
            _dists(pz, ndim, n)
            if case.get("host"):
                s["ptl"] = _host_population(case["nptl"], ndim, seed)
        s["pz"] = pz
    elif kind == "diagnostics":
        s["pz"] = pz = ParkerPusher(**workloads.config_2d(case["grid"], nptl_max=case["nptl"]))
        _dists(pz, 2, case["grid"], case["map"])
        pz.set_particles(_host_population(case["nptl"], 2, seed, splits=3))
        pz.sort_particles()  # the order that a mover call leaves
    elif kind == "fit":
        s["net"] = net = Mlp(6, case["nhidden"], case["nlayers"], case["nout"],
                             batch_max=case["batch"], seed=seed & 0xFFFF)
        s["p0"], s["seed"] = net.get_params(), seed
        net.set_data(*_fit_data(case, seed))
    else:
        s["net"] = _surrogate(case, seed)
        x = _query_rows(case["rows"], seed)
        if kind == "predict":
            s["x"] = x
        else:
            s["x"] = _DeviceRows(torch.from_numpy(x).cuda())
            s["spec"] = _DeviceRows(torch.empty(case["rows"], case["nout"], device="cuda"))
            s["spread"] = _DeviceRows(torch.empty(case["rows"], device="cuda"))
    return s


# ---- one pass ---------------------------------------------------------------
def _diagnose(pz):
    fg, loc = pz.calc_particle_distributions()
    return dict(quick=pz.quick_check(), fglobal=fg, flocal=loc[0])


def _moved(st):
    return {k: st[k] for k in ("steps", "nptl_current", "nptl_escaped", "leak", "leak_negp")}


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "step":
        st, d = s["pz"].step_once(s["st"], s["rands"], s["fixed"], 0.0, s["dtf"])
        return dict(state=st, deltas=d)
    if kind == "interval" and case["host"]:
        pz = s["pz"]
        pz.set_particles(s["ptl"])
        st = pz.particle_mover(0.0, s["dtf"], 1, 10)
        out = _diagnose(pz)
        out.update(stats=_moved(st), particles=pz.get_particles())
        return out
    if kind in ("interval", "frames"):
        pz = s["pz"]
        if kind == "frames":
            pz.copy_fields()
            pz.upload_fields(s["frames"][s["at"] % 2], 1)
            pz.calc_fields_gradients(1)
            s["at"] += 1
        pz.set_particles(s["none"])
        pz.inject_particles_spatial_uniform(case["nptl"], 1e-7, 1, 5.0, 0.0, 0.0, WHOLE_BOX)
        st = pz.particle_mover(0.0, s["dtf"], 1, 10)
        pz.split_particle(2.0, 1.001)
        out = _diagnose(pz)
        out.update(stats=_moved(st))
        return out
    if kind == "sweep":
        pz, v = s["pz"], s["v"]
        pz.set_particles(s["none"])
        pz.inject_variants(v["nptl"], 1e-7, 1, 5.0, 0.0, 0.0, v["boxes"])
        out = []
        for k in range(2):
            st = pz.particle_mover(0.01 * k, 0.01, 1, 10)
            f, cnt = pz.variant_distributions()
            out.append(dict(f=f, counts=cnt, stats=_moved(st)))
        return out
    if kind == "diagnostics":
        return _diagnose(s["pz"])
    if kind == "fit":
        s["net"].set_params(s["p0"])
        losses = s["net"].train(case["nsteps"], case["batch"], 2e-3, 2e-5, s["seed"])
        return dict(losses=losses, params=s["net"].get_params())
    if kind == "predict":
        spec, est = s["net"].predict(s["x"])
        return dict(spec=spec, spread=est)
    s["net"].predict_device(s["x"], s["spec"], s["spread"])
    return dict(spec=s["spec"].t, spread=s["spread"].t)


# ---- what a pass cannot do without -------------------------------------------
def _net_flops(case):
    dims = [6] + [case["nhidden"]] * case["nlayers"] + [case["nout"]]
    return sum(2 * k * n for k, n in zip(dims[:-1], dims[1:]))


def work(case):
    kind = case["kind"]
    # arithmetic of one step: interpolation of 14 (19) values, the diffusion
    # tensor and its divergence, the push
    per_step = {2: 250, 3: 550}
    if kind == "step":
        return dict(bytes=(10 * 8 + 1 + 10 * 8) * case["nptl"], flops=250 * case["nptl"])
    if kind in ("interval", "frames"):
        nd, n = case.get("ndim", 2), case["nptl"]
        nodes = (case["grid"] + 4) ** nd
        return dict(bytes=2 * 98 * n + 32 * nodes * (2 if kind == "frames" else 1),
                    flops=per_step[nd] * n * max(100, case["nsteps"]))
    if kind == "sweep":
        v = workloads.sweep_variants(case["nvar"], case["nmin"], case["nmax"])
        steps = np.maximum(100, 0.01 * 2 * v["kpara0"] * (2 * case["grid"]) ** 2)
        return dict(bytes=4 * 98 * float(v["nptl"].sum()) + 32 * (case["grid"] + 4) ** 2,
                    flops=2 * 250 * float((v["nptl"] * steps).sum()))
    if kind == "diagnostics":
        return dict(bytes=56 * case["nptl"] + 8 * 16 * case["map"] ** 2, flops=30 * case["nptl"])
    if kind == "fit":
        params = _net_flops(case) // 2
        return dict(bytes=case["nsteps"] * (30 * params + 4 * case["batch"] * (6 + case["nout"])),
                    flops=3 * case["nsteps"] * case["batch"] * _net_flops(case))
    return dict(bytes=4 * case["rows"] * (7 + case["nout"]) + 4 * _net_flops(case),
                flops=2 * case["rows"] * _net_flops(case))


# ---- the same in 64 bits ------------------------------------------------------
def _exact_step(case, seed):
    """push_particle_2d on the interpolated node fields and their central
    differences (mag_dependency = 0, no out-of-plane drift)."""
    n = case["grid"]
    cfg = _config(case, 2, 1000, 1024)
    dtf, st, r, fixed = _step_inputs(case, seed)
    f8 = _snapshot_2d(n, seed)[0].astype(np.float64)
    g = np.zeros(f8.shape + (2,))
    g[:, 1:-1, :, 0] = (f8[:, 2:] - f8[:, :-2]) * (0.5 * n)
    g[1:-1, :, :, 1] = (f8[2:] - f8[:-2]) * (0.5 * n)
    x, y, z, p, t, dt = st.T
    px, py = x * n, y * n
    ix, iy = np.floor(px).astype(int), np.floor(py).astype(int)
    rx, ry = (px - ix)[:, None], (py - iy)[:, None]

    def interp(a):
        a = a.reshape(n + 4, n + 4, -1)
        return ((1 - rx) * (1 - ry) * a[iy + 2, ix + 2] + rx * (1 - ry) * a[iy + 2, ix + 3] +
                (1 - rx) * ry * a[iy + 3, ix + 2] + rx * ry * a[iy + 3, ix + 3])

    v = interp(f8)
    d = interp(g).reshape(-1, 8, 2)
    bx, by, bz = v[:, 4], v[:, 5], v[:, 6]
    b = np.sqrt(bx * bx + by * by + bz * bz)
    kpa = cfg["kpara0"] * (p / cfg["p0"]) ** (3.0 - cfg["gamma_turb"])
    kpe = kpa * cfg["kret"]
    kpp = kpa - kpe
    dbx, dby, dbz, db = d[:, 4], d[:, 5], d[:, 6], d[:, 7]
    xx = 2 * kpp * bx * (dbx[:, 0] * b - bx * db[:, 0]) / b**3
    yy = 2 * kpp * by * (dby[:, 1] * b - by * db[:, 1]) / b**3
    xy = [kpp * ((dbx[:, i] * by + bx * dby[:, i]) / b**2 - 2 * bx * by * db[:, i] / b**3) for i in (0, 1)]
    vdp = (1.0 / (3 * cfg["charge"])) / np.sqrt((cfg["drift1"] / p) ** 2 + (cfg["drift2"] / p**2) ** 2)
    ux = v[:, 0] + vdp * (dbz[:, 1] / b**2 - 2 * bz * db[:, 1] / b**3) + xx + xy[1]
    uy = v[:, 1] + vdp * (-dbz[:, 0] / b**2 + 2 * bz * db[:, 0] / b**3) + xy[0] + yy
    dpdt = -p * (d[:, 0, 0] + d[:, 1, 1]) / 3.0
    m = np.minimum((0.5 / n) ** 2 / (2 * kpa), np.minimum(2 * kpe / ux**2, 2 * kpe / uy**2))
    m = np.clip(np.minimum(m, 0.1 * p / np.abs(dpdt)), cfg["dt_min_rel"] * dtf, cfg["dt_max_rel"] * dtf)
    h = np.where(fixed != 0, dt, m)
    sq = np.sqrt(h)
    dx = ux * h + (r[:, 0] * np.sqrt(2 * kpe) + r[:, 2] * np.sqrt(2 * kpp) * bx / b) * sq
    dy = uy * h + (r[:, 1] * np.sqrt(2 * kpe) + r[:, 2] * np.sqrt(2 * kpp) * by / b) * sq
    dp = np.maximum(dpdt * h, 0.25 * cfg["p0"] - p)
    return dict(state=np.stack([x + dx, y + dy, z, p + dp, t + h, h], 1),
                deltas=np.stack([dx, dy, 0 * dx, dp], 1))


def _exact_diagnostics(case, seed):
    P = _host_population(case["nptl"], 2, seed, splits=3)
    w, lp = P["weight"], np.log10(P["p"])
    m = case["map"]
    ip = np.floor((lp + 2.0) / (6.0 / 256)).astype(int)
    ok = (P["p"] > 1e-2) & (P["p"] <= 1e4) & (ip < 256)
    fg = np.bincount(ip[ok], w[ok], 256)
    jp = np.floor((lp + 2.0) / (6.0 / 16)).astype(int)
    ix, iy = (np.floor(P[a] / (1.0 / m)).astype(int) for a in "xy")
    ok = (jp >= 0) & (jp < 15) & (ix < m) & (iy < m)
    fl = np.bincount(((iy * m + ix) * 16 + jp)[ok], w[ok], m * m * 16)
    quick = dict(nptl_current=float(case["nptl"]), nptl_split=0.0, ntot=float(w.sum()), leak=0.0,
                 leak_negp=0.0, pdt_min=float(P["dt"].min()), pdt_max=float(P["dt"].max()),
                 pdt_avg=float(P["dt"].mean()), pmax=float(P["p"].max()))
    return dict(quick=quick, fglobal=fg, flocal=fl.reshape(1, m, m, 16, 1))


def _layers(case, p):
    dims = [6] + [case["nhidden"]] * case["nlayers"] + [case["nout"]]
    at, out = 0, []
    for k, n in zip(dims[:-1], dims[1:]):
        out += [p[at:at + k * n].view(k, n), p[at + k * n:at + k * n + n]]
        at += k * n + n
    return out


def _net64(layers, x):
    for i in range(0, len(layers), 2):
        x = x @ layers[i] + layers[i + 1]
        if i + 2 < len(layers):
            x = torch.nn.functional.silu(x)
    return x


def _philox_a(c0, step, c2, k0, k1):
    """First word of Philox4x32-10 at the counters (c0, step, c2, 0)."""
    m = 0xFFFFFFFF
    c = [c0, torch.full_like(c0, step), torch.full_like(c0, c2), torch.zeros_like(c0)]

    def mul(a, b):  # 32 x 32 -> (high, low), in 16-bit halves of b
        lo, hi = (b & 0xFFFF) * a, (b >> 16) * a
        t = (lo >> 16) + hi
        return (t >> 16) & m, ((t & 0xFFFF) << 16) | (lo & 0xFFFF)

    for i in range(10):
        (h0, l0), (h1, l1) = mul(0xD2511F53, c[0]), mul(0xCD9E8D57, c[2])
        c = [h1 ^ c[1] ^ k0, l1, h0 ^ c[3] ^ k1, l0]
        k0, k1 = (k0 + 0x9E3779B9) & m, (k1 + 0xBB67AE85) & m
    return c[0]


def _exact_fit(case, seed):
    """AdamW in 64 bits on the same mini-batches.  The parameters are left
    out: early updates are lr * sign(gradient), so a gradient near zero that
    BF16 products round to the other sign moves its weight by a whole step."""
    with Mlp(6, case["nhidden"], case["nlayers"], case["nout"], batch_max=1, seed=seed & 0xFFFF) as net:
        p0 = net.get_params()
    x, y = (torch.from_numpy(a).cuda().double() for a in _fit_data(case, seed))
    p = torch.from_numpy(p0).cuda().double().requires_grad_()
    opt = torch.optim.AdamW([p], betas=(0.9, 0.999), eps=1e-8, weight_decay=1e-4)
    rows = torch.arange(case["batch"], device="cuda")
    losses, ns = [], case["nsteps"]
    for s in range(ns):
        for q in opt.param_groups:
            q["lr"] = 2e-5 + 0.5 * (2e-3 - 2e-5) * (1.0 + math.cos(math.pi * s / max(1, ns - 1)))
        idx = (_philox_a(rows, s, 0x6D6C70, seed & 0xFFFFFFFF, seed >> 32) * len(x)) >> 32
        loss = torch.nn.functional.mse_loss(_net64(_layers(case, p), x[idx]), y[idx])
        opt.zero_grad()
        loss.backward()
        opt.step()
        losses.append(loss.detach())
    return dict(losses=torch.stack(losses), params=None)


def _exact_predict(case, seed):
    x = torch.from_numpy(_query_rows(case["rows"], seed)).cuda().double()
    f = []
    for i in range(2):
        p = torch.from_numpy(_weights(case, seed + i)).cuda().double()
        f.append((10.0 ** _net64(_layers(case, p), x) - FLOOR).clamp(min=0.0))
    mean = (f[0] + f[1]) / 2
    spread = ((f[0] - mean).abs().sum(1) + (f[1] - mean).abs().sum(1)) / 2
    return dict(spec=mean, spread=spread)


def exact(case, seed):
    kind = case["kind"]
    if kind == "step":
        return _exact_step(case, seed)
    if kind == "diagnostics":
        return _exact_diagnostics(case, seed)
    if kind == "fit":
        return _exact_fit(case, seed)
    if kind in ("predict", "predict_dev"):
        return _exact_predict(case, seed)
    # whole intervals: hundreds of steps whose lengths, wraps and redo steps
    # follow each particle's own path
    return None
