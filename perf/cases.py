"""Workloads of the seismic propagators, from the smallest call to survey size.

Each case is one call (or one short sequence of calls) of the public Python
API, with the sizes of this repository's configurations, tests and benchmark
or generic ones:

  listed()            the workloads, each with a name
  draw(rng)           one more workload of the same ranges
  prepare(case, seed) what a program holds before the call: models, data, handles
  run(state)          one pass through the public entry points, and its results
  work(case)          bytes and floating-point operations of one pass
  exact(case, seed)   the same results from plain torch in 64 bits

Grids are earth models (a velocity gradient, smooth dipping interfaces and an
anomaly, Gardner density, Vs = Vp / 1.732); recorded data are hyperbolic
Ricker events with noise, as a field record has them.
"""
import math

import numpy as np
import torch

from elastic_amd import learned, lib

# weights of the 10th-order staggered first derivative and of the 10th-order
# second derivative, as single-precision constants (they define the scheme)
_F = np.float32
C = [float(_F(a) / _F(b)) for a, b in ((35, 294912), (-405, 229376), (567, 40960), (-735, 8192), (19845, 16384))]
W = [float(_F(a) / _F(b)) for a, b in ((-5269, 1800), (5, 3), (-5, 21), (5, 126), (-5, 1008), (1, 3150))]
Z0 = 6.0e6  # impedance that scales stresses against velocities


def listed():
    return [
        # the smallest complete migration (the smoke test's grid): a user trying
        # the library, and the latency of one call
        dict(name="migrate_80x110", kind="migrate", nz=80, nx=110, nt=160, dx=10.0, dt=1e-3, fp=15.0, abc=10,
             adj_abc=0, snap_every=1, snap_prec="fp32", comp=0),
        # the reference's rtm.x on its layer configuration (300 x 300, 4 m, 2 s),
        # through the mirror of its operator module: the drop-in user's migration
        dict(name="operator_rtm_300x300", kind="operator", adj=1, nz=300, nx=300, nt=3535, dx=4.0, dt=5.65685e-4,
             fp=20.0, abc=40),
        # the same operator's other direction, Born modelling, on an odd grid
        dict(name="operator_born_231x347", kind="operator", adj=0, nz=231, nx=347, nt=1001, dx=10.0, dt=1e-3, fp=15.0,
             abc=40),
        # modelling of one shot's record on the 300 x 600 configuration (padded)
        dict(name="forward_390x690", kind="forward", nz=390, nx=690, nt=2000, dx=10.0, dt=1e-3, fp=15.0, abc=40),
        # the drop-in adjoint on host histories, as Fortran callers bind it
        dict(name="op3_390x690", kind="op3", nz=390, nx=690, nt=100),
        # a small survey: many small uneven shots per launch, per-shot images
        dict(name="batch_200x400_12", kind="batch", shots=12, nz=200, nx=400, wmin=300, wmax=400, nt=600, dx=10.0,
             dt=8e-4, fp=15.0, abc=40, adj_abc=1, snap_every=1, snap_prec="fp32", comp=0, graph=1, images=1, learned=0),
        # groups of the 64-shot 800 x 2400 survey, at its apertures: single
        # precision history, and bfloat16 snapshots with compensated images
        dict(name="batch_800x2400_7_fp32", kind="batch", shots=7, nz=800, nx=2400, wmin=600, wmax=1200, nt=480,
             dx=10.0, dt=8e-4, fp=15.0, abc=40, adj_abc=1, snap_every=1, snap_prec="fp32", comp=0, graph=1, images=0,
             learned=0),
        dict(name="batch_800x2400_14_bf16", kind="batch", shots=14, nz=800, nx=2400, wmin=600, wmax=1200, nt=480,
             dx=10.0, dt=8e-4, fp=15.0, abc=40, adj_abc=1, snap_every=4, snap_prec="bf16", comp=1, graph=1, images=0,
             learned=0),
        # the learned absorbing layer in both directions, on its 400 x 800 grids
        dict(name="batch_learned_400x800_6", kind="batch", shots=6, nz=400, nx=800, wmin=800, wmax=800, nt=400,
             dx=10.0, dt=1e-3, fp=15.0, abc=8, adj_abc=1, snap_every=4, snap_prec="bf16", comp=1, graph=0, images=0,
             learned=1),
        # 3D acoustic subdomains: an odd one with single precision snapshots,
        # and the 512^3 subdomain (with its halo) with bfloat16 ones
        dict(name="acoustic_203x181x247", kind="acoustic", n1=203, n2=181, n3=247, nt=200, abc=20, snap_every=5,
             snap_prec="fp32"),
        dict(name="acoustic_522", kind="acoustic", n1=522, n2=522, n3=522, nt=300, abc=40, snap_every=5,
             snap_prec="bf16"),
        # the 9-field 3D elastic adjoint step at the reference's test shape,
        # device resident, a block of steps from given fields
        dict(name="elastic3d_200", kind="elastic3d", ny=200, nz=200, nx=200, steps=24),
    ]


def _log(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    kind = rng.choice(["migrate", "operator", "forward", "op3", "batch", "batch", "acoustic", "acoustic", "elastic3d"])
    dt, dx = 1e-3, 10.0
    if kind in ("migrate", "operator", "forward"):
        c = dict(kind=kind, nz=_log(rng, 60, 500), nx=_log(rng, 60, 900))
        c["nt"] = max(60, min(_log(rng, 100, 3600), int(4.5e8 / (c["nz"] * c["nx"]))))
        c.update(dx=dx, dt=dt, fp=15.0, abc=rng.choice([10, 20, 40]) if min(c["nz"], c["nx"]) > 100 else 10)
        if kind == "operator":
            c["adj"] = rng.choice([0, 1])
        if kind == "migrate":
            j, prec, comp = rng.choice([(1, "fp32", 0), (1, "fp32", 0), (3, "fp32", 1), (4, "bf16", 1), (4, "fp16", 1)])
            c.update(adj_abc=rng.choice([0, 1, 1, 2]), snap_every=j, snap_prec=prec, comp=comp)
        return c
    if kind == "op3":
        c = dict(kind=kind, nz=_log(rng, 60, 500), nx=_log(rng, 60, 800))
        return dict(c, nt=max(3, min(_log(rng, 8, 200), int(2.5e7 / (c["nz"] * c["nx"])))))
    if kind == "batch":
        lrn = rng.choice([0, 0, 0, 1])
        nz = _log(rng, 90, 800)
        wmin = _log(rng, 100, 800)
        wmax = int(wmin * rng.uniform(1.0, 1.6))
        shots = rng.randint(1, 14)
        cells = shots * (nz + 90) * (0.5 * (wmin + wmax) + 90)
        nt = max(40, min(_log(rng, 120, 800), int(5e9 / cells), int((2e9 if lrn else 5e9) / cells)))
        j, prec, comp = rng.choice([(1, "fp32", 0), (1, "fp32", 0), (4, "bf16", 1), (4, "bf16", 1), (4, "fp16", 1)])
        return dict(kind=kind, shots=shots, nz=nz, nx=int(wmax * rng.uniform(1.0, 3.0)), wmin=wmin, wmax=wmax, nt=nt,
                    dx=dx, dt=8e-4, fp=15.0, abc=8 if lrn else 40, adj_abc=1, snap_every=j, snap_prec=prec, comp=comp,
                    graph=rng.choice([0, 1]), images=0, learned=lrn)
    if kind == "acoustic":
        n = [_log(rng, 41, 460) for _ in range(3)]
        nt = max(20, min(_log(rng, 40, 400), int(2e10 / (n[0] * n[1] * n[2]))))
        return dict(kind=kind, n1=n[0], n2=n[1], n3=n[2], nt=nt, abc=10 if min(n) < 90 else 20, snap_every=5,
                    snap_prec=rng.choice(["fp32", "bf16"]))
    n = [_log(rng, 20, 260) for _ in range(3)]
    return dict(kind=kind, ny=n[0], nz=n[1], nx=n[2],
                steps=max(3, min(_log(rng, 6, 60), int(1.9e8 / (n[0] * n[1] * n[2])))))


# --------------------------------------------------------------------------- earth models and data
def _rng(seed, *more):
    return np.random.default_rng([int(seed) & 0x7FFFFFFF, *more])


def _vp(nz, nx, rng, dx, dt, sharp=8.0):
    """Velocity gradient, five smooth dipping interfaces and one anomaly (m/s),
    slow enough for the time step (vp dt / dx below 0.5)."""
    z = np.arange(nz, dtype=np.float32)[:, None]
    x = np.arange(nx, dtype=np.float32)[None, :]
    vp = 1800.0 + 2400.0 * z / max(nz - 1, 1) + 0.0 * x
    for d, s, tilt in zip(rng.uniform(0.1 * nz, 0.95 * nz, 5), rng.choice([-1.0, 1.0], 5), rng.uniform(-0.05, 0.05, 5)):
        vp = vp + s * 100.0 * np.tanh((z - d - tilt * (x - nx / 2)) / sharp)
    cz, cx = rng.uniform(0.3, 0.7, 2) * (nz, nx)
    vp = vp + 250.0 * np.exp(-((z - cz) / 25.0) ** 2) * np.exp(-((x - cx) / 25.0) ** 2)
    return vp * min(1.0, 0.5 * dx / dt / 4950.0)


def _lame(vp):
    rho = 310.0 * vp ** 0.25
    mu = rho * (vp / 1.732) ** 2
    return [np.asfortranarray(a, np.float32) for a in (rho, rho * vp ** 2 - 2.0 * mu, mu)]


def _coefs(rho, lam, mu, dx, dt, dtype=np.float64):
    """Staggered, dt/dx-scaled coefficients m1_x, m1_z, m2, m3, m2m3."""
    r, l, m = (np.asarray(a, np.float64) for a in (rho, lam, mu))
    m1x, m1z = 1.0 / r, 1.0 / r
    m1x[:-1] = 2.0 / (r[1:] + r[:-1])
    m1z[:, :-1] = 2.0 / (r[:, 1:] + r[:, :-1])
    out = []
    for a in (l, m):
        b, q = a.copy(), 1.0 / a
        b[1:-1, 1:-1] = 4.0 / (q[1:-1, 1:-1] + q[2:, 1:-1] + q[1:-1, 2:] + q[2:, 2:])
        b[0], b[-1] = b[1], b[-2]
        b[:, 0], b[:, -1] = b[:, 1], b[:, -2]
        out.append(b)
    s = float(_F(dt)) / float(_F(dx))
    return [np.asfortranarray(s * a, dtype) for a in (m1x, m1z, out[0], out[1], out[0] + 2.0 * out[1])]


def _ricker(nt, dt, fp):
    t = (np.arange(1, nt + 1) - 125.0) * dt
    a = (math.pi * fp * t) ** 2
    return (1e8 * (1.0 - 2.0 * a) * np.exp(-a)).astype(np.float32)


def _record(nrx, nt, xs, dx, dt, fp, rng):
    """(5, nrx, nt) field record: three hyperbolic events and noise, the
    velocities in m/s and the stresses scaled by the impedance."""
    x = (np.arange(nrx, dtype=np.float32)[:, None] - xs) * dx
    t = np.arange(nt, dtype=np.float32)[None, :] * dt
    d = np.zeros((nrx, nt), np.float32)
    for t0, v, a in zip(rng.uniform(0.05, 0.8, 3) * nt * dt, rng.uniform(1800, 4000, 3), rng.uniform(-1, 1, 3)):
        u = (math.pi * fp) ** 2 * (t - np.sqrt(t0 * t0 + (x / v) ** 2)) ** 2
        d += a * (1.0 - 2.0 * u) * np.exp(-np.minimum(u, 80.0))
    d += 0.02 * rng.standard_normal((nrx, nt), dtype=np.float32)
    return np.stack([s * d for s in (0.6, 1.0, Z0, 0.8 * Z0, 0.5 * Z0)]).astype(np.float32)


def _perturbation(nz, nx, rng):
    """drho, dlambda, dmu: smooth random reflectivity inside the sponge."""
    z = np.arange(nz)[:, None]
    taper = np.clip((np.minimum(z, nz - 1 - z) - 20) / 20.0, 0, 1)
    band = sum(a * np.sin(k * z / nz * 2 * math.pi + p) for a, k, p in
               zip(rng.uniform(-1, 1, 4), rng.uniform(4, 16, 4), rng.uniform(0, 6, 4)))
    lat = 1.0 + 0.3 * np.sin(rng.uniform(1, 5) * np.arange(nx)[None, :] / nx * 2 * math.pi)
    return [np.asfortranarray(s * taper * band * lat, np.float32) for s in (50.0, 4e8, 3e8)]


def _single(case, seed):
    """Model, source and record of a one-shot workload."""
    rng = _rng(seed, 1)
    nz, nx, nt, dx, dt = (case[k] for k in ("nz", "nx", "nt", "dx", "dt"))
    pad = case["abc"] + 5
    d = dict(case, lame=_lame(_vp(nz, nx, rng, dx, dt)), wav=_ricker(nt, dt, case["fp"]),
             zs=min(pad + 2, nz - 1), xs=int(rng.integers(nx // 4, 3 * nx // 4)), zr=min(pad + 2, nz - 1))
    # the operator records every column of its grid, the calls with a padded
    # grid the physical ones
    d["rx0"], d["nrx"] = (0, nx) if case["kind"] == "operator" else (min(pad, nx // 3), nx - 2 * min(pad, nx // 3))
    if case.get("adj") == 0:
        d["dm"] = _perturbation(nz, nx, rng)
    elif case["kind"] != "forward":
        d["rec"] = _record(d["nrx"], nt, d["xs"] - d["rx0"], dx, dt, case["fp"], rng)
    return d


def _survey(case, seed):
    """Shot windows of a survey line: coefficients, geometry and records."""
    rng = _rng(seed, 2)
    pad = case["abc"] + 5
    nz, nx, nt, dx, dt = (case[k] for k in ("nz", "nx", "nt", "dx", "dt"))
    vp = _vp(nz, nx, rng, dx, dt)
    shots, coefs, recs = [], [], []
    apertures = _rng(7).integers(case["wmin"], case["wmax"] + 1, case["shots"])  # the survey's, whatever its model
    for k in range(case["shots"]):
        w = int(min(nx, apertures[k]))
        xs = int((k + 0.5) * nx / case["shots"])
        x0 = int(np.clip(xs - w // 2, 0, nx - w))
        coefs.append(_coefs(*_lame(np.pad(vp[:, x0:x0 + w], pad, mode="edge")), dx, dt, np.float32))
        shots.append(dict(nz=nz + 2 * pad, nx=w + 2 * pad, xs=pad + xs - x0, zs=pad + 2, zr=pad + 2, rx0=pad, nrx=w,
                          img_z0=pad, img_x0=pad, img_nz=nz, img_nx=w, stack_z0=0, stack_x0=x0))
        recs.append(_record(w, nt, xs - x0, dx, dt, case["fp"], rng))
    nets = [_net_params(rng) for _ in range(2)] if case["learned"] else None
    return dict(case, specs=shots, coefs=coefs, recs=recs, wav=_ricker(nt, dt, case["fp"]), nets=nets)


def _net_params(rng):
    """Weights of the size a trained layer has: corrections of about a
    thousandth of the local wavefield."""
    n = rng.standard_normal
    p = [n(245 * 32) / math.sqrt(245), 0.1 * n(32), n(32 * 32) / math.sqrt(32), 0.1 * n(32), 1e-3 * n(32 * 5), 1e-4 * n(5)]
    return np.concatenate(p).astype(np.float32)


def _volume(case, seed):
    """c = (v dt / dx)^2 of a 3D subdomain, the source and its amplitudes, and
    the receiver plane's record (level, y, x): two reflections of the source."""
    rng = _rng(seed, 3)
    n1, n2, n3, nt = (case[k] for k in ("n1", "n2", "n3", "nt"))
    z = np.arange(n1, dtype=np.float32)
    prof = (0.28 + 0.09 * z / n1) ** 2
    lat = [1.0 + 0.06 * np.sin(rng.uniform(1, 3) * 2 * math.pi * np.arange(n, dtype=np.float32) / n + rng.uniform(0, 6))
           for n in (n2, n3)]
    c = (lat[1].astype(np.float32)[:, None, None] * lat[0].astype(np.float32)[None, :, None]) * prof.astype(np.float32)
    t = np.arange(1, nt + 1, dtype=np.float64)
    a = (math.pi * (t - 25.0) / 18.0) ** 2
    pad = case["abc"] + 5
    src = (min(pad + 3, n1 // 2), n2 // 2 + int(rng.integers(-5, 6)), n3 // 2 + int(rng.integers(-5, 6)))
    lev, y, x = (torch.arange(n, dtype=torch.float32, device="cuda") for n in (nt, n3, n2))
    r2 = ((y - src[2])[:, None] ** 2 + (x - src[1])[None, :] ** 2) / 0.3 ** 2
    rec = torch.zeros((nt, n3, n2), dtype=torch.float32, device="cuda")
    for t0, g in zip(rng.uniform(0.1, 0.6, 2) * nt, rng.uniform(-1, 1, 2)):
        u = (math.pi / 18.0 * (lev[:, None, None] - torch.sqrt(t0 * t0 + r2)[None])) ** 2
        rec += 0.01 * g * (1.0 - 2.0 * u) * torch.exp(-u)
    inside = torch.zeros((n3, n2), dtype=torch.float32, device="cuda")
    inside[5:-5, 5:-5] = 1.0
    return dict(case, c=c.transpose(2, 1, 0), src=src, zr=min(pad + 1, n1 // 2), rec=(rec * inside).cpu().numpy(),
                amp=((1 - 2 * a) * np.exp(-a)).astype(np.float32))


class _Block:
    """A float32 torch tensor in the role of a device block of k fields."""

    def __init__(self, t):
        self.t, self.ptr, self.shape = t, t.data_ptr(), tuple(t.shape)

    def slab(self, k):
        return self.t[k].data_ptr()


def _elastic(case, seed):
    """Fields of three levels and coefficients (dt/dx-scaled), zero padding."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    ny, nz, nx = (case[k] for k in ("ny", "nz", "nx"))
    shp = (ny + 10, nx + 10, nz + 10)

    def block(k, lo, hi):
        t = torch.zeros((k,) + shp, dtype=torch.float32, device="cuda")
        t[:, 5:-5, 5:-5, 5:-5] = torch.rand((k, ny, nx, nz), generator=g, device="cuda") * (hi - lo) + lo
        return t

    fields = [block(9, -1.0, 1.0) for _ in range(3)]
    coef = block(6, 0.25, 0.35)
    coef[3:5] *= 0.4  # lambda, mu against lambda + 2 mu
    return fields, coef


# --------------------------------------------------------------------------- prepare and run
def prepare(case, seed):
    kind = case["kind"]
    if kind == "operator":
        d = _single(case, seed)
        d["op"] = lib.RtmOperator(d["nz"], d["dx"], d["nx"], d["dx"], d["dt"], d["xs"] + 1, d["zs"] + 1, d["zr"] + 1,
                                  d["fp"], d["nt"], d["abc"], 0, *d["lame"])
        n, r = (d["nz"], d["nx"]), (d["nt"], d["nx"])
        if case["adj"]:
            d["data"] = [np.asfortranarray(a.T) for a in d.pop("rec")]
            d["img"] = [np.zeros(n, np.float32, order="F") for _ in range(3)]
        else:
            d["data"] = [np.zeros(r, np.float32, order="F") for _ in range(5)]
            d["img"] = d["dm"]
        return d
    if kind in ("migrate", "forward"):
        d = _single(case, seed)
        d["coefs"] = _coefs(*d["lame"], d["dx"], d["dt"], np.float32)
        d["shot"] = lib.shot(d["nz"], d["nx"], d["nt"], d["dx"], d["dt"], d["xs"], d["zs"], d["zr"], d["rx0"], d["nrx"],
                             d["abc"], adj_abc=d.get("adj_abc", 0), snap_every=d.get("snap_every", 1),
                             snap_prec=lib.SNAP_PREC[d.get("snap_prec", "fp32")], comp_image=d.get("comp", 0))
        return d
    if kind == "op3":
        return _histories(case, seed)
    if kind == "batch":
        d = _survey(case, seed)
        b = lib.Batch(d["nt"], d["dx"], d["dt"], d["specs"], d["coefs"], d["wav"], abc=d["abc"], adj_abc=d["adj_abc"],
                      snap_every=d["snap_every"], snap_prec=d["snap_prec"], comp_image=d["comp"], use_graph=d["graph"],
                      stack_shape=(d["nz"], d["nx"]))
        for i, r in enumerate(d["recs"]):
            b.set_data(i, r)
        if d["nets"]:
            for p, put in zip(d["nets"], (b.set_learned, b.set_learned_adjoint)):
                net = learned.Net()
                net.params = p
                put(net)
        return dict(case, batch=b)
    if kind == "acoustic":
        d = _volume(case, seed)
        a = lib.Acoustic3D(d["c"], d["amp"], d["src"], d["zr"], abc=d["abc"], snap_every=d["snap_every"],
                           snap_prec=d["snap_prec"])
        a.set_data(d["rec"])
        return dict(case, handle=a)
    fields, coef = _elastic(case, seed)
    return dict(case, fields=fields, coef=_Block(coef), work=[_Block(torch.empty_like(t)) for t in fields])


def run(s):
    kind = s["kind"]
    if kind == "operator":
        s["op"].op(s["adj"], *s["img"], *s["data"])
        return dict(zip(("drho", "dlambda", "dmu"), s["img"])) if s["adj"] else dict(record=s["data"])
    if kind == "migrate":
        return lib.migrate(s["shot"], s["coefs"], s["wav"], s["rec"])
    if kind == "forward":
        rec, last = lib.forward(s["shot"], s["coefs"], s["wav"], want_last=True)
        return dict(record=rec, last=last)
    if kind == "op3":
        return lib.rtm_op3(s["hist"], s["coefs"])
    if kind == "batch":
        b = s["batch"]
        b.migrate()
        out = dict(stack=b.stack((s["nz"], s["nx"])))
        if s["images"]:
            out["images"] = [b.image(i) for i in range(s["shots"])]
        return out
    if kind == "acoustic":
        s["handle"].migrate()
        return s["handle"].image()
    for w, f in zip(s["work"], s["fields"]):
        w.t.copy_(f)
    torch.cuda.current_stream().synchronize()  # the library runs on a stream of its own
    roles = lib.el3_steps_dev(s["work"], s["coef"], s["steps"])
    return dict(zip(("now", "before", "out"), (r.t for r in roles)))


def _histories(case, seed):
    """Adjoint histories before the scan: the injected receiver rows of every
    level and a smooth field, with the coefficients of a model."""
    rng = _rng(seed, 4)
    nz, nx, nt = (case[k] for k in ("nz", "nx", "nt"))
    g = np.sin(np.arange(nz)[:, None] * 0.11 + np.arange(nx)[None, :] * 0.07).astype(np.float32)
    hist = []
    for f, s in enumerate((1.0, 1.0, 1e-3, 1e-3, 1e-3)):
        h = np.zeros((nt, nx, nz), np.float32)
        h += (s * 0.1 * rng.uniform(0.5, 1.0)) * g.T * np.cos(0.3 * np.arange(nt) + f).astype(np.float32)[:, None, None]
        h[:, :, min(7, nz - 1)] += s * rng.standard_normal((nt, nx), dtype=np.float32)
        hist.append(h.transpose(2, 1, 0))
    return dict(case, hist=hist, coefs=_coefs(*_lame(_vp(nz, nx, rng, 10.0, 1e-3)), 10.0, 1e-3, np.float32))


def _shot_sizes(case):
    """(rows, columns) of every shot's grid; window widths at their mean."""
    if case["kind"] != "batch":
        return [(case["nz"], case["nx"])]
    pad = 2 * (case["abc"] + 5)
    w = min(case["nx"], 0.5 * (case["wmin"] + case["wmax"]))
    return [(case["nz"] + pad, w + pad)] * case["shots"]


def work(case):
    """A level of a step reads the two levels before it and the coefficients
    and writes its own; histories and images go through memory once a level
    that is imaged. Differences: 15 operations each."""
    kind = case["kind"]
    if kind == "acoustic":
        n = float(case["n1"]) * case["n2"] * case["n3"]
        k, b = case["nt"] // case["snap_every"], 2 if case["snap_prec"] == "bf16" else 4
        return dict(bytes=n * (2 * case["nt"] * 16 + k * (2 * b + 8) + 4), flops=n * 2 * case["nt"] * 45.0)
    if kind == "elastic3d":
        n = float(case["ny"]) * case["nz"] * case["nx"]
        return dict(bytes=n * 168 * case["steps"], flops=n * case["steps"] * 320.0)
    n = float(sum(a * b for a, b in _shot_sizes(case)))
    nt = case["nt"]
    if kind == "op3":
        return dict(bytes=n * nt * 40 + n * 20, flops=n * nt * 140.0)
    if kind == "forward":
        return dict(bytes=n * nt * 80, flops=n * nt * 140.0)
    if kind == "operator" and not case["adj"]:
        return dict(bytes=n * nt * (80 + 8 + 80 + 8 + 12), flops=n * nt * 350.0)
    j = case.get("snap_every", 1)
    hist = 8.0 if j == 1 and case.get("snap_prec", "fp32") == "fp32" else 4.0 * (4 if case["snap_prec"] == "fp32" else 2) / j
    img = (48.0 if case.get("comp") else 24.0) / j
    flops = n * nt * (140 + 140 + 75.0 / j)
    if case.get("learned"):
        cells = sum(16.0 * (a + b) for a, b in _shot_sizes(case))
        flops += 2 * nt * cells * 2 * 9024
    return dict(bytes=n * nt * (160 + 2 * hist + img), flops=flops)


# --------------------------------------------------------------------------- the same in 64 bits
_D = dict(dtype=torch.float64, device="cuda")


def _t(a):
    return torch.tensor(np.ascontiguousarray(a, np.float64), **_D)


def _diff(n, plus):
    """Matrix of the staggered difference S+ (plus) or S- of n samples."""
    m = np.zeros((n, n))
    for k, c in enumerate(C, 1):
        for i in range(n):
            for at, s in ((i + (6 if plus else 5) - k, c), (i - (5 if plus else 6) + k, -c)):
                if 0 <= at < n:
                    m[i, at] += s
    return _t(m)


def _taper(n, abc):
    k = np.ones(n)
    if abc > 0:
        f = np.exp(-0.09 * np.minimum(np.arange(1, abc + 6) / abc, 1.0) ** 2)
        k[:abc + 5] *= f[::-1]
        k[n - abc - 5:] *= f
    return k


class _Grid:
    """One shot's grid in 64 bits: coefficients restricted to each operator's
    rows and columns, difference matrices, sponge."""

    def __init__(self, nz, nx, coefs, abc, dx, dt):
        self.nz, self.nx, self.dx, self.dt = nz, nx, float(_F(dx)), float(_F(dt))
        self.c = []
        for a, x0, z0 in zip(coefs, (5, 4, 4, 5, 4), (4, 5, 4, 5, 4)):
            t = torch.zeros((nz, nx), **_D)
            t[z0:nz - 5, x0:nx - 5] = _t(a)[z0:nz - 5, x0:nx - 5]
            self.c.append(t)
        self.zp, self.zm = _diff(nz, True), _diff(nz, False)
        self.xp, self.xm = _diff(nx, True).T.contiguous(), _diff(nx, False).T.contiguous()
        self.k = _t(np.outer(_taper(nz, abc), _taper(nx, abc))) if abc > 0 else None

    def apply(self, y):
        """The forward operators on level y: the increments of the five fields."""
        m1x, m1z, m2, m3, m23 = self.c
        vx, vz, xx, zz, xz = y
        dx, dz = vx @ self.xp, self.zp @ vz
        return torch.stack([m1x * (xx @ self.xm + self.zp @ xz), m1z * (xz @ self.xp + self.zm @ zz),
                            m23 * dx + m2 * dz, m2 * dx + m23 * dz, m3 * (self.zm @ vx + vz @ self.xm)])

    def apply_t(self, y):
        """Their transposes."""
        m1x, m1z, m2, m3, m23 = self.c
        vx, vz, xx, zz, xz = y
        p2, p3, p4 = m3 * xz, m1x * vx, m1z * vz
        return -torch.stack([(m23 * xx + m2 * zz) @ self.xm + self.zp @ p2, self.zm @ (m2 * xx + m23 * zz) + p2 @ self.xp,
                             p3 @ self.xp, self.zp @ p4, self.zm @ p3 + p4 @ self.xm])

    def strains(self, v):
        """S4, S5, S6 of the source velocities v (2, nz, nx)."""
        s = torch.zeros((3, self.nz, self.nx), **_D)
        a, b = (slice(4, self.nz - 5), slice(4, self.nx - 5)), (slice(5, self.nz - 5), slice(5, self.nx - 5))
        s[0][a] = ((v[0] @ self.xp) / self.dx)[a]
        s[1][a] = ((self.zp @ v[1]) / self.dx)[a]
        s[2][b] = ((self.zm @ v[0] + v[1] @ self.xm) / self.dx)[b]
        return s


def _forward64(g, nt, zs, xs, wav, zr=None, rx0=0, nrx=0, source=None, layer=None, keep=None):
    """Levels 1..nt of the source run (or with source(L) of a run of those
    sources): the record (5, nrx, nt), the last two levels, and of the levels
    keep(L) the velocities and their change to the next level."""
    old, now = torch.zeros((5, g.nz, g.nx), **_D), torch.zeros((5, g.nz, g.nx), **_D)
    rec = torch.zeros((5, max(nrx, 0), nt), **_D)
    v, dv = {}, {}
    for L in range(1 if source else 2, nt + 1):
        new = old + g.apply(now)
        if source:
            new += source(L)
        else:
            new[2:4, zs, xs] += g.dt * float(wav[L - 2])
        if g.k is not None and (source or L >= 3):
            new *= g.k
        if keep and keep(L - 1):
            v[L - 1] = now[:2]
            dv[L - 1] = new[:2] - now[:2]
        if layer and L >= 3:
            layer.correct(new, now, old)
        if nrx:
            rec[:, :, L - 1] = new[:, zr, rx0:rx0 + nrx]
        old, now = now, new
    if keep and keep(nt):
        v[nt] = now[:2]
    return rec, (old, now), v, dv


def _migrate64(g, nt, zs, xs, wav, zr, rx0, rec, adj_abc, j, layer=None, layer_adj=None):
    """Images drho, dlambda, dmu (3, nz, nx) of one shot."""
    _, _, v, dv = _forward64(g, nt, zs, xs, wav, layer=layer, keep=lambda L: L >= 1 and L % j == 0)
    data = _t(rec)
    nrx = data.shape[1]
    late, next_ = torch.zeros((5, g.nz, g.nx), **_D), torch.zeros((5, g.nz, g.nx), **_D)
    img = torch.zeros((3, g.nz, g.nx), **_D)
    k = g.k if adj_abc else None
    for L in range(nt, 0, -1):
        # adj_abc 2 keeps damped levels: T(L) = K R(L), R(L) = data + K T(L+2) + Op^T T(L+1)
        new = (late * k if adj_abc == 2 and k is not None else late) + g.apply_t(next_)
        new[:, zr, rx0:rx0 + nrx] += data[:, :, L - 1]
        if k is not None and (adj_abc == 1 or L >= 2):
            new *= k
        if L % j == 0:
            a = new * k if adj_abc == 2 and k is not None and L >= 3 else new
            s4, s5, s6 = g.strains(v[L])
            s12 = dv[L] / g.dt if L < nt else torch.zeros((2, g.nz, g.nx), **_D)
            img[0] += j * (a[0] * s12[0] + a[1] * s12[1])
            img[1] -= j * (a[2] + a[3]) * (s4 + s5)
            img[2] -= j * (a[4] * s6 + 2 * a[3] * s5 + 2 * a[2] * s4)
        if layer_adj:
            layer_adj.correct(new, next_, late)
        late, next_ = next_, new
    return img


def _born64(g, nt, zs, xs, wav, zr, rx0, nrx, dm):
    _, _, v, dv = _forward64(g, nt, zs, xs, wav, keep=lambda L: L >= 1)
    d = [_t(a) for a in dm]

    def source(L):
        s4, s5, s6 = g.strains(v[L])
        s12 = dv[L] / g.dt if L < nt else torch.zeros((2, g.nz, g.nx), **_D)
        s3 = s4 + s5
        return torch.stack([d[0] * s12[0], d[0] * s12[1], -2 * d[2] * s4 - d[1] * s3, -2 * d[2] * s5 - d[1] * s3, -d[2] * s6])

    return _forward64(g, nt, zs, xs, wav, zr, rx0, nrx, source=source)[0]


class _Layer:
    """The learned layer in 64 bits (weights and features rounded to bfloat16,
    as the layer defines them)."""

    def __init__(self, g, params, adjoint):
        nz, nx, R, B = g.nz, g.nx, 5, 8
        cols, rows = np.arange(R, nx - R), np.arange(R + B, nz - R - B)
        cells = []
        for e in range(4):
            for d in range(B):
                along = cols if e < 2 else rows
                at = np.full(along.size, (R + d) if e in (0, 2) else (nz if e == 1 else nx) - R - 1 - d)
                cells.append(np.stack([at, along] if e < 2 else [along, at]).tolist() + [[e] * along.size, [d] * along.size])
        iz, ix, e, d = (np.concatenate([np.asarray(c[k]) for c in cells]).astype(np.int64) for k in range(4))
        dz, dx = np.select([e == 0, e == 1], [1, -1], 0), np.select([e == 2, e == 3], [1, -1], 0)
        kn, m = np.meshgrid(np.arange(9), np.arange(-2, 3), indexing="xy")  # (5, 9): offset, inward step
        z = iz[:, None, None] + kn * dz[:, None, None] + m * (e >= 2)[:, None, None]
        x = ix[:, None, None] + kn * dx[:, None, None] + m * (e < 2)[:, None, None]
        self.own = torch.tensor(iz * nx + ix, device="cuda")
        self.patch = torch.tensor((z * nx + x).reshape(iz.size, 45), device="cuda")
        self.unit = _t([Z0 if (f < 2) == bool(adjoint) else 1.0 for f in range(5)])
        m1, m3, m23 = (g.c[k].reshape(-1)[self.own] for k in (0, 3, 4))
        st = torch.zeros((iz.size, 15), **_D)
        r = torch.arange(iz.size, device="cuda")
        st[r, torch.tensor(e, device="cuda")] = 1.0
        st[r, 4 + torch.tensor(d, device="cuda")] = 1.0
        st[:, 12], st[:, 13] = (m1 * m23).sqrt(), (m1 * m3).sqrt()
        st[:, 14] = torch.where(m1 > 0, (m23 / m1).sqrt() / Z0, torch.zeros_like(m1))
        self.static = st
        p = torch.tensor(params).to(torch.bfloat16).to(torch.float64).cuda()
        cut = [245 * 32, 32, 32 * 32, 32, 32 * 5, 5]
        w1, self.b1, w2, self.b2, w3, self.b3 = torch.split(p, cut)
        self.w1, self.w2, self.w3 = w1.reshape(245, 32), w2.reshape(32, 32), w3.reshape(32, 5)

    def correct(self, new, near, far):
        """Adds the correction to the band cells of level new, from the levels
        next to it in time, and clears the rim."""
        n = self.own.numel()
        a = (near.reshape(5, -1)[:, self.patch] / self.unit[:, None, None]).permute(1, 0, 2).reshape(n, 225)
        b = (far.reshape(5, -1)[:, self.own] / self.unit[:, None]).T
        raw = torch.cat([a, b], 1)
        s = raw.abs().amax(1)
        live = s > 1e-30
        x = torch.cat([torch.where(live[:, None], raw / s.clamp_min(1e-30)[:, None], torch.zeros_like(raw)), self.static], 1)
        x = x.to(torch.bfloat16).to(torch.float64)
        h = torch.nn.functional.gelu(x @ self.w1 + self.b1)
        y = torch.nn.functional.gelu(h @ self.w2 + self.b2) @ self.w3 + self.b3
        y = torch.where(live[:, None], y * s[:, None] * self.unit, torch.zeros_like(y))
        new.reshape(5, -1)[:, self.own] += y.T
        for r in (slice(0, 5), slice(-5, None)):
            new[:, r] = 0.0
            new[:, :, r] = 0.0


def _acoustic64(d):
    """Image of the subdomain: source pass, then the receiver pass."""
    n1, n2, n3, nt, j = (d[k] for k in ("n1", "n2", "n3", "nt", "snap_every"))
    kt = [_taper(n, d["abc"]) for n in (n3, n2, n1)]
    k = _t(kt[0])[5:-5, None, None] * _t(kt[1])[None, 5:-5, None] * _t(kt[2])[None, None, 5:-5]
    ins = (slice(5, n3 - 5), slice(5, n2 - 5), slice(5, n1 - 5))

    def at(p, axis, o):
        s = list(ins)
        s[axis] = slice(5 + o, p.shape[axis] - 5 + o)
        return p[tuple(s)]

    def step(p, pp, c):
        lap = 3 * W[0] * p[ins]
        for q in range(1, 6):
            for axis in range(3):
                lap = lap.add_(at(p, axis, q) + at(p, axis, -q), alpha=W[q])
        pp[ins] = k * (2 * p[ins] - pp[ins] + c * lap)

    zero = lambda: torch.zeros((n3, n2, n1), **_D)  # noqa: E731
    sz, sx, sy = d["src"]

    c, rec = _t(d["c"].transpose(2, 1, 0))[ins], _t(d["rec"])
    p, pp, keep = zero(), zero(), {}
    for t in range(1, nt + 1):
        step(p, pp, c)
        pp[sy, sx, sz] += float(d["amp"][t - 1])
        p, pp = pp, p
        if t % j == 0:
            keep[t] = p.clone()
    p, pp, img = zero(), zero(), zero()
    for t in range(nt, 0, -1):
        step(p, pp, c)
        pp[5:-5, 5:-5, d["zr"]] += rec[t - 1, 5:-5, 5:-5]
        p, pp = pp, p
        if t % j == 0:
            img += keep.pop(t) * p
    return img.cpu().numpy().transpose(2, 1, 0)


def _elastic64(case, seed):
    """nsteps of the 9-field step: out += in1 + gathers of coefficient * in."""
    fields, coef = _elastic(case, seed)
    now, before, out = (f.double() for f in fields)
    m1y, m1x, m1z, m2, m3, m23 = coef.double()
    n = (case["ny"], case["nx"], case["nz"])
    Y, X, Z = 0, 1, 2

    def part(p, axis, o):
        return p[tuple(slice(5 + (o if a == axis else 0), 5 + n[a] + (o if a == axis else 0)) for a in range(3))]

    def ga(p, axis):  # offsets -5..4
        return sum(C[5 - d] * (part(p, axis, -d) - part(p, axis, d - 1)) for d in range(1, 6))

    def gb(p, axis):  # offsets -4..5
        return sum(C[5 - d] * (part(p, axis, 1 - d) - part(p, axis, d)) for d in range(1, 6))

    def mid(f):
        return f[:, 5:-5, 5:-5, 5:-5]

    for s in range(case["steps"]):
        vy, vx, vz, yy, xx, zz, xy, xz, yz = now
        pxy, pxz, pyz, qx, qy, qz = m3 * xy, m3 * xz, m3 * yz, m1x * vx, m1y * vy, m1z * vz
        inc = torch.stack([
            ga(m23 * yy + m2 * (zz + xx), Y) + gb(pyz, Z) + gb(pxy, X),
            ga(m23 * xx + m2 * (yy + zz), X) + gb(pxy, Y) + gb(pxz, Z),
            ga(m23 * zz + m2 * (xx + yy), Z) + gb(pyz, Y) + gb(pxz, X),
            gb(qy, Y), gb(qx, X), gb(qz, Z), gb(qy, X) + gb(qx, Y), gb(qx, Z) + gb(qz, X), gb(qy, Z) + gb(qz, Y)])
        mid(out).add_(mid(before) + inc)
        if s < case["steps"] - 1:
            out, now, before = before, out, now
    return dict(now=now, before=before, out=out)


def exact(case, seed):
    kind = case["kind"]
    if kind == "acoustic":
        if 2.0 * case["n1"] * case["n2"] * case["n3"] * case["nt"] > 1.2e10:  # more than about 20 seconds
            return None
        return _acoustic64(_volume(case, seed))
    if kind == "elastic3d":
        return _elastic64(case, seed)
    if kind == "op3":
        d = _histories(case, seed)
        g = _Grid(case["nz"], case["nx"], d["coefs"], 0, 10.0, 1e-3)
        h = [torch.tensor(a.transpose(2, 0, 1).astype(np.float64), device="cuda") for a in d["hist"]]
        for L in range(case["nt"] - 3, -1, -1):
            inc = g.apply_t([a[L + 1] for a in h])
            for a, b in zip(h, inc):
                a[L] += a[L + 2] + b
        return [a.permute(1, 2, 0).cpu().numpy() for a in h]
    if kind == "batch":
        d = _survey(case, seed)
        if sum(s["nz"] * s["nx"] for s in d["specs"]) * case["nt"] > 8e9:
            return None
        stack, images = torch.zeros((3, case["nz"], case["nx"]), **_D), []
        for s, c, r in zip(d["specs"], d["coefs"], d["recs"]):
            g = _Grid(s["nz"], s["nx"], c, case["abc"], case["dx"], case["dt"])
            layers = [_Layer(g, p, a) for p, a in zip(d["nets"], (0, 1))] if d["nets"] else (None, None)
            img = _migrate64(g, case["nt"], s["zs"], s["xs"], d["wav"], s["zr"], s["rx0"], r, case["adj_abc"],
                             case["snap_every"], *layers)
            at = (slice(None), slice(s["img_z0"], s["img_z0"] + s["img_nz"]), slice(s["img_x0"], s["img_x0"] + s["img_nx"]))
            stack[:, :, s["stack_x0"]:s["stack_x0"] + s["img_nx"]] += img[at]
            images.append(tuple(img.cpu().numpy()))
        out = dict(stack=tuple(stack.cpu().numpy()))
        if case["images"]:
            out["images"] = images
        return out
    d = _single(case, seed)
    nt = case["nt"]
    # the operator forms the coefficients itself, the other calls are given them
    coefs = _coefs(*d["lame"], d["dx"], d["dt"], np.float64 if kind == "operator" else np.float32)
    g = _Grid(d["nz"], d["nx"], coefs, d["abc"], d["dx"], d["dt"])
    at = (d["zs"], d["xs"], d["wav"])
    if kind == "operator":
        # its own wavelet: silent for the first 24 samples
        wav = np.where(np.arange(1, nt + 1) >= 25, _ricker(nt, float(_F(d["dt"])), d["fp"]).astype(np.float64), 0.0)
        at = (d["zs"], d["xs"], wav)
        if case["adj"]:
            img = _migrate64(g, nt, *at, d["zr"], d["rx0"], d["rec"], 0, 1)
            return dict(zip(("drho", "dlambda", "dmu"), img.cpu().numpy()))
        rec = _born64(g, nt, *at, d["zr"], d["rx0"], d["nrx"], d["dm"])
        return dict(record=[a.T.cpu().numpy() for a in rec])
    if kind == "forward":
        rec, last, _, _ = _forward64(g, nt, *at, d["zr"], d["rx0"], d["nrx"])
        return dict(record=rec.cpu().numpy(), last=[a.cpu().numpy() for lev in last for a in lev])
    img = _migrate64(g, nt, *at, d["zr"], d["rx0"], d["rec"], case["adj_abc"], case["snap_every"])
    return tuple(img.cpu().numpy())
