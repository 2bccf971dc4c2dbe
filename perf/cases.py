"""What a user of this package has it do, as measurable cases.

    listed()            the cases, plain dicts
    draw(rng)           one more case of the same ranges
    prepare(case, seed) what a program holds before the call: model, plan, wavelet, source cell
    run(state)          one pass through the public entry points, and its results
    work(case)          bytes and operations one pass cannot do without
    exact(case, seed)   the results in 64 bits, from torch alone

Kinds of pass:
    loop       the reference front-end's loop: DRIVER_InsertSource + DRIVER_Propagate for every
               step, then the pressure snapshot by DRIVER_Update_pointers
    shot       one shot of a survey over an initialised model: fields to zero, a captured
               multi-step run, the receiver gather
    batch      many shots on sub-grids of their own, advanced together, their gathers
    model_run  a whole modelling call on a new model: initialise, run, snapshot, finalise
    ref64      the FP64 reference run: create, run, gather

The library keeps one grid (one batch) per process, so a survey program initialises its model
once and then runs shot after shot on it: for loop, shot and batch the model belongs to the
case (the plan) and the shot - its source cell and wavelet - to the seed.  For model_run and
ref64, which set the model up inside the call, the model is the seed's too.
"""
import math

import numpy as np
import torch

import fletcher_petrobras_amd as F

BORD = 4


def _case(name, kind, n, steps, precision="fp32", variant="fused", absorb=16, h=(12.5, 12.5, 12.5),
          every=4, tuned=False, shots=0):
    return {"name": name, "kind": kind, "nx": n[0], "ny": n[1], "nz": n[2], "absorb": absorb,
            "dx": h[0], "dy": h[1], "dz": h[2], "steps": steps, "precision": precision,
            "variant": variant, "every": every, "tuned": tuned, "shots": shots}


def listed():
    return [
        # the smallest calls: a teaching-size grid through the unmodified front-end's loop, where
        # the launches and waits of a step cost more than its cells
        _case("loop_tiny", "loop", (40, 36, 32), 100, absorb=8),
        # the reference's smallest published grid, 88^3, through the same loop, untuned
        _case("loop_88", "loop", (88, 88, 88), 200),
        # the headline grid, 344^3, FP32 through the per-step API (tuned as the benchmark does)
        _case("loop_344", "loop", (344, 344, 344), 120, tuned=True),
        # a survey shot on an odd-sized grid, FP32, captured multi-step run with receivers
        _case("shot_fp32_odd", "shot", (301, 257, 333), 150, tuned=True),
        # the fastest form that keeps the accuracy bar, block floating-point coefficients, 344^3
        _case("shot_q16r_344", "shot", (344, 344, 344), 150, precision="q16r", tuned=True),
        # FP32 with recomputed angular coefficients, unequal spacings, a wide shallow grid
        _case("shot_fp32r_aniso", "shot", (470, 262, 150), 150, precision="fp32r",
              h=(12.5, 10.0, 8.0), tuned=True),
        # the reference's original form: direct 64-point mixed derivatives
        _case("shot_direct", "shot", (152, 200, 176), 60, variant="direct"),
        # the reference's der1der1 structure: first-derivative volumes, then the update
        _case("shot_twopass", "shot", (184, 168, 152), 100, variant="twopass"),
        # a batch of shots with ragged apertures, FP32
        _case("batch_fp32", "batch", (168, 152, 128), 60, tuned=True, shots=12),
        # the same kind in FP16 recompute, smaller and more of them
        _case("batch_fp16r", "batch", (136, 144, 96), 100, precision="fp16r", tuned=True, shots=20),
        # the command-line program's whole call on a new model, 88^3
        _case("model_run_88", "model_run", (88, 88, 88), 300),
        # the FP64 accuracy reference of a window
        _case("ref64_window", "ref64", (104, 96, 112), 300),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["loop", "loop", "shot", "shot", "shot", "batch", "model_run", "ref64"])
    variant, precision, shots, tuned = "fused", "fp32", 0, False
    if kind == "shot":
        variant = rng.choice(["fused", "fused", "fused", "direct", "twopass"])
        if variant == "fused":
            precision = rng.choice(["fp32", "fp32r", "fp16r", "q16r", "fp16", "bf16"])
        tuned = variant == "fused" and rng.random() < 0.6
    elif kind == "batch":
        precision = rng.choice(["fp32", "fp16r", "q16r"])
        shots = rng.randint(3, 20)
        tuned = rng.random() < 0.5
    lo, hi = {"loop": (20, 344), "shot": (64, 344), "batch": (60, 168), "model_run": (40, 120),
              "ref64": (40, 120)}[kind]
    if kind == "shot" and variant != "fused":
        hi = 208
    base = _log(rng, lo, hi)
    n = [max(20, min(hi, int(base * rng.uniform(0.75, 1.3)))) for _ in range(3)]
    h = (12.5, 12.5, 12.5) if rng.random() < 0.7 else (12.5, 10.0, 8.0)
    steps = {"loop": 100, "shot": 100, "batch": 50, "model_run": 200, "ref64": 200}[kind]
    c = _case("", kind, n, steps if variant != "direct" else 50, precision=precision, variant=variant,
              absorb=rng.choice([8, 12, 16]), h=h, tuned=tuned, shots=shots)
    del c["name"]
    return c


# ---------------------------------------------------------------------- inputs

def _shape(c, n=None):
    nx, ny, nz = n or (c["nx"], c["ny"], c["nz"])
    e = 2 * BORD + 2 * c["absorb"]
    return (nz + e, ny + e, nx + e)


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _model(shape, absorb, seed):
    """Heterogeneous TTI model: vpz growing with depth plus smooth anomalies, random velocities
    in the absorbing zone, smooth epsilon > delta, theta, phi, vsv from sigma = 0.75.  Six
    float32 arrays in the order of F.MODEL_NAMES, on the host."""
    dev = _device()
    r = np.random.RandomState(seed % (1 << 31))
    ax = [torch.linspace(0, 1, s, dtype=torch.float32, device=dev) for s in shape]
    z, y, x = ax[0][:, None, None], ax[1][None, :, None], ax[2][None, None, :]

    def smooth(k):
        f, g = r.uniform(1.0, 4.0, (k, 3)), r.uniform(0, 2 * math.pi, (k, 3))
        t = 0.0
        for i in range(k):
            t = t + (torch.sin(2 * math.pi * f[i, 0] * z + g[i, 0]) * torch.sin(2 * math.pi * f[i, 1] * y + g[i, 1]) *
                     torch.sin(2 * math.pi * f[i, 2] * x + g[i, 2]))
        return t / k  # in [-1, 1]

    vpz = 1800.0 + 2200.0 * z + 350.0 * smooth(3)
    b = BORD
    depth = torch.zeros(shape, dtype=torch.float32, device=dev)  # 0 inside, 1 at the outer rim
    for axis, s in enumerate(shape):
        i = torch.arange(s, device=dev, dtype=torch.float32)
        d = torch.clamp((b + absorb - torch.minimum(i, s - 1 - i)) / absorb, 0, 1)
        depth = torch.maximum(depth, d.reshape([-1 if k == axis else 1 for k in range(3)]))
    gen = torch.Generator(device=dev)
    gen.manual_seed(int(r.randint(1 << 30)))
    vpz = vpz * (1.0 - 0.6 * depth * torch.rand(shape, generator=gen, device=dev))
    eps = 0.18 + 0.08 * smooth(2)
    dlt = 0.05 + 0.04 * smooth(2)
    theta = 0.5 + 0.45 * smooth(2)
    phi = 0.8 + 0.7 * smooth(2)
    vsv = vpz * torch.sqrt((eps - dlt) / 0.75)
    return [np.ascontiguousarray(a.expand(shape).cpu().numpy()) for a in (vpz, vsv, eps, dlt, phi, theta)]


def _dt(c):
    """One dt per case: the velocity stays below 4400 m/s and epsilon below 0.26."""
    return float(np.float32(0.35 * min(c["dx"], c["dy"], c["dz"]) / (4400.0 * math.sqrt(1.52))))


def _wavelet(c, seed):
    """Ricker wavelet of a peak frequency of its own, as float32 samples of the steps."""
    r = np.random.RandomState((seed * 7 + 3) % (1 << 31))
    n, dt = c["steps"], _dt(c)
    f = r.uniform(0.8, 1.2) * 1.2 / (0.4 * n * dt)
    u = (math.pi * f * (np.arange(n) * dt - 1.2 / f)) ** 2
    return ((1.0 - 2.0 * u) * np.exp(-u) * r.uniform(0.5, 2.0)).astype(np.float32)


def _source_cell(c, shape, seed):
    r = np.random.RandomState((seed * 5 + 1) % (1 << 31))
    e = BORD + c["absorb"]
    sz, sy, sx = shape
    ix, iy, iz = int(r.randint(e, sx - e)), int(r.randint(e, sy - e)), min(e + 2 + int(r.randint(6)), sz - e)
    return (iz * sy + iy) * sx + ix


def _receivers(c):
    return BORD + c["absorb"] + 1


def _apertures(c):
    """Interior extents (nx, ny, nz) of the batch's shots: at most the case's, ragged in x and y."""
    r = np.random.RandomState((c["nx"] * 31 + c["shots"]) % (1 << 31))
    return [(int(c["nx"] * r.uniform(0.55, 1.0)), int(c["ny"] * r.uniform(0.55, 1.0)), c["nz"])
            for _ in range(c["shots"])]


def _batch_models(c):
    out = []
    for k, n in enumerate(_apertures(c)):
        shape = _shape(c, n)
        out.append((shape, _model(shape, c["absorb"], 9000 + k), _source_cell(c, shape, 100 + k)))
    return out


def _plan_model(c):
    return _model(_shape(c), c["absorb"], 1234)


# The library's one grid and one batch of this process: the plan that was set up last.
_current = {"key": None, "plan": None}


def _driver(c):
    d = F.Driver(variant=c["variant"], precision=c["precision"], tiles=(12, 0))
    d.set_stream_hints(False)
    d.set_lane_pairs(True)
    return d


def _plan(c):
    """The set-up plan of a case (model on the device, tiles, receivers)."""
    key = tuple(sorted((k, v) for k, v in c.items() if k != "name"))
    if _current["key"] == key:
        return _current["plan"]
    if isinstance(_current["plan"], F.Batch):
        _current["plan"].destroy()
    elif _current["plan"] is not None:
        _current["plan"].finalize()
    _current["key"] = _current["plan"] = None
    h = (c["dx"], c["dy"], c["dz"])
    if c["kind"] == "batch":
        F.Driver().set_device_precompute(True)
        shots = [{"model": m, "isource": i, "rec_iz": _receivers(c)} for _, m, i in _batch_models(c)]
        p = F.Batch(shots, h, _dt(c), precision=c["precision"], tiles=(12, 0))
        p.set_lane_pairs(True)
        p.reset()
        if c["tuned"]:
            p.autotune(2)
    else:
        p = _driver(c)
        p.set_device_precompute(True)
        p.initialize(_shape(c), h, _dt(c), _plan_model(c))
        if c["tuned"]:
            p.autotune(3)
        if c["kind"] == "shot":
            p.record_traces(_receivers(c), c["every"], c["steps"] // c["every"])
    _current["key"], _current["plan"] = key, p
    return p


def prepare(case, seed):
    c = dict(case)
    shape = _shape(c)
    s = {"case": c, "wavelet": _wavelet(c, seed), "isource": _source_cell(c, shape, seed)}
    if c["kind"] in ("model_run", "ref64"):
        s["model"] = _model(shape, c["absorb"], seed)
    else:
        _plan(c)
    if c["kind"] in ("loop", "model_run"):
        s["pc"] = np.zeros(shape, np.float32)  # the front-end's own snapshot array
    return s


# ---------------------------------------------------------------------- one pass

def run(state):
    c, src, isrc = state["case"], state["wavelet"], state["isource"]
    h, dt, shape = (c["dx"], c["dy"], c["dz"]), _dt(c), _shape(c)
    if c["kind"] == "loop":
        d = _plan(c)
        d.reset_fields()
        for it in range(1, c["steps"] + 1):
            d.insert_source(it - 1, isrc, float(src[it - 1]))
            d.propagate(it)
        return {"pc": d.update_pointers(state["pc"])}
    if c["kind"] == "shot":
        d = _plan(c)
        d.reset_fields()
        d.run(c["steps"], isrc, src=src)
        return {"traces": d.traces()}
    if c["kind"] == "batch":
        b = _plan(c)
        b.reset()
        b.run(c["steps"], rec_every=c["every"], max_traces=c["steps"] // c["every"], src=src)
        return {"traces": [b.traces(k) for k in range(c["shots"])]}
    if c["kind"] == "model_run":
        _current["key"] = _current["plan"] = None  # the call takes the library's grid
        d = _driver(c)
        d.set_device_precompute(False)
        d.initialize(shape, h, dt, state["model"])
        d.run(c["steps"], isrc, src=src)
        pc = d.update_pointers(state["pc"])
        d.finalize()
        return {"pc": pc}
    r = F.Ref64(shape, h, dt, state["model"])
    r.run(c["steps"], isrc, src=src, rec_iz=_receivers(c), rec_every=c["every"],
          max_traces=c["steps"] // c["every"])
    out = {"traces": r.traces(), "pc": r.field("pc")}
    r.destroy()
    return out


# ---------------------------------------------------------------------- what a pass needs

_COEF_BYTES = {"fp32": 40, "bf16": 20, "fp16": 20, "fp16r": 12, "q16r": 12, "fp32r": 24}


def work(case):
    """Per updated cell and step: both fields of the current and the previous level read, the
    new level written, the coefficients read; the whole modelling calls also read the model and
    write the snapshot.  Operations: der2 13, der1 11 (direct mixed derivative 67) flops."""
    c = dict(case)
    if c["kind"] == "batch":
        cells = sum(n[0] * n[1] * n[2] for n in [[e + 2 * c["absorb"] for e in a] for a in _apertures(c)])
    else:
        sz, sy, sx = _shape(c)
        cells = (sx - 2 * BORD) * (sy - 2 * BORD) * (sz - 2 * BORD)
    wide = 2 if c["kind"] == "ref64" else 1
    per = wide * (24 + _COEF_BYTES[c["precision"]])
    flops = (525 if c["variant"] == "direct" else 233) * cells * c["steps"]
    total = per * cells * c["steps"]
    if c["kind"] in ("model_run", "ref64"):
        total += 24 * cells
    if c["kind"] in ("loop", "model_run"):
        total += 4 * cells
    return {"bytes": total, "flops": flops}


# ---------------------------------------------------------------------- 64-bit results

_W1 = (4.0 / 5.0, -1.0 / 5.0, 4.0 / 105.0, -1.0 / 280.0)
_W2 = (-205.0 / 72.0, 8.0 / 5.0, -1.0 / 5.0, 8.0 / 315.0, -1.0 / 560.0)


def _cut(f, axis, shift, lo, hi):
    """f displaced by shift along axis, over indices [lo, hi) of that axis."""
    return f.narrow(axis, lo + shift, hi - lo)


def _d1(f, axis, h):
    s = f.shape[axis]
    t = None
    for k, w in enumerate(_W1, 1):
        v = (_cut(f, axis, k, BORD, s - BORD) - _cut(f, axis, -k, BORD, s - BORD)) * (w / h)
        t = v if t is None else t.add_(v)
    return t


def _d2(f, axis, h):
    s = f.shape[axis]
    t = _cut(f, axis, 0, BORD, s - BORD) * (_W2[0] / h / h)
    for k, w in enumerate(_W2[1:], 1):
        t.add_(_cut(f, axis, k, BORD, s - BORD), alpha=w / h / h)
        t.add_(_cut(f, axis, -k, BORD, s - BORD), alpha=w / h / h)
    return t


def _inner(f, axes):
    for a in axes:
        f = f.narrow(a, BORD, f.shape[a] - 2 * BORD)
    return f


def _derivatives(f, h):
    """xx, yy, zz, xy, yz, xz over the update domain (axes 2 x, 1 y, 0 z)."""
    hx, hy, hz = h
    xx = _d2(_inner(f, (0, 1)), 2, hx)
    yy = _d2(_inner(f, (0, 2)), 1, hy)
    zz = _d2(_inner(f, (1, 2)), 0, hz)
    fx = _d1(f, 2, hx)
    xy = _d1(_inner(fx, (0,)), 1, hy)
    xz = _d1(_inner(fx, (1,)), 0, hz)
    del fx
    yz = _d1(_d1(_inner(f, (2,)), 1, hy), 0, hz)
    return xx, yy, zz, xy, yz, xz


def _exact_run(c, shape, model, isrc, src, want_traces):
    dev = _device()
    vpz, vsv, eps, dlt, phi, theta = [_inner(torch.from_numpy(m).to(dev), (0, 1, 2)).double() for m in model]
    h, dt = (c["dx"], c["dy"], c["dz"]), _dt(c)
    st, ct, sp, cp = torch.sin(theta), torch.cos(theta), torch.sin(phi), torch.cos(phi)
    a = [st * st * cp * cp, st * st * sp * sp, ct * ct, 2 * st * st * sp * cp, 2 * st * ct * sp, 2 * st * ct * cp]
    del st, ct, sp, cp, theta, phi
    vz = vpz * vpz * (dt * dt)
    vx, vn, vs = vz * (1 + 2 * eps), vz * (1 + 2 * dlt), vsv * vsv * (dt * dt)
    del vpz, vsv, eps, dlt
    lev = [torch.zeros(shape, dtype=torch.float64, device=dev) for _ in range(4)]  # pp pc qp qc
    iz, r = divmod(isrc, shape[1] * shape[2])
    iy, ix = divmod(r, shape[2])
    traces = []
    for it in range(1, c["steps"] + 1):
        pp, pc, qp, qc = lev
        pc[iz, iy, ix] += float(src[it - 1])
        qc[iz, iy, ix] += float(src[it - 1])
        h1, h2 = [], []
        for f in (pc, qc):
            d = _derivatives(f, h)
            lap = d[0] + d[1] + d[2]
            t = a[0] * d[0]
            for k in range(1, 6):
                t.addcmul_(a[k], d[k])
            h1.append(t)
            h2.append(lap.sub_(t))
        rp = vx * h2[0] + vz * h1[1] + vs * (h1[0] - h1[1])
        rq = vn * h2[0] + vz * h1[1] - vs * (h2[0] - h2[1])
        del h1, h2, d, t, lap
        for old, cur, rhs in ((pp, pc, rp), (qp, qc, rq)):
            o = _inner(old, (0, 1, 2))
            o.neg_().add_(_inner(cur, (0, 1, 2)), alpha=2.0).add_(rhs)
        del rp, rq
        lev = [pc, pp, qc, qp]
        if want_traces and it % c["every"] == 0:
            traces.append(_inner(lev[1][_receivers(c)], (0, 1)).clone())
    return (torch.stack(traces) if want_traces else None), lev[1]


def exact(case, seed):
    c = dict(case)
    src = _wavelet(c, seed)
    if c["kind"] == "batch":
        return {"traces": [_exact_run(c, shape, m, i, src, True)[0] for shape, m, i in _batch_models(c)]}
    shape = _shape(c)
    model = _model(shape, c["absorb"], seed) if c["kind"] in ("model_run", "ref64") else _plan_model(c)
    tr, pc = _exact_run(c, shape, model, _source_cell(c, shape, seed), src, c["kind"] in ("shot", "ref64"))
    if c["kind"] == "ref64":
        return {"traces": tr, "pc": pc}
    return {"traces": tr} if c["kind"] == "shot" else {"pc": pc}
