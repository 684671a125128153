"""Workloads of the library's public entry points, for timing and for
comparing outputs: what a program that uses the library calls, over the range
of sizes it is used at.

Kinds of case
-------------
``step``   the drop-in: a host model's arrays up, one driver step, arrays
           down.  ``moved`` says how much: ``headline`` uploads the step's
           forcing and reads the eight headline fluxes back (the state stays
           on the device), ``all`` moves every field both ways, as a host
           model that owns the state does.
``run``    the device-resident run of a window of half-hourly steps in plain
           FP64 or mixed precision, then the results read back.
``hybrid`` the same with the surrogate's warm start of the leaf iteration.
``train``  Adam batches of the surrogate on samples held on the device.
``net``    the surrogate's forward pass and gradient for host rows.

``order`` is the tile order a production run sets (class, temperature band,
soil, leaf area) or the caller's own.  ``forcing`` of a run: ``kept`` was
synthesised before the run, ``synth`` is generated for the window as part of
the pass (a run longer than its forcing window), ``met`` comes from a met
file's variables in host memory.  ``soil`` also reads the soil state back, as
a program does that writes both.  ``check`` adds the driver's consistency
sums.
"""
import math

import numpy as np

from cable_amd import gpu
from cable_amd import surrogate
from cable_amd.fields import BY_NAME, FIELDS
from cable_amd.workload import DOY, TFRZ, Workload, add_snow, synth_forcing

FLUXES = ["canopy%rnet", "canopy%fe", "canopy%fh", "canopy%fev", "canopy%fes", "canopy%fgpp", "ssnow%runoff",
          "rad%trad"]
SURFACE = ["ssnow%tss", "ssnow%snowd", "canopy%cansto"]
SOIL = ["ssnow%tgg", "ssnow%wb", "ssnow%wbice"]
STATE = [f.name for f in FIELDS if f.role == "STATE"]
WRITTEN = [f.name for f in FIELDS if f.role in ("STATE", "DIAG")]

PREC = {"fp64": gpu.PREC_FP64, "mixed": gpu.PREC_MIXED}
CAP, RESID = 4, 0.5          # the hybrid's polish passes and residual limit, as the benchmark runs it
LR = 2e-3

# Bytes a tile-step cannot do without (state read and written once, the eight
# forcing fields, the per-tile parameters, the eight outputs) and its
# floating-point operations (an average over a day, additions and products).
STEP_BYTES = {"fp64": 1016, "mixed": 756, "hybrid": 764}
STEP_FLOPS = 12000
NET_FLOPS = 2 * (24 * 128 + 2 * 128 * 128 + 128 * 8)

# Means and standard deviations of the surrogate's 24 inputs and 8 targets
# over a day of the synthetic workload, and a least-squares fit of the first
# three targets (leaf temperature, leaf-surface CO2 of both leaves) to the
# inputs, both normalised.
NORM = [119.2, 335.0, 11.81, 5.998, 3.002, 985.1, 0.2706, 3.037, 44.1, 0.1203, 9.28, 8.398, 1500.0, 0.04765, -0.07216,
        0.001, 0.8729, 0.8791, -0.01979, 0.6461, -2.927, 23.63, 0.02691, 1115.0,
        149.2, 49.04, 7.817, 3.653, 1.6, 20.2, 0.3277, 1.702, 23.4, 0.3254, 11.19, 1.627, 1.0, 0.03033, 0.1929, 1.0,
        0.2805, 4.691, 2.308, 2.669, 5.949, 51.55, 0.04682, 1754.0,
        1.112, 0.9671, 0.9825, 0.8531, 0.06405, 0.07802, 41.49, 54.01,
        3.024, 0.06079, 0.02975, 4.93, 0.1095, 0.08884, 64.91, 112.6]
FIT = [[0.84, 0.23, -0.25, 0.02, -0.03, 0.0, -0.13, -0.08, -0.06, -0.01, -0.05, 0.01, 0.0, 0.07, 0.0, 0.0, -0.06, 0.27,
        -0.05, -0.06, 0.08, -0.04, 0.04, 0.05],
       [-0.49, 0.0, -0.07, -0.12, 0.06, 0.01, -0.04, -0.1, -0.3, -0.07, 0.04, 0.07, 0.0, -0.1, -0.03, 0.0, -0.17, -0.01,
        0.01, -0.07, -0.08, -0.04, 0.02, 0.05],
       [-0.4, 0.03, -0.07, -0.03, 0.05, 0.01, -0.16, 0.0, -0.19, -0.06, -0.02, 0.06, 0.0, -0.08, 0.02, 0.0, -0.2, -0.12,
        0.01, -0.04, -0.04, -0.01, 0.0, 0.03]]
LAYERS = [(24, 128), (128, 128), (128, 128), (128, 8)]


def listed():
    return [
        # a coupled host model's single site with a small ensemble: one call
        # per half hour, all latency
        dict(name="step_fp64_77", kind="step", tiles=77, precision="fp64", moved="headline", snow=True),
        # the drop-in at a GPU's share of a global grid, state resident
        dict(name="step_fp64_262144", kind="step", tiles=262144, precision="fp64", moved="headline", snow=False),
        # the drop-in for a host model that keeps the state itself
        dict(name="step_all_fp64_49149", kind="step", tiles=49149, precision="fp64", moved="all", snow=True),
        # a regional run of a few thousand tiles in plain FP64, a day at a time
        dict(name="run_fp64_4093", kind="run", tiles=4093, steps=48, first=0, precision="fp64", snow=True, order=True,
             forcing="kept", soil=True, check=False),
        # the benchmark's plain FP64 size, a day
        dict(name="run_fp64_262144", kind="run", tiles=262144, steps=48, first=0, precision="fp64", snow=False,
             order=True, forcing="kept", soil=False, check=False),
        # a national grid in mixed precision, every field of the soil read
        # back at the end of the day
        dict(name="run_mixed_20011", kind="run", tiles=20011, steps=48, first=0, precision="mixed", snow=True,
             order=True, forcing="kept", soil=True, check=False),
        # a quarter of a day driven from a met file's variables
        dict(name="met_mixed_131071", kind="run", tiles=131071, steps=12, first=16, precision="mixed", snow=False,
             order=True, forcing="met", soil=False, check=False),
        # the benchmark's mixed-precision size, a day
        dict(name="run_mixed_1048576", kind="run", tiles=1048576, steps=48, first=0, precision="mixed", snow=False,
             order=True, forcing="kept", soil=False, check=False),
        # the hybrid over a day: a regional grid, and the benchmark's size
        # with the window's forcing generated as a production run does
        dict(name="hybrid_65537", kind="hybrid", tiles=65537, steps=48, first=0, precision="mixed", snow=True,
             order=True, forcing="kept", soil=True),
        dict(name="hybrid_1048576", kind="hybrid", tiles=1048576, steps=48, first=0, precision="mixed", snow=False,
             order=True, forcing="synth", soil=False),
        # surrogate training at the benchmark's batch
        dict(name="train_2048", kind="train", batch=2048, batches=32, samples=524288),
        # a gradient and a prediction for host rows (diagnosing the network)
        dict(name="net_5000", kind="net", rows=5000),
    ]


def _log_int(rng, lo, hi):
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return max(lo, min(hi, n))


def draw(rng):
    kind = rng.choice(["step", "run", "run", "run", "hybrid", "hybrid", "train", "net"])
    if kind == "step":
        moved = rng.choice(["headline", "headline", "all"])
        return dict(kind=kind, tiles=_log_int(rng, 32, 262144 if moved == "headline" else 65536),
                    precision=rng.choice(["fp64", "fp64", "mixed"]), moved=moved, snow=rng.random() < 0.5)
    if kind == "run":
        prec, forcing = rng.choice(["fp64", "mixed"]), rng.choice(["kept", "kept", "synth", "met"])
        most = 131072 if forcing == "met" else 262144 if prec == "fp64" else 1048576
        return dict(kind=kind, tiles=_log_int(rng, 256, most), steps=rng.randint(8, 12 if forcing == "met" else 48),
                    first=2 * rng.randint(0, 23), precision=prec, snow=rng.random() < 0.5, order=rng.random() < 0.8,
                    forcing=forcing, soil=rng.random() < 0.5, check=rng.random() < 0.25)
    if kind == "hybrid":
        return dict(kind=kind, tiles=_log_int(rng, 256, 1048576), steps=rng.randint(8, 48),
                    first=2 * rng.randint(0, 23), precision="mixed", snow=rng.random() < 0.5,
                    order=rng.random() < 0.8, forcing=rng.choice(["kept", "synth"]), soil=rng.random() < 0.5)
    if kind == "train":
        return dict(kind=kind, batch=rng.choice([256, 500, 1024, 2048, 2048, 4096]), batches=rng.randint(8, 48),
                    samples=_log_int(rng, 16384, 524288))
    return dict(kind=kind, rows=_log_int(rng, 16, 20000))


# ---------------------------------------------------------------------------
# inputs

def _workload(case, seed):
    wl = Workload(case["tiles"], 1, seed=7000 + int(seed), forcing=False)
    return add_snow(wl) if case["snow"] else wl


def _params(seed):
    """A network as training leaves it, near enough: the fit above carried
    through the first units of each layer (hard-swish is the identity above
    3, so they ride on an offset of 8), small weights in the rest."""
    rng = np.random.default_rng(90000 + int(seed))
    w = [rng.uniform(-0.05, 0.05, s) for s in LAYERS]
    b = [np.zeros(s[1]) for s in LAYERS]
    fit = np.array(FIT).T
    w[0][:, :24] = np.eye(24)
    b[0][:24] = 8.0
    w[1][:, :3] = 0.0
    w[1][:24, :3] = fit
    b[1][:3] = 8.0 - 8.0 * fit.sum(0)
    w[2][:, :3] = 0.0
    w[2][:3, :3] = np.eye(3)
    w[3][:] = rng.uniform(-0.01, 0.01, LAYERS[3])
    w[3][:3, :] = 0.0
    w[3][:3, :3] = np.eye(3)
    b[3][:3] = -8.0
    return np.concatenate([np.concatenate([x.ravel(), y]) for x, y in zip(w, b)]).astype(np.float32)


def _rows(rng, n):
    """Raw samples: inputs of the workload's spread, targets a smooth map of
    them with some scatter."""
    norm = np.array(NORM, dtype=np.float32)
    z = rng.standard_normal((n, 24), dtype=np.float32)
    t = rng.standard_normal((n, 8), dtype=np.float32) * np.float32(0.1)
    t[:, :3] += z @ np.array(FIT, dtype=np.float32).T
    t[:, 3:] += np.tanh(z[:, :5] + z[:, 5:10] * z[:, 10:15] * np.float32(0.5))
    return z, t, norm


def _met(case, wl, seed):
    """A met file's variables for the window (FP32, in the file's units)."""
    n, ns = case["tiles"], case["steps"]
    rng = np.random.default_rng(50000 + int(seed))
    hod = (0.5 * (case["first"] + np.arange(ns)))[:, None].astype(np.float32)
    u = [rng.random((ns, n), dtype=np.float32) for _ in range(5)]
    tair = (wl.t0[None, :] + 5.0 * np.sin(2.0 * np.pi * (hod - 9.0) / 24.0)).astype(np.float32)
    sun = np.maximum(0.0, 1000.0 * np.sin(2.0 * np.pi * (hod - 6.0) / 24.0))
    es = 6.112 * np.exp(17.67 * (tair - 273.15) / (tair - 29.65))
    psurf = 95000.0 + 7000.0 * u[4]
    rain = np.where(u[3] < 0.1, -np.log1p(-u[2]), 0.0) / 1800.0
    return {"swdown": (sun * (0.5 + 0.5 * u[0])).astype(np.float32), "lwdown": (250.0 + 170.0 * u[1]).astype(np.float32),
            "tair": tair, "qair": (0.622 * (0.3 + 0.6 * u[2]) * es / (psurf * 0.01)).astype(np.float32),
            "wind": (0.5 + 5.0 * u[3]).astype(np.float32), "psurf": psurf.astype(np.float32),
            "rainf": rain.astype(np.float32), "tair_offset": 0.0, "psurf_scale": 0.01, "rainf_scale": 1800.0}


def _prepare_step(case, seed):
    wl = _workload(case, seed)
    g = gpu.from_workload(wl, precision=PREC[case["precision"]], full=True)
    # the host's forcing of a morning's steps, in turn
    f = synth_forcing(wl.t0, wl.lat, 20, 4, seed=seed)
    steps = []
    for k in range(4):
        tk, rain = f["met%tk"][k], f["met%precip"][k]
        one = {"met%fsd": np.stack([f["met%fsd"][k]] * 2), "met%tvair": tk.copy(), "met%tvrad": tk,
               "met%precip_sn": np.where(tk <= TFRZ, rain, 0.0), "met%ca": np.full(wl.n, 400.0e-6),
               "met%doy": np.full(wl.n, DOY)}
        one.update({n: f[n][k] for n in ("met%fld", "met%tk", "met%qv", "met%ua", "met%pmb", "met%precip",
                                         "met%coszen")})
        steps.append(one)
    s = {"case": case, "g": g, "forcing": steps, "k": 0, "dels": wl.dels}
    if case["moved"] == "all":
        host = {x.name: np.zeros(x.shape(wl.n)) for x in FIELDS}
        for d in (wl.params, wl.state0):
            for name, v in d.items():
                if name in host:
                    host[name][...] = np.asarray(v, dtype=np.float64).reshape(host[name].shape)
        s["host"] = host
    else:
        s["out"] = {n: np.empty(BY_NAME[n].shape(wl.n)) for n in FLUXES + SURFACE}
    return s


def _prepare_run(case, seed):
    wl = _workload(case, seed)
    order = gpu.class_order(wl.iveg, wl.isoilm, wl.vlai, tair=wl.t0) if case["order"] else None
    g = gpu.from_workload(wl, precision=PREC[case["precision"]], full=False, order=order)
    s = {"case": case, "g": g, "seed": int(seed), "t0": wl.t0, "lat": wl.lat, "dels": wl.dels}
    if case["forcing"] == "kept":
        g.synth_forcing(case["first"], case["steps"], s["seed"], wl.t0, wl.lat, dels=wl.dels)
    if case["forcing"] == "met":
        s["met"] = _met(case, wl, seed)
    if case["kind"] == "hybrid":
        g.set_surrogate(_params(seed), np.array(NORM, dtype=np.float32))
        g.set_launch_timing(False)
    elif case["check"]:
        g.consistency_check(True)
    s["names"] = FLUXES + SURFACE + (SOIL if case["soil"] else [])
    s["out"] = {n: np.empty(BY_NAME[n].shape(wl.n)) for n in s["names"]}
    return s


def prepare(case, seed):
    kind = case["kind"]
    if kind == "step":
        return _prepare_step(case, seed)
    if kind in ("run", "hybrid"):
        return _prepare_run(case, seed)
    rng = np.random.default_rng(30000 + int(seed))
    if kind == "train":
        z, t, norm = _rows(rng, case["samples"])
        net = surrogate.MLP(batch=case["batch"], params=surrogate.init_params(int(seed)), norm=norm)
        net.load_samples(z * norm[24:48] + norm[:24], t * norm[56:64] + norm[48:56])
        return {"case": case, "net": net, "seed": int(seed)}
    z, t, norm = _rows(rng, case["rows"])
    net = surrogate.MLP(batch=case["rows"], params=surrogate.init_params(int(seed)), norm=norm)
    return {"case": case, "net": net, "x": z, "t": t}


# ---------------------------------------------------------------------------
# one pass

def _typed(precision, arrays):
    """The values in the type the device holds them in (FP32 for the mixed
    path's default reals)."""
    narrow = precision == "mixed"
    return [a.astype(np.float32) if narrow and BY_NAME[n].prec == "F" else a for n, a in arrays]


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "step":
        g, k = state["g"], state["k"]
        state["k"] = k + 1
        met = state["forcing"][k % 4]
        if case["moved"] == "all":
            host = state["host"]
            for n, v in met.items():
                host[n] = v
            g.upload_fields(host)
            g.step(k + 1, state["dels"])
            g.download_fields(WRITTEN, out=host)
            return _typed(case["precision"], [(n, host[n]) for n in FLUXES + STATE])
        g.upload_fields(met)
        g.step(k + 1, state["dels"])
        out = g.download_fields(FLUXES + SURFACE, out=state["out"])
        return _typed(case["precision"], out.items())
    if kind in ("run", "hybrid"):
        g, first, steps, dels = state["g"], case["first"], case["steps"], state["dels"]
        if case["forcing"] == "synth":
            g.synth_forcing(first, steps, state["seed"], state["t0"], state["lat"], dels=dels)
        elif case["forcing"] == "met":
            g.set_met(first, steps, dels, state["met"], state["lat"], start=(0.0, 172, 6, 2001))
        if kind == "hybrid":
            g.run_hybrid(first, steps, dels, max_passes=CAP, resid_max=RESID)
        else:
            g.run(first, steps, dels)
        out = _typed(case["precision"], g.download_fields(state["names"], out=state["out"]).items())
        if kind == "run" and case["check"]:
            c = g.consistency_values()
            out.append(np.array([c["new_sumbal"], c["sum_fe"], c["sum_fpn"], c["ebal_tot"], c["wbal_tot"]]))
        return out
    net = state["net"]
    if kind == "train":
        losses = net.train(epochs=case["batches"] * case["batch"] / case["samples"], lr=LR, seed=state["seed"])
        return [losses, net.params()]
    y = net.forward(state["x"])
    loss, grad = net.gradient(state["x"], state["t"])
    return [y, loss, grad]


def work(case):
    kind = case["kind"]
    if kind == "step":
        vals = sum(f.n for f in FIELDS)
        written = sum(BY_NAME[n].n for n in WRITTEN)
        size = 8 if case["precision"] == "fp64" else 4
        moved = (vals + written if case["moved"] == "all" else 14 + 11) * size
        return {"bytes": case["tiles"] * (moved + (vals + written) * size), "flops": case["tiles"] * STEP_FLOPS}
    if kind in ("run", "hybrid"):
        ts = case["tiles"] * case["steps"]
        form = "hybrid" if kind == "hybrid" else case["precision"]
        return {"bytes": ts * STEP_BYTES[form],
                "flops": ts * (STEP_FLOPS + (0.3 * NET_FLOPS if kind == "hybrid" else 0))}
    if kind == "train":
        # samples, and parameters with both moments read and written
        rows = case["batch"] * case["batches"]
        return {"bytes": rows * 128 + case["batches"] * surrogate.NPARAM * 24, "flops": 3 * rows * NET_FLOPS}
    n = case["rows"]
    return {"bytes": n * (24 * 8 + 8 * 8) + surrogate.NPARAM * 12, "flops": 4 * n * NET_FLOPS}


# ---------------------------------------------------------------------------
# 64-bit values, where there are any (the physics has none in plain numpy)

def _unpack(p):
    w, b, o = [], [], 0
    for i, n in LAYERS:
        w.append(p[o:o + i * n].reshape(i, n))
        b.append(p[o + i * n:o + i * n + n])
        o += i * n + n
    return w, b


def _forward64(p, x):
    w, b = _unpack(p)
    zs, hs = [], [x]
    for k in range(4):
        z = hs[-1] @ w[k] + b[k]
        zs.append(z)
        hs.append(z * np.clip(z + 3.0, 0.0, 6.0) / 6.0 if k < 3 else z)
    return zs, hs


def _gradient64(p, x, t):
    w, _ = _unpack(p)
    zs, hs = _forward64(p, x)
    d = hs[-1] - t
    loss = float(np.mean(d * d))
    d = 2.0 * d / d.size
    out = []
    for k in range(3, -1, -1):
        out.append(np.concatenate([(hs[k].T @ d).ravel(), d.sum(0)]))
        if k:
            z = zs[k - 1]
            d = (d @ w[k].T) * np.where(z < -3.0, 0.0, np.where(z > 3.0, 1.0, (2.0 * z + 3.0) / 6.0))
    return loss, np.concatenate(out[::-1])


def _mix64(z):
    m = (1 << 64) - 1
    z = (z + 0x9E3779B97F4A7C15) & m
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & m
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & m
    return z ^ (z >> 31)


def _sample_order(seed, n, count):
    """The documented order of the training samples: each epoch a keyed
    bijection of the next power of two, walked until it lands below n."""
    bits = max(1, (n - 1).bit_length())
    mask, sh = np.uint64((1 << bits) - 1), np.uint64((bits + 1) // 2)
    out = np.empty(count, dtype=np.int64)
    for e in range(-(-count // n)):
        keys = [_mix64((seed ^ _mix64(4 * e + r)) & ((1 << 64) - 1)) for r in range(4)]
        x = np.arange(min(n, count - e * n), dtype=np.uint64)
        todo = np.arange(x.size)
        while todo.size:
            v = x[todo]
            for key in keys:
                v = (v * np.uint64(key | 1)) & mask
                v ^= v >> sh
                v = (v + np.uint64(key >> 32)) & mask
            x[todo] = v
            todo = todo[v >= np.uint64(n)]
        out[e * n:e * n + x.size] = x
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind not in ("train", "net"):
        return None
    rng = np.random.default_rng(30000 + int(seed))
    p = np.random.default_rng(int(seed))
    parts = []
    for k, (i, n) in enumerate(LAYERS):
        lim = np.sqrt(6.0 / i) * (0.5 if k == 3 else 1.0)
        parts += [p.uniform(-lim, lim, i * n), np.zeros(n)]
    p = np.concatenate(parts).astype(np.float32).astype(np.float64)
    if kind == "net":
        z, t, _ = _rows(rng, case["rows"])
        z, t = z.astype(np.float64), t.astype(np.float64)
        loss, grad = _gradient64(p, z, t)
        return [_forward64(p, z)[1][-1], loss, grad]
    z, t, norm = _rows(rng, case["samples"])
    x, y = (z * norm[24:48] + norm[:24]).astype(np.float64), (t * norm[56:64] + norm[48:56]).astype(np.float64)
    norm = norm.astype(np.float64)
    nb, batch = case["batches"], case["batch"]
    order = _sample_order(int(seed), case["samples"], nb * batch)
    m, v, losses = np.zeros_like(p), np.zeros_like(p), []
    lr = LR + (0.1 * LR - LR) * 0.5
    for k in range(nb):
        rows = order[k * batch:(k + 1) * batch]
        loss, g = _gradient64(p, (x[rows] - norm[:24]) / norm[24:48], (y[rows] - norm[48:56]) / norm[56:64])
        losses.append(loss)
        m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
        p = p - lr * (m / (1.0 - 0.9 ** (k + 1))) / (np.sqrt(v / (1.0 - 0.999 ** (k + 1))) + 1e-8)
    return [np.array(losses), p]
