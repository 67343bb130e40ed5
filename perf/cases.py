"""Cases that measure this framework on what its users have it do.

Every case goes through the public entry points (DyadHIP, QuasiStationarySites,
surrogate.qs_solve, mlp.MLP).  Kinds:

  step      a batch of release sites advanced by Step(dt, k), then what a
            program reads at an output interval (states, streams, mouths,
            currents, effluxes, release statistics; whole fields where the
            batch is small enough to be written out)
  protocol  the reference solver's own loop, RunRD / RunMC / Update per step
  coupled   2D clefts inside 3D cytosol boxes with a depleting jSR
  pool2d    the reference's test input (2D, Ca and Mg, sarcolemma, jSR pool,
            cytosol pool with leak and SERCA), fields written at the end
  solve     the full-solver fallback of the quasi-stationary path
  qs        event-driven release sites with the learned surrogate
  predict   the ensemble on feature rows held on the host
  train     an epoch of ensemble training, updated weights read back

A case is a dict of plain values; see listed() for what each one stands for.
"""
import dataclasses
import json
import math
import os

import numpy as np
import torch

from casim_amd import abi, autotune, config, mlp, rng, spark_compare, surrogate, workloads
from casim_amd.dyad import DyadHIP

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
WEIGHTS = os.path.join(ROOT, "casim_amd", "surrogate_weights.npz")
TEST_INPUT = os.path.join(ROOT, "tests", "golden", "test_input_Parameters.json")
M1, M2 = rng.M1, rng.M2


def listed():
    return [
        # the quasi-stationary path's fallback: a handful of sites, thousands of dependent steps (create, solve,
        # read the mouths); the smallest batch that is in use, bound by latency
        {"name": "solve_6sites", "kind": "solve", "sites": 6, "extent": 320, "steps": 2000},
        # the single-dyad configuration with its 32 sites, one output interval of the reference's example inputs
        # (500 steps), every field written out
        {"name": "single_32sites_f64", "kind": "step", "geometry": "single", "sites": 32, "nx": 61, "ny": 61, "nz": 5,
         "precision": 64, "steps": 500, "pool": False, "warm": 300, "fields": True},
        # the benchmark's batch and graph length, both precisions: the largest calls
        {"name": "batch_4096sites_f64", "kind": "step", "geometry": "batch", "sites": 4096, "nx": 81, "ny": 81,
         "nz": 5, "precision": 64, "steps": 100, "pool": False, "fields": False},
        {"name": "batch_4096sites_f32", "kind": "step", "geometry": "batch", "sites": 4096, "nx": 81, "ny": 81,
         "nz": 5, "precision": 32, "steps": 100, "pool": False, "fields": False},
        # an untuned, ragged shape with a depleting jSR and an odd step count (spark statistics runs)
        {"name": "ragged_701sites_jsr", "kind": "step", "geometry": "batch", "sites": 701, "nx": 77, "ny": 79, "nz": 5,
         "precision": 64, "steps": 151, "pool": True, "fields": False},
        # the coupled configuration: 201 x 201 clefts in 51^3 boxes, two box steps
        {"name": "coupled_512sites", "kind": "coupled", "sites": 512, "steps": 100},
        # the reference's test input at its batch size (NumBatch 100), one output interval
        {"name": "pool2d_100sites", "kind": "pool2d", "sites": 100, "steps": 500},
        # a host that keeps the reference's step protocol, one call per DyadSeries method
        {"name": "protocol_128sites", "kind": "protocol", "sites": 128, "nx": 61, "ny": 61, "nz": 5, "warm": 300,
         "steps": 20},
        # the surrogate-driven path on the benchmark's sites, and a smaller batch with a depleting jSR
        {"name": "qs_4096sites", "kind": "qs", "sites": 4096, "t_max": 20.0, "deplete": False},
        {"name": "qs_300sites_jsr", "kind": "qs", "sites": 300, "t_max": 5.0, "deplete": True},
        # held-out evaluation of the committed ensemble (1024 geometries, about 55 k mouths)
        {"name": "predict_55k", "kind": "predict", "rows": 55003},
        # one epoch of the five-member ensemble at the training script's batch size
        {"name": "train_16k", "kind": "train", "rows": 16384, "batch": 1024},
    ]


def draw(rng_):
    """One more case: sizes over the ranges that the listed ones span, most of
    them over their logarithm."""
    def logint(a, b):
        return int(round(math.exp(rng_.uniform(math.log(a), math.log(b)))))

    kind = rng_.choice(["step"] * 5 + ["protocol", "coupled", "pool2d", "solve", "qs", "qs", "predict", "predict", "train"])
    if kind == "step":
        geometry = rng_.choice(["single", "batch", "batch"])
        lo, hi, warm = (48, 72, 300) if geometry == "single" else (74, 96, 0)
        c = {"warm": warm, "kind": kind, "geometry": geometry, "nx": rng_.randint(lo, hi), "ny": rng_.randint(lo, hi),
             "nz": rng_.choice([4, 5, 5, 5, 6]), "precision": rng_.choice([64, 64, 32]), "pool": rng_.random() < 0.3}
        c["sites"] = logint(1, 3000)
        c["steps"] = logint(10, 1000)
        # no more node-steps than half of the largest listed case
        limit = 0.5 * 4096 * 81 * 81 * 5 * 100
        c["steps"] = max(2, min(c["steps"], int(limit / (c["sites"] * c["nx"] * c["ny"] * c["nz"]))))
        c["fields"] = c["sites"] <= 40
        return c
    if kind == "protocol":
        return {"kind": kind, "sites": logint(1, 400), "nx": rng_.randint(48, 72), "ny": rng_.randint(48, 72),
                "nz": rng_.choice([4, 5, 5]), "warm": 300, "steps": rng_.randint(3, 30)}
    if kind == "coupled":
        return {"kind": kind, "sites": logint(4, 400), "steps": 50 * rng_.randint(1, 4)}
    if kind == "pool2d":
        return {"kind": kind, "sites": logint(1, 400), "steps": logint(50, 500)}
    if kind == "solve":
        return {"kind": kind, "sites": logint(1, 100), "extent": 4 * rng_.randint(74, 90), "steps": logint(500, 3000)}
    if kind == "qs":
        return {"kind": kind, "sites": logint(16, 4096), "t_max": round(rng_.uniform(0.5, 20.0), 2),
                "deplete": rng_.random() < 0.5}
    if kind == "predict":
        return {"kind": kind, "rows": logint(1, 200000)}
    return {"kind": "train", "rows": logint(2000, 24000), "batch": rng_.choice([512, 1024, 2048, rng_.randint(400, 4096)])}


# ---- inputs -----------------------------------------------------------------


def _package_seed(seed):
    g = np.random.default_rng([7, seed])
    return tuple(int(v) for v in g.integers(1, M2 - 1, 6))


def _clusters(sites, seed, **kw):
    """batched_dyads with one site of the largest cluster (100 RyRs), so that
    the arrays of every seed have the same shape, the RyR nearest the rim open
    at the start (its calcium reaches the rim within a call)."""
    sp = workloads.batched_dyads(sites, seed=_package_seed(seed), geometry_seed=seed, **kw)
    sp.sites[0] = workloads.batched_dyads(1, geometry_seed=seed, n_min=100, n_max=100, **kw).sites[0]
    c = (sp.nx - 1) * sp.dx / 2.0
    sp.init_channel = [int(np.argmax([max(abs(p[0] - c), abs(p[1] - c)) for p in site])) for site in sp.sites]
    return sp


def _spec(c, seed):
    """The site batch of a step or protocol case."""
    p = abi.CASIM_FP32 if c.get("precision") == 32 else abi.CASIM_FP64
    if c.get("geometry", "single") == "batch":
        # the clusters of batched_dyads, centred on a square that holds them on either grid
        sp = _clusters(c["sites"], seed, precision=p, extent_nm=4.0 * (min(c["nx"], c["ny"]) - 1))
    else:
        sp = workloads.single_dyad(c["sites"], seed=_package_seed(seed), precision=p)
        g = np.random.default_rng([11, seed])
        sp.init_channel = [int(v) for v in g.integers(0, 25, c["sites"])]
        # the 5 x 5 lattice keeps its pitch, centred on the grid at hand
        cx, cy = 2.0 * (c["nx"] - 1), 2.0 * (c["ny"] - 1)
        lattice = [(cx + 31.0 * i, cy + 31.0 * j, 0) for i in range(-2, 3) for j in range(-2, 3)]
        sp.sites = [list(lattice) for _ in range(c["sites"])]
    return dataclasses.replace(sp, nx=c["nx"], ny=c["ny"], nz=c["nz"], z=4.0 * (c["nz"] - 1))


def _solve_inputs(c, seed):
    sp = _clusters(c["sites"], seed, extent_nm=float(c["extent"]))
    gen = np.random.default_rng([13, seed])
    return sp, surrogate.random_open_sets(sp, gen), gen.uniform(200.0, 1200.0, c["sites"])


def _features(net, rows, seed):
    """Feature rows spread as the ensemble's training rows are."""
    g = np.random.default_rng([17, seed])
    mean, std = net.norm[0], net.norm[1]
    return (mean + 0.5 * std * g.standard_normal((rows, net.n_in), dtype=np.float32)).astype(np.float32)


def _pool2d_spec(c, seed):
    with open(TEST_INPUT) as f:
        j = json.load(f)
    sp = config.from_json(j["Dyad"], n_sites=c["sites"], base_dir=os.path.dirname(TEST_INPUT),
                          seed=_package_seed(seed))
    g = np.random.default_rng([19, seed])
    sp.init_channel = [int(v) for v in g.integers(0, sp.max_channels(), c["sites"])]
    return sp, config.pools_from_json(j, sp), float(j["dt, ns"]) * 1e-6


def prepare(case, seed):
    c = case
    if c["kind"] == "solve":
        sp, open_sets, jsr = _solve_inputs(c, seed)
        return {"case": c, "spec": sp, "open": open_sets, "jsr": jsr}
    if c["kind"] == "qs":
        sp = _clusters(c["sites"], seed)
        net, lin = surrogate.load_model(WEIGHTS)
        pools = spark_compare.depleting_pool() if c["deplete"] else None
        qs = surrogate.QuasiStationarySites(sp, np.full(c["sites"], 1000.0), c["t_max"], net, pools=pools, lin=lin)
        return {"case": c, "qs": qs, "net": net}
    if c["kind"] == "predict":
        net, _ = surrogate.load_model(WEIGHTS)
        return {"case": c, "net": net, "x": _features(net, c["rows"], seed)}
    if c["kind"] == "train":
        old, _ = surrogate.load_model(WEIGHTS)
        x = _features(old, c["rows"], seed)
        y = np.log(old.predict(x)[0])  # targets of the kind that the ensemble learns
        net = mlp.MLP(57, width=256, depth=4, members=5, seed=seed % 100003 + 1)
        net.fit_normalization(x, y)
        net.set_data(x, y)
        return {"case": c, "net": net, "seed": seed % 1009}
    if c["kind"] == "coupled":
        sp = workloads.coupled_dyads(c["sites"], seed=_package_seed(seed))
        g = np.random.default_rng([23, seed])
        sp.init_channel = [int(v) for v in g.integers(0, 64, c["sites"])]
        dev = DyadHIP(sp)
        autotune.apply(dev, sp)
        dev.AttachPools(workloads.coupled_pools())
        dev.AttachCytosolBox(workloads.coupled_box(sp))
        dev.InitOpeningAll()
        dev.UpdatePools()
        return {"case": c, "dev": dev, "dt": sp.meta["dt_ms"]}
    if c["kind"] == "pool2d":
        sp, pools, dt = _pool2d_spec(c, seed)
        dev = DyadHIP(sp)
        dev.AttachPools(pools)
        dev.InitOpeningAll()
        dev.UpdatePools()
        return {"case": c, "dev": dev, "dt": dt}
    sp = _spec(c, seed)
    dev = DyadHIP(sp)
    autotune.apply(dev, sp)
    state = {"case": c, "dev": dev, "dt": workloads.DT_MS, "rim": sp.rim_arrays(), "jsr": sp.jsr_array([1000.0])}
    if c.get("pool"):
        dev.AttachPools(spark_compare.depleting_pool())
    dev.InitOpeningAll()
    if c.get("pool"):
        dev.UpdatePools(*state["rim"])
    else:
        dev.Update(*state["rim"], state["jsr"])
    if c.get("warm"):  # a run in progress
        dev.Step(state["dt"], c["warm"])
    return state


def run(state):
    c = state["case"]
    if c["kind"] == "solve":
        return {"mouths": surrogate.qs_solve(DyadHIP, state["spec"], state["open"], state["jsr"], c["steps"])}
    if c["kind"] == "qs":
        qs = state["qs"]
        qs.Reset()
        stats = qs.RunSimulation()
        now, low = qs.GetJsr()
        return {"stats": stats, "window": qs.GetWindowStats(), "states": qs.GetChannelsStates(), "jsr": now,
                "jsr_lowest": low}
    if c["kind"] == "predict":
        mean, spread, raw = state["net"].predict(state["x"])
        return {"mean": mean, "spread": spread, "raw": raw}
    if c["kind"] == "train":
        net = state["net"]
        loss = net.train(1, batch=c["batch"], lr=1e-3, seed=state["seed"])
        return {"loss": loss, "params": [net.params(e) for e in range(net.members)]}
    dev = state["dev"]
    if c["kind"] == "protocol":
        currents, effluxes = [], []
        for _ in range(c["steps"]):
            dev.RunRD(state["dt"])
            dev.RunMC(state["dt"])
            dev.Update(*state["rim"], state["jsr"])
            currents.append(dev.GetTotalSRCurrent())
            effluxes.append(dev.GetEffluxes())
        return {"currents": np.stack(currents), "effluxes": np.stack(effluxes), "mouths": dev.GetIonsNearChannels(),
                "states": dev.GetChannelsStates(), "rng": dev.GetRngStates().astype(np.int64)}
    dev.Step(state["dt"], c["steps"])
    out = {"mouths": dev.GetIonsNearChannels(), "states": dev.GetChannelsStates(),
           "rng": dev.GetRngStates().astype(np.int64), "current": dev.GetTotalSRCurrent(),
           "stats": dev.GetReleaseStats()}
    if c.get("pool") or c["kind"] != "step":
        out["jsr"], out["cytosol"], out["cytosol_bound"] = dev.GetPools()
    if c["kind"] == "coupled":
        return out
    if c.get("precision") == 32:
        # the values of an FP32 state, as they are held (its effluxes are differences of near-equal values and are
        # read from FP64 runs)
        out["mouths"], out["current"] = out["mouths"].astype(np.float32), out["current"].astype(np.float32)
        if c.get("pool"):
            out["jsr"] = out["jsr"].astype(np.float32)
    else:
        out["effluxes"] = dev.GetEffluxes()
    if c["kind"] == "pool2d" or c.get("fields"):
        fields = dev.GetConcentrations()
        out["fields"] = {k: v.astype(np.float32) for k, v in fields.items()} if c.get("precision") == 32 else fields
    return out


# ---- the work that cannot be left out ----------------------------------------


def _step_work(sites, nodes, interior, grid, face_nodes, diffusing, bound, steps, size, extra=0):
    """A state read once and written once, and the arithmetic of every step:
    14 operations per diffusing field and node (Laplacian, Euler step), 9 per
    bound field (free buffer, reaction, its sum)."""
    state = sites * (grid * nodes + face_nodes) * size
    return {"bytes": 2.0 * state + extra, "flops": float(steps) * sites * interior * (14 * diffusing + 9 * bound)}


def work(case):
    c = case
    if c["kind"] in ("step", "protocol", "solve"):
        nx, ny, nz = (c["extent"] // 4 + 1, c["extent"] // 4 + 1, 5) if c["kind"] == "solve" else (c["nx"], c["ny"], c["nz"])
        return _step_work(c["sites"], nx * ny * nz, (nx - 2) * (ny - 2) * nz, 3, 2 * nx * ny, 3, 2.4, c["steps"],
                          4 if c.get("precision") == 32 else 8)
    if c["kind"] == "coupled":
        w = _step_work(c["sites"], 201 * 201, 199 * 199, 4, 0, 3, 3, c["steps"], 8)
        box = _step_work(c["sites"], 51 ** 3, 49 * 49 * 50, 4, 0, 3, 3, c["steps"] // 50, 8)
        return {k: w[k] + box[k] for k in w}
    if c["kind"] == "pool2d":
        return _step_work(c["sites"], 31 * 41, 29 * 39, 6, 0, 6, 4, c["steps"], 8)
    weights = 57 * 256 + 3 * 256 * 256 + 256
    if c["kind"] == "predict":
        return {"bytes": c["rows"] * (57 + 2 + 5) * 4.0 + 5 * weights * 2.0, "flops": 2.0 * 5 * weights * c["rows"]}
    if c["kind"] == "train":
        rows = c["rows"] // min(c["batch"], c["rows"]) * min(c["batch"], c["rows"])
        return {"bytes": rows * 58 * 4.0 + 5 * weights * 4.0 * 6, "flops": 6.0 * 5 * weights * rows}
    # qs: about three events per site, each one an ensemble evaluation of its 54 mouths
    events = 3.0 * c["sites"]
    return {"bytes": events * 54 * 57 * 4.0 + 5 * weights * 2.0, "flops": events * 54 * 2.0 * 5 * weights}


# ---- 64-bit values ------------------------------------------------------------


class _Streams:
    """MRG32k3a streams of a batch of sites in exact integers."""

    def __init__(self, states):
        s = np.asarray(states, dtype=np.int64)
        self.s = [s[:, k].copy() for k in range(6)]

    def _u01(self, at):
        s = [v[at] for v in self.s]
        p1 = (1403580 * s[1] - 810728 * s[0]) % M1
        p2 = (527612 * s[5] - 1370589 * s[3]) % M2
        for k, v in enumerate((s[1], s[2], p1, s[4], s[5], p2)):
            self.s[k][at] = v
        d = p1 - p2
        return np.where(p1 > p2, d, d + M1).astype(np.float64) * rng.NORM

    def draw(self, at):
        u = self._u01(at)
        u = u + self._u01(at) * rng.FACT
        return np.where(u < 1.0, u, u - 1.0)


class _Exact:
    """The plain step of a batch in 64 bits (torch on whole fields, numpy for
    the channels): constant rim, jSR constant or SRPool's pool."""

    def __init__(self, sp, jsr, pools=None, states=None, init=True):
        self.sp, self.pools = sp, pools
        S, M = sp.n_sites, sp.max_channels()
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.bound = sp.bound_fields()
        self.binit = sp.bound_init()
        shape = (S, sp.nx, sp.ny, sp.nz)
        self.C = torch.full(shape, sp.ions[0].c0, dtype=torch.float64, device=dev)
        zmask = torch.ones(sp.nz, dtype=torch.float64, device=dev)
        zmask[1:-1] = 0.0
        self.mask = [zmask if sp.buffers[u].faces_only else torch.ones_like(zmask) for _, u, *_ in self.bound]
        self.B = [torch.full(shape, float(b), dtype=torch.float64, device=dev) * m
                  for b, m in zip(self.binit, self.mask)]
        self.n = np.array([len(s) for s in sp.sites])
        self.valid = np.arange(M)[None, :] < self.n[:, None]
        gx = np.zeros((S, M), dtype=np.int64)
        gy = np.zeros((S, M), dtype=np.int64)
        for s, site in enumerate(sp.sites):
            xy = np.array([(p[0], p[1]) for p in site])
            gx[s, :len(site)] = ((xy[:, 0] + 0.5 * sp.dx) / sp.dx).astype(np.int64)
            gy[s, :len(site)] = ((xy[:, 1] + 0.5 * sp.dy) / sp.dy).astype(np.int64)
        flat = ((np.arange(S)[:, None] * sp.nx + gx) * sp.ny + gy) * sp.nz
        self.node = torch.from_numpy(flat).to(dev)
        self.hot = torch.from_numpy(flat[self.valid]).to(dev)
        self.st = np.where(self.valid, 0, -1).astype(np.int32) if states is None else np.asarray(states).copy()
        self.streams = _Streams(sp.rng_states)
        if init:
            every = np.arange(S)
            for i in range(M + 1):
                self.streams.draw(every[self.n + 1 > i])
            self.st[every, np.asarray(sp.init_channel)] = 1
        self.jsr = np.broadcast_to(np.asarray(jsr, dtype=np.float64), (S,)).copy()
        self.g = sp.channel_types[0].conductance[0]
        self.steps = 0
        n0 = (self.st == 1).sum(axis=1).astype(np.float64)
        self.stat = {"n": n0, "amp": n0.copy(), "ttp": np.zeros(S), "tte": np.zeros(S), "q": np.zeros(S)}
        self.update()

    def mouth(self, f):
        return f.reshape(-1)[self.node].cpu().numpy()

    def update(self):
        """Mouths, currents and site totals of the present state."""
        self.ca = self.mouth(self.C)
        self.J = np.where(self.valid, (self.st == 1) * (self.g * (self.jsr[:, None] - self.ca)), 0.0)
        self.total = self.J.sum(axis=1)

    def gate(self, dt):
        par = self.sp.channel_types[0].params
        x = self.ca * 1e-3
        opening = np.minimum(par["kopen0"] * x ** par["ncaopen"], par["kopenmax"]) * 1e-3
        closing = par["kclose0"] * x ** par["ncaclose"] * 1e-3
        thr = np.where(self.st == 1, closing, opening) * dt
        for i in range(self.st.shape[1]):
            at = np.nonzero(self.valid[:, i])[0]
            hit = at[self.streams.draw(at) < thr[at, i]]
            if len(hit):
                self.st[hit, i] ^= 1
                self.streams.draw(hit)
        self.steps += 1
        t, q = self.steps * dt, self.stat
        n = (self.st == 1).sum(axis=1).astype(np.float64)
        q["tte"] = np.where(n != q["n"], t, q["tte"])
        q["ttp"] = np.where(n > q["amp"], t, q["ttp"])
        q["amp"] = np.maximum(q["amp"], n)
        q["q"] = q["q"] + n * dt
        q["n"] = n

    def lap(self, f):
        sp, c = self.sp, f[:, 1:-1, 1:-1]
        out = (f[:, 2:, 1:-1] + f[:, :-2, 1:-1] - 2 * c) / sp.dx ** 2 + (f[:, 1:-1, 2:] + f[:, 1:-1, :-2] - 2 * c) / sp.dy ** 2
        up = torch.cat([c[..., 1:], c[..., -2:-1]], dim=-1)
        down = torch.cat([c[..., 1:2], c[..., :-1]], dim=-1)
        return out + (up + down - 2 * c) / sp.dz ** 2

    def diffuse(self, dt):
        """One explicit step of every field with the currents of update()."""
        sp = self.sp
        inner = (slice(None), slice(1, -1), slice(1, -1))
        c = self.C[inner]
        evo = sp.ions[0].D * self.lap(self.C)
        new = []
        for (_, u, D, kon, koff), m, f in zip(self.bound, self.mask, self.B):
            b = f[inner]
            r = (koff * b - kon * c * (sp.buffers[u].total - b)) * m
            evo += r
            new.append(b + ((D * self.lap(f) if D > 0 else 0.0) - r) * dt)
        J = torch.zeros(self.C.numel(), dtype=torch.float64, device=self.C.device)
        J[self.hot] = torch.from_numpy(self.J[self.valid]).to(self.C.device)
        evo += J.reshape(self.C.shape)[inner]
        self.C[inner] = c + evo * dt
        for f, v in zip(self.B, new):
            f[inner] = v

    def advance_pool(self, dt):
        p = self.pools
        volume = 0.5 * self.sp.dx * self.sp.dy * self.sp.dz
        beta = 1 + p.jsr_cq_sites[0] * p.jsr_k_cq[0] * p.jsr_cq_total / (p.jsr_k_cq[0] + self.jsr) ** 2
        refill = (p.nsr_c[0] - self.jsr) / p.jsr_tau_refill[0]
        return self.jsr + dt / beta * (refill - self.total * volume / p.jsr_volume)

    def step(self, dt, clamped=False):
        jsr = self.advance_pool(dt) if self.pools is not None else self.jsr
        if not clamped:
            self.gate(dt)
        self.diffuse(dt)
        self.jsr = jsr
        self.update()

    def mouths(self):
        rows = [self.ca] + [self.mouth(f) for f in self.B]
        rows += [self.sp.buffers[u].total - rows[1 + k] for k, (_, u, *_r) in enumerate(self.bound)]
        return np.where(self.valid[None], np.stack(rows), 0.0)

    def effluxes(self):
        sp = self.sp
        gm = 3.0 / (4 * math.pi * sp.radius ** 3)
        sx, sy = sp.dy * sp.dz / sp.dx, sp.dx * sp.dz / sp.dy
        out = np.zeros((sp.n_sites, 1 + len(self.B)))
        for k, (f, D) in enumerate(zip([self.C] + self.B, [sp.ions[0].D] + [t[2] for t in self.bound])):
            if D == 0.0:
                continue
            v = f[..., :-1]
            gx = sum(2 * v[:, a] - 1.5 * v[:, b] - 0.5 * v[:, e] for a, b, e in ((1, 0, 2), (-2, -1, -3)))
            gy = sum(2 * v[:, :, a] - 1.5 * v[:, :, b] - 0.5 * v[:, :, e] for a, b, e in ((1, 0, 2), (-2, -1, -3)))
            out[:, k] = (D * gm * (sx * gx[:, 1:-1].sum(dim=(1, 2)) + sy * gy.sum(dim=(1, 2)))).cpu().numpy()
        return out

    def rng(self):
        return np.stack(self.streams.s, axis=1)

    def release(self):
        q = self.stat
        ratio = np.divide(q["q"], q["tte"], out=np.zeros_like(q["q"]), where=q["tte"] > 0)
        return np.stack([q["amp"], q["ttp"], q["tte"], q["q"], ratio, q["n"]], axis=1)


def _exact_predict(c, seed):
    net, _ = surrogate.load_model(WEIGHTS)
    x = _features(net, c["rows"], seed).astype(np.float64)
    z = np.load(WEIGHTS, allow_pickle=False)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    h0 = torch.from_numpy((x - z["in_mean"].astype(np.float64)) / z["in_std"].astype(np.float64)).to(dev)
    raw = []
    for p in z["params"].astype(np.float64):
        p, h, at = torch.from_numpy(p).to(dev), h0, 0
        for l, (a, b) in enumerate([(57, 256)] + [(256, 256)] * 3 + [(256, 1)]):
            h = h @ p[at:at + a * b].reshape(a, b) + p[at + a * b:at + a * b + b]
            at += a * b + b
            if l < 4:
                h = h * torch.sigmoid(h)
        raw.append(h[:, 0] * float(z["out"][1]) + float(z["out"][0]))
    raw = torch.stack(raw)
    v = torch.exp(raw)
    mean = v.mean(dim=0)
    return {"mean": mean.cpu().numpy(), "spread": (v.std(dim=0, unbiased=False) / mean).cpu().numpy(),
            "raw": raw.cpu().numpy()}


def exact(case, seed):
    """The first pass's outputs in 64 bits.  None where it has no short form:
    the coupled and cytosol-pool steps (FP64 throughout), the event-driven
    sites (whose events follow the BF16 ensemble's own values) and training."""
    c = case
    if c["kind"] == "predict":
        return _exact_predict(c, seed)
    if c["kind"] == "solve":
        sp, open_sets, jsr = _solve_inputs(c, seed)
        e = _Exact(sp, jsr, states=open_sets, init=False)
        for _ in range(c["steps"]):
            e.step(workloads.DT_MS, clamped=True)
        return {"mouths": e.mouths()[0]}
    if c["kind"] not in ("step", "protocol"):
        return None
    sp, dt = _spec(c, seed), workloads.DT_MS
    pools = spark_compare.depleting_pool() if c.get("pool") else None
    e = _Exact(sp, 1000.0, pools)
    for _ in range(c.get("warm", 0)):
        e.step(dt)
    currents, effluxes = [], []
    for _ in range(c["steps"]):
        e.step(dt)
        if c["kind"] == "protocol":
            currents.append(e.total[None].copy())
            effluxes.append(e.effluxes())
    if c["kind"] == "protocol":
        return {"currents": np.stack(currents), "effluxes": np.stack(effluxes), "mouths": e.mouths(), "states": e.st,
                "rng": e.rng()}
    out = {"mouths": e.mouths(), "states": e.st, "rng": e.rng(), "current": e.total[None], "stats": e.release()}
    if pools is not None:
        out["jsr"], out["cytosol"], out["cytosol_bound"] = e.jsr[None], None, None
    if c.get("precision") != 32:
        out["effluxes"] = e.effluxes()
    if c.get("fields"):
        names = sp.field_names()
        out["fields"] = {k: f.cpu().numpy() for k, f in zip(names, [e.C] + e.B)}
    return out
