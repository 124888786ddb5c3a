"""Workloads of the energy path, as a user's program runs them through the
Python API: one trial move at a time on a device-resident box, the strategy
calls, the full energy, coordinate frames and NPT rescales, whole Monte Carlo
runs of one box and of many boxes advanced together, and the job server.

Boxes come from the package's own generators (rigid TIP3P water at 0.95-1.05
g/cm3, rc 9 A; 16-site bicyclic molecules at 1.10 g/cm3, rc 12 A; 3:2 mixtures
of water and methanol, rc 11 A): the kinds, densities, cutoffs and sizes
(64-20,000 molecules) of the benchmark and of the tests.  A case is a family
of calls and its sizes:

  move      trial_move on one box, `calls` of them (a host-driven loop)
  strategy  molecule_energy, set_molecule, molecule_energy, and set_molecule
            back when the move is refused: the calls a metrosim-style loop makes
  energy    system_energy (start-up of a run, or a point of an analysis)
  frame     upload of a new configuration, then system_energy
  volume    volume_scale, system_energy, and volume_scale back: an NPT move
            driven from the host
  run       `boxes` boxes advanced `ticks` times by `sweeps` moves each, then
            every box's statistics and coordinates
  serve     `boxes` jobs of `sweeps` moves on average submitted to a running
            server, until the last one is done
"""
import math

import numpy as np
import torch

import mcgpu_amd as m

P_ATM = 1.4584e-5  # kcal/mol/A^3
KIND = {"water": m.WATER, "bicyclic": m.BICYCLIC, "mixture": m.MIXTURE}
CUTOFF = {"water": 9.0, "bicyclic": 12.0, "mixture": 11.0, "stream": 9.0}
LEN = {"water": 3.0, "bicyclic": 16.0, "mixture": 4.2, "stream": 3.0}
# molecules per A^3; a "stream" is water boxes with every fourth a bicyclic
# one of at most 600 molecules (its work is counted as water's)
DENSITY = {"water": 0.0334, "bicyclic": 0.00565, "mixture": 20000 / 96.45 ** 3, "stream": 0.0334}
NEIGHBOR = {"brute": m.NEIGHBOR_BRUTE, "cell": m.NEIGHBOR_CELL, "verlet": m.NEIGHBOR_VERLET}


# ------------------------------------------------------------------ cases


def _case(name, family, kind, n, fp64, neighbor, calls=1, boxes=1, n_low=0, sweeps=0, ticks=0,
          npt=False):
    c = dict(family=family, kind=kind, n=n, n_low=n_low or n, fp64=fp64, neighbor=neighbor,
             calls=calls, boxes=boxes, sweeps=sweeps, ticks=ticks, npt=npt)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest call: one move of the 256-water box, all latency
        _case("move_water256", "move", "water", 256, True, "brute"),
        # a host-driven loop on a large box with Verlet lists
        _case("moves_mixture6001_verlet", "move", "mixture", 6001, True, "verlet", calls=24),
        # a reference-shaped strategy loop with cell lists and FP32 pair terms
        _case("strategy_bicyclic1055_mixed", "strategy", "bicyclic", 1055, False, "cell", calls=8),
        # start-up energy of a small box without neighbour structure
        _case("energy_water700_mixed", "energy", "water", 700, False, "brute"),
        # start-up energy of the largest box
        _case("energy_mixture20000", "energy", "mixture", 20000, True, "cell"),
        # re-evaluation of stored configurations, an odd size
        _case("frame_bicyclic1733", "frame", "bicyclic", 1733, True, "cell"),
        # one NPT volume proposal from the host, refused
        _case("volume_water4096_mixed", "volume", "water", 4096, False, "cell"),
        # an ordinary run: one small box, all pairs
        _case("run_water256", "run", "water", 256, True, "brute", sweeps=2000, ticks=1),
        # one large box of large molecules, cell lists, FP32 pair terms
        _case("run_bicyclic4000_mixed", "run", "bicyclic", 4000, False, "cell", sweeps=1000, ticks=1),
        # many water boxes advanced together
        _case("run_512_water_mixed", "run", "water", 4096, False, "policy", boxes=512, n_low=64,
              sweeps=2000, ticks=1),
        # constant-pressure boxes of mixed molecules, a volume move per 500 moves
        _case("run_48_npt_mixture", "run", "mixture", 3000, True, "policy", boxes=48, n_low=200,
              sweeps=500, ticks=4, npt=True),
        # the job server on a burst of NVT and NPT jobs of both precisions
        _case("serve_160_jobs", "serve", "stream", 4096, True, "policy", boxes=160, n_low=128,
              sweeps=4000, npt=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(["move", "strategy", "energy", "frame", "volume", "run", "run", "run", "serve"])
    kind = rng.choice(["water", "bicyclic", "mixture"])
    top = {"water": 16384, "bicyclic": 4000, "mixture": 20000}[kind]
    fp64 = rng.random() < 0.5
    if family == "serve":
        n = _log_int(rng, 300, 1500 if kind == "bicyclic" else 4096)
        return _case(None, "serve", "stream" if kind == "water" else kind, n, True, "policy", boxes=_log_int(rng, 8, 120),
                     n_low=128, sweeps=_log_int(rng, 1000, 4000), npt=rng.random() < 0.7)
    if family == "run":
        boxes = 1 if rng.random() < 0.4 else _log_int(rng, 2, 300)
        top = min(top, 20000 if boxes == 1 else 4096)
        n = _log_int(rng, 100, max(100, min(top, 150000 // boxes)))
        if kind == "bicyclic":
            n = min(n, max(100, 20000 // boxes))
        npt = rng.random() < 0.3
        return _case(None, "run", kind, n, fp64, rng.choice(["policy", "policy", "brute", "cell"])
                     if n <= 4096 else "cell", boxes=boxes, n_low=rng.choice([n, max(64, n // 16)]),
                     sweeps=500 if npt else _log_int(rng, 200, 2000), ticks=2 if npt else 1, npt=npt)
    n = _log_int(rng, 64, top)
    near = rng.choice(["cell", "cell", "brute"]) if family in ("energy", "frame", "volume") else \
        rng.choice(["brute", "cell", "verlet"])
    if n > 6000 and near == "brute":
        near = "cell"
    calls = _log_int(rng, 1, 32) if family in ("move", "strategy") else 1
    return _case(None, family, kind, n, fp64, near, calls=calls)


# ----------------------------------------------------------------- inputs


def _box(kind, n, seed, rng):
    """One start configuration; water boxes vary in density and temperature."""
    kw = dict(cutoff=CUTOFF[kind], temperature=298.0, seed=seed, mc_seed=1 + seed % 2147483646)
    if kind == "water":
        kw.update(density=float(rng.uniform(0.95, 1.05)), temperature=float(rng.uniform(250, 400)))
    elif kind == "bicyclic":
        kw.update(density=1.10)
    else:
        kw.update(edge=(n / DENSITY["mixture"]) ** (1.0 / 3.0), n_second=(2 * n) // 5)
    return m.HostBox.generate(KIND[kind], n, **kw)


def _boxes(case, seed):
    """The case's boxes: sizes spread over the logarithm of [n_low, n] (the
    same for every seed), the first one n.  Past 48 boxes the configurations repeat (as one start file serves many
    runs), each with a generator seed of its own."""
    rng = np.random.default_rng([seed, 77])
    out = []
    for k in range(min(case["boxes"], 48)):
        at = 1.0 - (k * 0.6180339887498949) % 1.0  # 1 for the first, then evenly spread
        n = int(round(case["n_low"] * (case["n"] / case["n_low"]) ** at))
        kind = case["kind"]
        if kind == "stream":
            kind = "bicyclic" if k % 4 == 3 else "water"
            n = min(n, 600) if kind == "bicyclic" else n
        out.append(_box(kind, n, int(rng.integers(1, 1 << 40)), rng))
    return [out[k % len(out)] for k in range(case["boxes"])]


def _neighbor(case, box):
    """Cell lists once they shrink the scan (at least 4 cells per edge and
    1,000 molecules), else every molecule."""
    if case["neighbor"] != "policy":
        return NEIGHBOR[case["neighbor"]]
    d = box.desc()
    return m.NEIGHBOR_CELL if min(d.box) >= 4 * d.cutoff and d.n_molecules >= 1000 else m.NEIGHBOR_BRUTE


def _proposals(a, calls, seed):
    """Rigid trial moves of `calls` distinct molecules where the box has that
    many: a rotation of up to 15 degrees per axis about the first primary and
    a shift of up to 0.15 A, the first primary kept in the box."""
    rng = np.random.default_rng([seed, 99])
    xyz = np.stack([a["x"], a["y"], a["z"]])
    mols = rng.permutation(len(a["mol_start"]))
    out = []
    for k in range(calls):
        i = int(mols[k % len(mols)])
        s, l = int(a["mol_start"][i]), int(a["mol_len"][i])
        p = int(a["primary_index"][a["mol_pidx_start"][i]]) - s
        new = xyz[:, s:s + l].copy()
        c = new[:, p:p + 1].copy()
        for ax, t in enumerate(np.deg2rad(rng.uniform(-15, 15, 3))):
            r = np.eye(3)
            u, v = (ax + 1) % 3, (ax + 2) % 3
            r[u, u] = r[v, v] = math.cos(t)
            r[u, v], r[v, u] = -math.sin(t), math.sin(t)
            new = r @ (new - c) + c
        new += rng.uniform(-0.15, 0.15, (3, 1))
        for d in range(3):
            new[d] += a["box"][d] * ((new[d, p] < 0) * 1.0 - (new[d, p] > a["box"][d]) * 1.0)
        out.append((i, np.ascontiguousarray(new.reshape(-1)), float(rng.random()),
                    np.ascontiguousarray(xyz[:, s:s + l].reshape(-1))))
    return out


def _frame(a, seed):
    """Another configuration of the box: every molecule shifted by up to 0.05 A."""
    rng = np.random.default_rng([seed, 55])
    rep = np.repeat(rng.uniform(-0.05, 0.05, (3, len(a["mol_len"]))), a["mol_len"], axis=1)
    return [np.ascontiguousarray(a[k] + rep[d]) for d, k in enumerate("xyz")]


VOLUME_FACTOR = 1.0037


def _job(case, k, box, rng):
    """Parameters of one run: every second job of an NPT case is NPT in a
    server (all of them in a plain run), and precisions alternate there."""
    serve = case["family"] == "serve"
    kw = dict(precision=m.FP64 if (case["fp64"] if not serve else k % 2 == 0) else m.MIXED,
              neighbor=_neighbor(case, box), seed=int(rng.integers(1, 2 ** 31 - 1)))
    if case["npt"] and (not serve or k % 4 < 2):
        kw.update(ensemble=m.NPT, volume_interval=500, pressure=P_ATM, max_volume_delta=0.01)
    if serve:
        kw["steps"] = int(round(case["sweeps"] * math.exp(rng.uniform(-0.7, 0.7))))
    else:
        kw["steps"] = 1 << 40  # the program stops the run, not the step count
    return kw


def prepare(case, seed):
    boxes = _boxes(case, seed)
    s = dict(case=case, boxes=boxes)
    rng = np.random.default_rng([seed, 33])
    if case["family"] == "run":
        b = s["batch"] = m.Batch(case["boxes"], 3 << 30)
        s["slots"] = [b.add(box, **_job(case, k, box, rng)) for k, box in enumerate(boxes)]
        for slot in s["slots"]:
            b.stats(slot)
    elif case["family"] == "serve":
        s["jobs"] = [(box, _job(case, k, box, rng)) for k, box in enumerate(boxes)]
        s["server"] = m.Server(case["boxes"], 2000, 3 << 30, tick_budget_us=2000.0)
        s["server"].start()
    else:
        box = boxes[0]
        db = s["box"] = m.DeviceBox(box, m.FP64 if case["fp64"] else m.MIXED)
        kind = NEIGHBOR[case["neighbor"]]
        if kind != m.NEIGHBOR_BRUTE:
            db.neighbor(kind, 0.2875 * box.desc().cutoff)
        a = box.arrays()
        if case["family"] in ("move", "strategy"):
            s["proposals"] = _proposals(a, case["calls"], seed)
            s["kT"] = a["kT"]
        if case["family"] == "frame":
            s["frame"] = _frame(a, seed)
    return s


# ------------------------------------------------------------------- runs


def _moves(s):
    db = s["box"]
    res = [db.trial_move(i, xyz, u) for i, xyz, u, _ in s["proposals"]]
    return dict(old=np.array([r.old_energy for r in res]), new=np.array([r.new_energy for r in res]),
                delta=np.array([r.delta for r in res]), accepted=np.array([r.accepted for r in res]))


def _strategy(s):
    db, old, new, acc = s["box"], [], [], []
    for i, xyz, u, back in s["proposals"]:
        old.append(db.molecule_energy(i))
        db.set_molecule(i, xyz)
        new.append(db.molecule_energy(i))
        de = new[-1] - old[-1]
        acc.append(int(de < 0 or math.exp(-min(de / s["kT"], 700.0)) >= u))
        if not acc[-1]:
            db.set_molecule(i, back)
    return dict(old=np.array(old), new=np.array(new), accepted=np.array(acc))


def _stats(b, slots):
    st = [b.stats(k) for k in slots]
    return dict(energy=np.array([x.energy for x in st]),
                start_energy=np.array([x.start_energy for x in st]),
                box=np.array([list(x.box) for x in st]),
                steps=np.array([x.steps_done for x in st]),
                accepted=np.array([x.accepted for x in st]),
                volume_moves=np.array([x.volume_moves for x in st]),
                volume_accepted=np.array([x.volume_accepted for x in st]))


def run(s):
    case = s["case"]
    family = case["family"]
    if family == "move":
        return _moves(s)
    if family == "strategy":
        return _strategy(s)
    db = s.get("box")
    if family == "energy":
        return dict(energy=db.system_energy(), pairs=db.system_pairs())
    if family == "frame":
        db.upload(*s["frame"])
        return dict(energy=db.system_energy(), pairs=db.system_pairs())
    if family == "volume":
        db.volume_scale(VOLUME_FACTOR)
        out = dict(energy=db.system_energy(), pairs=db.system_pairs(), size=db.size())
        db.volume_scale(1.0 / VOLUME_FACTOR)
        return out
    if family == "run":
        b = s["batch"]
        for _ in range(case["ticks"]):
            b.run(case["sweeps"])
        out = _stats(b, s["slots"])
        xyz = [b.download(k) for k in s["slots"]]
        for d, k in enumerate("xyz"):
            out[k] = np.concatenate([p[d] for p in xyz])
        return out
    srv = s["server"]
    ids = [srv.submit(box, **kw) for box, kw in s["jobs"]]
    srv.wait()
    res = [srv.poll(i) for i in ids]
    return dict(energy=np.array([r.final_energy for r in res]),
                start_energy=np.array([r.start_energy for r in res]),
                steps=np.array([r.steps for r in res]),
                accepted=np.array([r.accepted for r in res]),
                status=np.array([r.status for r in res]))


# ------------------------------------------------------------------- work

# FP64 operations of one site pair: displacement 3, r^2 5, 1/r about 8, LJ and
# Coulomb 9, sum 1 (the wrap is not counted)
PAIR_FLOPS = 26


def _pairs_per_position(kind, n, rc):
    """Mean site pairs of one molecule at one position."""
    hits = min(n - 1.0, 4.18879 * rc ** 3 * DENSITY[kind])
    return hits * LEN[kind] ** 2


def work(case):
    kind, n = case["kind"], case["n"]
    rc = min(CUTOFF[kind], 0.5 * (n / DENSITY[kind]) ** (1.0 / 3.0))
    per = _pairs_per_position(kind, n, rc)
    site_bytes = 24.0 * n * LEN[kind]
    f = case["family"]
    if f in ("move", "strategy"):
        # the in-range molecules' sites and the primaries tested for range
        cand = float(n) if case["neighbor"] == "brute" else min(n, 27.0 * rc ** 3 * DENSITY[kind])
        one = 24.0 * cand + 24.0 * (per / LEN[kind] + 2 * LEN[kind])
        return dict(bytes=case["calls"] * one, flops=case["calls"] * (2 * per * PAIR_FLOPS + 16.0 * cand))
    if f in ("energy", "frame", "volume"):
        return dict(bytes=site_bytes * {"energy": 1, "frame": 3, "volume": 5}[f],
                    flops=0.5 * n * per * PAIR_FLOPS)
    # runs: each box read and written once; mean size of a log-uniform range
    lo, hi = case["n_low"], n
    mean_n = n if hi <= lo else (hi - lo) / math.log(hi / lo)
    per = _pairs_per_position(kind, mean_n, rc)
    moves = case["boxes"] * case["sweeps"] * max(1, case["ticks"])
    return dict(bytes=2 * 24.0 * case["boxes"] * mean_n * LEN[kind], flops=moves * 2 * per * PAIR_FLOPS)


# ------------------------------------------------------------------ exact


def _wrap(d, L):
    return d + L * (d < -0.5 * L).to(d.dtype) - L * (d > 0.5 * L).to(d.dtype)


class _Exact:
    """One box in 64-bit torch: every pair summed directly."""

    def __init__(self, a):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        t = lambda v, dt=torch.float64: torch.as_tensor(np.asarray(v), dtype=dt, device=dev)
        self.a, self.dev = a, dev
        self.X = t(np.stack([a["x"], a["y"], a["z"]], 1))
        self.L, self.rc2, self.kT = t(a["box"]), float(a["cutoff"]) ** 2, float(a["kT"])
        real = (a["sigma"] >= 0) & (a["epsilon"] >= 0)
        self.sig, self.eps = t(np.where(real, a["sigma"], 0.0)), t(np.where(real, a["epsilon"], 0.0))
        self.q = t(np.where(real, a["charge"], 0.0))
        self.start, self.len = a["mol_start"].astype(np.int64), a["mol_len"].astype(np.int64)
        self.prim = a["primary_index"][a["mol_pidx_start"]].astype(np.int64)
        self.primt = t(self.prim, torch.int64)
        self.mol_of = t(np.repeat(np.arange(len(self.len)), self.len), torch.int64)
        m_len = int(self.len.max())
        pad = np.minimum(self.start[:, None] + np.arange(m_len), len(a["x"]) - 1)
        self.pad = t(pad, torch.int64)
        self.has = t(np.arange(m_len) < self.len[:, None], torch.bool)

    def _pair(self, r2, ia, ib):
        s2 = self.sig[ia] * self.sig[ib] / r2
        s6 = s2 * s2 * s2
        e = 4.0 * torch.sqrt(self.eps[ia] * self.eps[ib]) * (s6 * s6 - s6)
        return e + 332.06 * self.q[ia] * self.q[ib] / torch.sqrt(r2)

    def molecule(self, i, xyz):
        """Energy of molecule i at xyz [len, 3] with every other molecule."""
        s, l = int(self.start[i]), int(self.len[i])
        d = _wrap(self.X[self.primt] - xyz[int(self.prim[i]) - s], self.L)
        near = (d * d).sum(1) <= self.rc2
        near[i] = False
        b = torch.nonzero(near[self.mol_of])[:, 0]
        d = _wrap(self.X[b][:, None] - xyz[None], self.L)
        ia = torch.arange(s, s + l, device=self.dev)
        return float(self._pair((d * d).sum(2), ia[None], b[:, None]).sum())

    def system(self):
        """(energy, site pairs) of the box."""
        n, e, pairs = len(self.len), 0.0, 0
        P = self.X[self.primt]
        chunk = max(1, 20_000_000 // n)
        for i0 in range(0, n, chunk):
            d = _wrap(P[None] - P[i0:i0 + chunk, None], self.L)
            ij = torch.nonzero((d * d).sum(2) <= self.rc2)
            i, j = ij[:, 0] + i0, ij[:, 1]
            i, j = i[j > i], j[j > i]
            step = max(1, 30_000_000 // self.pad.shape[1] ** 2)
            for k in range(0, len(i), step):
                ia, ib = self.pad[i[k:k + step]][:, :, None], self.pad[j[k:k + step]][:, None, :]
                ok = self.has[i[k:k + step]][:, :, None] & self.has[j[k:k + step]][:, None, :]
                d = _wrap(self.X[ib] - self.X[ia], self.L)
                r2 = torch.where(ok, (d * d).sum(3), torch.ones_like(d[..., 0]))
                e += float(torch.where(ok, self._pair(r2, ia, ib), torch.zeros_like(r2)).sum())
                pairs += int(ok.sum())
        return e, pairs

    def put(self, i, xyz):
        s = int(self.start[i])
        self.X[s:s + len(xyz)] = xyz

    def at(self, i):
        s = int(self.start[i])
        return self.X[s:s + int(self.len[i])].clone()

    def tail(self):
        """Tail correction of a box of one kind of molecule (pi to the nine
        digits of the reference's constant, which the run's correction keeps)."""
        l, rc3 = int(self.len[0]), self.rc2 ** 1.5
        s = self.sig[:l].cpu().numpy()
        p = self.eps[:l].cpu().numpy()
        s6 = (s[:, None] * s[None]) ** 3
        terms = 4.0 * np.sqrt(p[:, None] * p[None]) * s6 * (s6 / (9 * rc3 ** 3) - 1 / (3 * rc3))
        return 2 * 3.14159265 * len(self.len) ** 2 / float(self.L.prod()) * float(terms.sum())


class _Rand:
    """The C library's rand() (additive feedback, 31 words)."""

    def __init__(self, seed):
        r = [seed or 1]
        for _ in range(30):
            r.append((16807 * r[-1]) % 2147483647)
        self.r = r + r[:3]
        for i in range(34, 344):
            self.next()

    def next(self):
        v = (self.r[-31] + self.r[-3]) & 0xFFFFFFFF
        self.r = self.r[-33:] + [v]
        return v >> 1

    def real(self, a, b):
        return (b - a) * (self.next() / 2147483647) + a


def _chain(ex, a, seed, steps):
    """`steps` Monte Carlo moves; returns (sum of accepted changes, accepted)."""
    g, n, de_sum, acc = _Rand(seed), len(ex.len), 0.0, 0
    mt, mr, L = float(a["max_translate"]), float(a["max_rotate"]), [float(v) for v in a["box"]]
    for _ in range(steps):
        i = int(g.real(0, n))
        l = int(ex.len[i])
        v = int(g.real(0, l))
        shift = np.array([g.real(-mt, mt) for _ in range(3)])
        rot = [g.real(-mr, mr) * 3.14159265358979 / 180.0 for _ in range(3)]
        old = ex.at(i)
        x = old.cpu().numpy()
        c = x[v].copy()
        new = x - c
        for ax, t in enumerate(rot):
            u, w = (ax + 1) % 3, (ax + 2) % 3
            U, W = new[:, u].copy(), new[:, w].copy()
            new[:, u], new[:, w] = U * math.cos(t) + W * math.sin(t), W * math.cos(t) - U * math.sin(t)
        new = new + c
        new[v] = c
        new = new + shift
        p = int(ex.prim[i]) - int(ex.start[i])
        for d in range(3):
            new[:, d] += L[d] * ((new[p, d] < 0) * 1.0 - (new[p, d] > L[d]) * 1.0)
        new = torch.as_tensor(new, device=ex.dev)
        de = ex.molecule(i, new) - ex.molecule(i, old)
        if de < 0 or math.exp(-min(de / ex.kT, 700.0)) >= g.real(0.0, 1.0):
            ex.put(i, new)
            de_sum += de
            acc += 1
    return de_sum, acc


def _exact_moves(case, seed, ex, a):
    old, new, acc = [], [], []
    for i, xyz, u, _ in _proposals(a, case["calls"], seed):
        pos = torch.as_tensor(xyz.reshape(3, -1).T.copy(), device=ex.dev)
        old.append(ex.molecule(i, ex.at(i)))
        new.append(ex.molecule(i, pos))
        de = new[-1] - old[-1]
        acc.append(de < 0 or math.exp(-min(de / ex.kT, 700.0)) >= u)
        if acc[-1]:
            ex.put(i, pos)
    out = dict(old=np.array(old), new=np.array(new), accepted=None)
    return dict(out, delta=np.array(new) - np.array(old)) if case["family"] == "move" else out


def exact(case, seed):
    f = case["family"]
    if f == "serve" or case["boxes"] > 1 or case["npt"] or case["sweeps"] > 2000:
        return None
    box = _boxes(case, seed)[0]
    a = box.arrays()
    ex = _Exact(a)
    if f in ("move", "strategy"):
        return _exact_moves(case, seed, ex, a)
    if f == "frame":
        ex.X = torch.as_tensor(np.stack(_frame(a, seed), 1), device=ex.dev)
    if f == "volume":
        p = ex.X[ex.primt]
        ex.X = ex.X + (p * VOLUME_FACTOR - p)[ex.mol_of]
        ex.L = ex.L * VOLUME_FACTOR
    e, pairs = ex.system()
    if f == "volume":
        return dict(energy=e, pairs=None, size=ex.L.cpu().numpy())
    if f != "run":
        return dict(energy=e, pairs=None)
    if case["kind"] == "mixture":
        return None
    e += ex.tail()
    kw = _job(case, 0, box, np.random.default_rng([seed, 33]))
    de, _ = _chain(ex, a, kw["seed"], case["sweeps"] * case["ticks"])
    out = {k: None for k in ("steps", "accepted", "volume_moves", "volume_accepted")}
    X = ex.X.cpu().numpy()
    out.update(energy=np.array([e + de]), start_energy=np.array([e]), box=np.array([a["box"]]),
               x=X[:, 0], y=X[:, 1], z=X[:, 2])
    return out
