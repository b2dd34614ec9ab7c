"""The work this framework is used for, as cases that can be timed: strict
Metropolis sweeps of one lattice (the C ABI through spparks_amd.Lattice), the
same through an input script (the library API), a batch of replicas, and a
queue of solves through the serving loop.  A pass advances the state a
program holds and takes the results: Naccept and energy after every sweep,
and the whole state (spins and seeds) as a snapshot in host memory.

Kinds:
  lattice  one resident lattice: n sweeps, then a snapshot
  script   an input script's `run`, then the energy and the site array
  batch    a block of sweeps of every replica of an ensemble, then a snapshot of each
  serve    a queue of solves, served to the last
"""
import math

import numpy as np
import torch

from spparks_amd import hip, workloads
from spparks_amd.batch import Batch, replica_bytes, replica_desc, serve
from spparks_amd.spparks import spparks

NEIGHBOURS = {"sq/4n": 4, "sq/8n": 8, "sc/6n": 6, "sc/26n": 26}
MIX = workloads.ENSEMBLE_SEED   # fixes an ensemble's or queue's sizes, Q and kT; a pass's seed fixes the draws
EVENT_OPS = 20                  # integer operations of a site event beside its comparisons


def lattice(name, app, style, nx, ny, nz, q, kt, sweeps):
    return {"name": name, "kind": "lattice", "app": app, "style": style, "nx": nx, "ny": ny, "nz": nz, "q": q,
            "kT": kt, "sweeps": sweeps}


def listed():
    return [
        # a program that steps a small 2d Ising model and looks after every
        # sweep: launches and latency only
        lattice("ising-sq4n-64-step", "ising", "sq/4n", 64, 64, 1, 2, 2.269, 1),
        # the small grain-growth script, run as a script: 100 sweeps with
        # stats after every one
        {"name": "script-potts-sq8n-128", "kind": "script", "app": "potts", "style": "sq/8n", "nx": 128, "ny": 128,
         "nz": 1, "q": 100, "kT": 0.5, "time": 1.0},
        # a mid-sized critical Ising model, edges no power of two
        lattice("ising-sq4n-1000", "ising", "sq/4n", 1000, 1000, 1, 2, 2.269, 200),
        # the large critical Ising model
        lattice("ising-sq4n-4096", "ising", "sq/4n", 4096, 4096, 1, 2, 2.269, 1000),
        # the same model with the single-flip rule on a ragged box
        lattice("ising-single-sq4n-3000x2006", "ising/single", "sq/4n", 3000, 2006, 1, 2, 2.269, 200),
        # 2d grain growth on a large ragged box
        lattice("potts-sq8n-1500x1002", "potts", "sq/8n", 1500, 1002, 1, 100, 0.5, 100),
        # 3d Potts with few states and near neighbours, ragged
        lattice("potts-sc6n-150x130x110", "potts", "sc/6n", 150, 130, 110, 50, 0.8, 100),
        # 3d grain growth, small and with more states than 16 bits hold
        lattice("potts-sc26n-64-q100000", "potts", "sc/26n", 64, 64, 64, 100000, 0.5, 50),
        # 3d grain growth, large
        lattice("potts-sc26n-256", "potts", "sc/26n", 256, 256, 256, 10000, 0.5, 200),
        # the same with proposals from the neighbours
        lattice("potts-neigh-sc26n-256", "potts/neigh", "sc/26n", 256, 256, 256, 10000, 0.5, 50),
        # an ensemble of mixed 2d Ising and 3d Potts replicas
        {"name": "ensemble-64", "kind": "batch", "ising": 32, "potts": 32, "mix": MIX, "sweeps": 100},
        # a queue of 3d grain-growth solves
        {"name": "serving-24", "kind": "serve", "requests": 24, "mix": MIX + 5, "live": 64},
    ]


def _even(x):
    return max(2, 2 * round(x / 2))


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["lattice"] * 10 + ["script", "batch", "serve"])
    if kind == "batch":
        return {"kind": kind, "ising": rng.randint(2, 32), "potts": rng.randint(2, 32), "mix": rng.randint(1, 10**6),
                "sweeps": rng.randint(5, 100)}
    if kind == "serve":
        c = {"kind": kind, "requests": rng.randint(4, 20), "mix": rng.randint(1, 10**6), "live": rng.randint(16, 64)}
        while sum(n * sweeps for _, _, n, _, sweeps in _parts(c)) > 6e9:   # about half of the listed queue
            c["requests"] -= 1
        return c
    if kind == "script":
        return {"kind": kind, "app": "potts", "style": "sq/8n", "nx": _even(_log(rng, 32, 512)),
                "ny": _even(_log(rng, 32, 512)), "nz": 1, "q": round(_log(rng, 3, 200)),
                "kT": round(rng.uniform(0.2, 1.0), 3), "time": 1.0}
    app = rng.choice(["ising", "ising", "ising/single", "potts", "potts", "potts", "potts", "potts/neigh",
                      "potts/neighonly"])
    if app.startswith("ising"):
        style, lo, hi, q, kt = "sq/4n", 16, 4096, 2, rng.uniform(1.5, 3.5)
    else:
        style = rng.choice(["sq/8n", "sq/4n", "sc/6n", "sc/26n", "sc/26n", "sc/26n"])
        lo, hi = (16, 2048) if style.startswith("sq") else (8, 224)
        q, kt = round(_log(rng, 3, 1e6 if style == "sc/26n" else 1000)), rng.uniform(0.2, 1.0)
    nx, ny = _even(_log(rng, lo, hi)), _even(_log(rng, lo, hi))
    nz = 1 if style.startswith("sq") else _even(_log(rng, lo, hi))
    most = (4e8 if "neigh" in app else 2e9) / (nx * ny * nz)
    sweeps = max(1, min(round(_log(rng, 1, 200)), int(most)))
    c = lattice("", app, style, nx, ny, nz, q, round(kt, 3), sweeps)
    del c["name"]
    return c


# ------------------------------------------------------------------ states
def _start(seed):
    """(generator seed of `set site range`, base of the site seeds)."""
    g = np.random.default_rng(seed)
    return int(g.integers(1, 2**31 - 1)), float(g.random())


def _pinned(n):
    return torch.empty(n, dtype=torch.int32, pin_memory=True)


def _ensemble(c, seed):
    reps = workloads.ensemble_replicas(c["ising"], c["potts"], c["sweeps"], c["mix"])
    return [dict(r, seed=1 + (seed * 1009 + r["id"]) % 899999999) for r in reps]


def _queue(c, seed):
    reqs = workloads.serving_requests(200.0, c["requests"], c["mix"])
    return [dict(r, arrive=0.0, seed=1 + (seed * 1009 + r["id"]) % 899999999) for r in reqs]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "lattice":
        L = hip.Lattice(case["app"], case["style"], case["nx"], case["ny"], case["nz"], case["q"], case["kT"])
        s0, rseed = _start(seed)
        L.set_range(s0, 1, case["q"])
        L.init_seeds(rseed)
        L.prepare(case["sweeps"])
        return {"kind": kind, "L": L, "sweeps": case["sweeps"], "spin": _pinned(L.n), "seed": _pinned(L.n)}
    if kind == "script":
        s = spparks("", ["-screen", "none", "-log", "none"])
        for line in ("seed %d" % (1 + seed % 899999999), "app_style potts %d" % case["q"], "dimension 2",
                     "lattice sq/8n 1.0",
                     "region box block 0 %d 0 %d -0.5 0.5" % (case["nx"], case["ny"]), "create_box box",
                     "create_sites box", "set site range 1 %d" % case["q"], "sweep color/strict",
                     "temperature %g" % case["kT"], "diag_style energy", "stats 0.01", "run 0.0"):
            s.command(line)
        return {"kind": kind, "s": s, "run": "run %g" % case["time"], "n": case["nx"] * case["ny"]}
    if kind == "batch":
        reps = _ensemble(case, seed)
        sites = [r["shape"][0] * r["shape"][1] * r["shape"][2] for r in reps]
        pool = sum(replica_bytes(r["app"], r["lattice"], *r["shape"], nspins=r["nspins"]) for r in reps)
        B = Batch(pool, len(reps))
        # the program runs the ensemble on for as long as it is called
        ids = [B.add(replica_desc(r["app"], r["lattice"], *r["shape"], nspins=r["nspins"], temperature=r["kT"],
                                  seed=r["seed"], nsweeps=10**9)) for r in reps]
        at = np.concatenate([[0], np.cumsum(sites)])
        return {"kind": kind, "B": B, "ids": ids, "sweeps": case["sweeps"], "at": [int(x) for x in at],
                "spin": _pinned(int(at[-1])), "seed": _pinned(int(at[-1]))}
    return {"kind": kind, "requests": _queue(case, seed), "live": case["live"]}


def run(state):
    kind = state["kind"]
    if kind == "lattice":
        L = state["L"]
        _, nacc, energy = L.sweeps(state["sweeps"])
        hip._check(L.L.spk_hip_download(L.h, state["spin"].data_ptr(), state["seed"].data_ptr()))
        return {"naccept": nacc, "energy": energy, "spin": state["spin"], "seed": state["seed"]}
    if kind == "script":
        s = state["s"]
        s.command(state["run"])
        energy = s.energy()
        return {"energy": energy, "spin": np.ctypeslib.as_array(s.extract("site", 1), (state["n"],)).copy()}
    if kind == "batch":
        B, spin, seed, at = state["B"], state["spin"], state["seed"], state["at"]
        B.run(state["sweeps"])
        status = [B.status(i) for i in state["ids"]]
        for k, i in enumerate(state["ids"]):
            hip._check(B.L.spk_hip_batch_download(B.h, i, spin[at[k]:].data_ptr(), seed[at[k]:].data_ptr()))
        return {"done": np.array([x[0] for x in status]), "naccept": np.array([x[2] for x in status]),
                "energy": np.array([x[3] for x in status]), "spin": spin, "seed": seed}
    res, _ = serve(state["requests"], 16 << 30, state["live"])
    return {"naccept": np.array([r["naccept"] for r in res]), "energy": np.array([r["energy"] for r in res]),
            "checksum": np.array([r["checksum"] for r in res], np.uint64).view(np.int64),
            "status": np.array([r["status"] for r in res])}


# ---------------------------------------------------- work of one pass
def _parts(case):
    """(app, style, sites, Q, sweeps) of every lattice of a pass."""
    if case["kind"] in ("lattice", "script"):
        n = case["nx"] * case["ny"] * case["nz"]
        return [(case["app"], case["style"], n, case["q"], case.get("sweeps", 100))]
    reps = _ensemble(case, 0) if case["kind"] == "batch" else _queue(case, 0)
    return [(r["app"], r["lattice"], int(np.prod(r["shape"])), r["nspins"], r["sweeps"]) for r in reps]


def work(case):
    nbytes = flops = 0
    for app, style, n, q, sweeps in _parts(case):
        state = n * (4 + (1 if q <= 255 else 2 if q <= 65535 else 4))
        out = 0 if case["kind"] == "serve" else 4 * n if case["kind"] == "script" else 8 * n
        nbytes += 2 * state + out
        flops += n * sweeps * ((1 if app.startswith("ising") else 2) * NEIGHBOURS[style] + EVENT_OPS)
    return {"bytes": nbytes, "flops": flops}


# ------------------------------------------------------- results in 64 bits
IM = 2**31 - 1


def _mul(a, b):
    """a*b mod 2^31-1 of int64 tensors below it: the product stays below 2^62."""
    return (a * b) % IM


def _initial(case, seed, dev):
    s0, rseed = _start(seed)
    n = case["nx"] * case["ny"] * case["nz"]
    gid = torch.arange(1, n + 1, dtype=torch.int64, device=dev)
    s, p = torch.full_like(gid, s0), 16807
    for bit in range(32):
        s = torch.where((gid >> bit) & 1 == 1, _mul(s, torch.full_like(s, p)), s)
        p = p * p % IM
    q = case["q"]
    spin = torch.clamp((s.double() * (1.0 / IM) * q).long() + 1, max=q).int()
    x = rseed * IM + gid.double()
    k = torch.where(x >= IM, x - IM, x).long()
    k[k == 0] = 1
    shape = (case["nz"], case["ny"], case["nx"])
    return spin.view(shape), _mul(k, torch.full_like(k, pow(16807, 100, IM))).view(shape)


def _offsets(style):
    three, far = style.startswith("sc"), {"sq/4n": 1, "sc/6n": 1, "sq/8n": 2, "sc/26n": 3}[style]
    return [(i, j, k) for i in (-1, 0, 1) for j in (-1, 0, 1) for k in ((-1, 0, 1) if three else (0,))
            if 1 <= i * i + j * j + k * k <= far]


def _event(app, q, kt, old, seed, nb):
    """(new spin, new seed) of the strict event of every site; kt > 0."""
    nn = len(nb)
    draw1 = _mul(seed, torch.full_like(seed, 16807))
    u, event = draw1.double() * (1.0 / IM), torch.ones_like(old, dtype=torch.bool)
    if app == "ising":
        prop, s = torch.where(u < 0.5, 1, 2).int(), draw1
    elif app == "ising/single":
        prop, s = 3 - old, seed
    elif app == "potts":
        prop, s = torch.clamp((q * u).long() + 1, max=q).int(), draw1
    else:
        fresh = []
        for m in range(nn):
            f = nb[m] != old
            for i in range(m):
                f &= nb[i] != nb[m]
            fresh.append(f)
        nevent = sum(f.long() for f in fresh)
        if app == "potts/neigh":
            pick, s = (nn * u).long(), draw1
            event = pick < nevent
        else:
            event = nevent > 0
            s = torch.where(event, draw1, seed)
            pick = torch.minimum((nevent * u).long(), nevent - 1)
        prop, seen = old.clone(), torch.zeros_like(nevent)
        for m in range(nn):
            prop = torch.where(event & fresh[m] & (seen == pick), nb[m], prop)
            seen += fresh[m]
    d = torch.zeros_like(old)
    for v in nb:
        d += (v != prop).int() - (v != old).int()
    up = event & (d > 0)
    draw2 = _mul(s, torch.full_like(s, 16807))
    table = torch.tensor([1.0] + [math.exp(-k * (1.0 / kt)) for k in range(1, nn + 1)], dtype=torch.float64,
                         device=old.device)
    passed = ~(draw2.double() * (1.0 / IM) > table[d.clamp(min=0).long()])
    keep = event & (~up | passed)
    return torch.where(keep, prop, old), torch.where(up, draw2, s)


def exact(case, seed):
    if case["kind"] != "lattice" or not case["kT"] > 0:
        return None
    style, app = case["style"], case["app"]
    n = case["nx"] * case["ny"] * case["nz"]
    per = NEIGHBOURS[style] * (20 if "neigh" in app else 1) + EVENT_OPS
    if n * case["sweeps"] * per > 5e11 or case["sweeps"] * per > 1e5:
        return None   # too long
    dev = torch.device("cuda")
    spin, seeds = _initial(case, seed, dev)
    off, energies = _offsets(style), []
    checker = style in ("sq/4n", "sc/6n")
    half = off[: len(off) // 2]   # each pair of neighbours once
    if checker:
        z, y, x = (torch.arange(k, device=dev) for k in spin.shape)
        parity = (z[:, None, None] + y[None, :, None] + x[None, None, :]) & 1
    for _ in range(case["sweeps"]):
        for c in range(2 if checker else 4 if style == "sq/8n" else 8):
            if checker:
                nb = [torch.roll(spin, (-k, -j, -i), (0, 1, 2)) for i, j, k in off]
                new, ns = _event(app, case["q"], case["kT"], spin, seeds, nb)
                spin, seeds = torch.where(parity == c, new, spin), torch.where(parity == c, ns, seeds)
                continue
            par = (c >> 2, (c >> 1) & 1, c & 1)   # z, y, x
            sub = lambda a, p: a[p[0]::2, p[1]::2, p[2]::2]  # noqa: E731
            nb = []
            for i, j, k in off:
                d = (k, j, i)
                p = [par[m] ^ (d[m] & 1) for m in range(3)]
                # site 2a + par + d lies at index a + (par + d - p) / 2 of its sub-grid
                nb.append(torch.roll(sub(spin, p), [-((par[m] + d[m] - p[m]) // 2) for m in range(3)], (0, 1, 2)))
            new, ns = _event(app, case["q"], case["kT"], sub(spin, par), sub(seeds, par), nb)
            sub(spin, par).copy_(new)
            sub(seeds, par).copy_(ns)
        energies.append(2 * sum((torch.roll(spin, (-k, -j, -i), (0, 1, 2)) != spin).sum() for i, j, k in half))
    return {"naccept": None, "energy": torch.stack(energies).double(), "spin": None, "seed": None}
