"""The work whose speed is followed from change to change.

Every case is one call that a user's program makes through the public entry
points: a batch of replicas advanced by some sweeps with its measured frames
(engine.Batch.run), or one (T, h) point through the drop-in modules
(isinglib / heisenberglib .MCMainFunction).  The lattices, couplings,
temperature and field ranges are those of mcsolver_amd.workloads; sizes go
from one lattice of a few hundred sites to 10^7 sites in one batch, with odd
edge lengths among them (an odd periodic edge needs a third colour, so these
are not only remainders of the even case).

A batch starts from spins spread around the ordered state, as a run has them
after its first sweeps; a batch of Wolff clusters starts from a few hundred
Metropolis sweeps at its temperature, because cluster sizes follow from the
correlations of an equilibrated lattice.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from mcsolver_amd import _lib as L
from mcsolver_amd import heisenberglib, isinglib
from mcsolver_amd import lattice as lat
from mcsolver_amd import workloads as W
from mcsolver_amd.engine import Batch, ReplicaSpec, compile_graph

NBINS = 16
COMPONENTS = {"ising": 1, "xy": 2, "honeycomb": 3, "triangular": 3, "cubic": 3}
LINKS = {"ising": 4, "xy": 4, "honeycomb": 9, "triangular": 6, "cubic": 6}
RANGES = {"ising": (1.5, 3.5), "xy": (0.7, 1.2), "honeycomb": (0.1, 2.0), "triangular": (0.05, 1.0),
          "cubic": (1.2, 1.7)}  # temperatures of each model's scan


def _batch(name, model, edges, temps, sweeps, *, store="f32", fields=1, swap=0, per_frame=1, thermal=0, pairs=True,
           charge=False, wolff=0):
    """edges: the edge lengths in the batch ("16 24": two lattices, each with
    every temperature and field); sweeps: measured and unmeasured sweeps in
    all, `thermal` of them unmeasured first, then one frame each `per_frame`;
    swap: replica exchange along the temperatures each so many sweeps (0:
    none); wolff: clusters per frame instead of sweeps."""
    return {"name": name, "kind": "batch", "model": model, "edges": edges, "temps": temps, "fields": fields,
            "store": "i8" if model == "ising" else store, "sweeps": sweeps, "thermal": thermal,
            "per_frame": per_frame, "swap": swap, "pairs": pairs, "charge": charge, "wolff": wolff}


def _point(name, model, edge, thermal, frames):
    return {"name": name, "kind": "point", "model": model, "edge": edge, "thermal": thermal, "frames": frames}


def listed():
    return [
        # one (T, h) point of a reference user's scan through the drop-in
        # module: tuples in, observables out; one lattice cannot fill the GPU,
        # so this is the latency of a sweep plus the call's host work
        _point("point_ising_32", "ising", 32, 1000, 3000),
        # the same for a Heisenberg lattice with full exchange tensors
        _point("point_heis_honeycomb_16", "honeycomb", 16, 500, 1000),
        # a small temperature scan in one batch: the smallest launches
        _batch("ising_32_16T", "ising", "32", 16, 200),
        # a finite-size Ising point of a large lattice, thermalised and then
        # measured every fifth sweep
        _batch("ising_250_40T", "ising", "250", 40, 50, thermal=25, per_frame=5),
        # the Binder scan that bench.py times: seven lattices in one launch,
        # 64 tempering rungs each, swaps and a frame every sweep (production)
        _batch("xy_ladders_7x64T", "xy", "16 24 32 48 64 96 128", 64, 100, swap=1, pairs=False),
        # a smaller scan with odd edges, sparse swaps and sparse frames
        _batch("xy_ladders_odd_4x24T", "xy", "15 33 50 75", 24, 100, swap=5, per_frame=5, pairs=True),
        # a two-orbital magnet with nine full tensors a site
        _batch("honeycomb_64_64T", "honeycomb", "64", 64, 50),
        # the same model in 16-bit storage on an odd lattice, thermalising
        # before it measures
        _batch("honeycomb_45_f16_24T", "honeycomb", "45", 24, 50, store="f16", thermal=30),
        # a skyrmion phase diagram: fields x temperatures, topological charge
        # every sweep; 32-bit spins do not fit LDS, 16-bit spins do
        _batch("triangular_128_32x32", "triangular", "128", 32, 5, fields=32, charge=True),
        _batch("triangular_128_f16_32x32", "triangular", "128", 32, 10, store="f16", fields=32, charge=True),
        # a three-dimensional magnet around its critical temperature: the
        # largest batch, Metropolis
        _batch("cubic_64_128T", "cubic", "64", 128, 8, per_frame=2),
        # the same lattice at T_c with cluster updates
        _batch("cubic_64_wolff_16", "cubic", "64", 16, 4, wolff=16),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the listed ones' ranges: any model, edge lengths spread over
    their logarithm (odd ones as likely as even), and as many sweeps as keep
    it below the listed case of its kind."""
    pick = rng.choice(("point", "ising", "xy", "xy", "honeycomb", "triangular", "cubic", "cubic", "wolff"))
    if pick == "point":
        if rng.random() < 0.5:
            c = _point("", "ising", _log(rng, 6, 48), rng.randrange(200, 1000), rng.randrange(500, 2500))
        else:
            c = _point("", "honeycomb", _log(rng, 5, 16), rng.randrange(100, 500), rng.randrange(200, 1000))
    elif pick == "xy":
        edges = sorted(_log(rng, 12, 128) for _ in range(rng.randrange(1, 6)))
        c = _batch("", "xy", " ".join(map(str, edges)), rng.randrange(8, 65), rng.randrange(20, 100),
                   swap=rng.choice((0, 1, 1, 4)), per_frame=rng.choice((1, 1, 3)), pairs=rng.random() < 0.5)
    elif pick == "wolff":
        c = _batch("", "cubic", str(_log(rng, 12, 64)), rng.randrange(4, 17), rng.randrange(2, 5),
                   wolff=rng.randrange(4, 17))
    else:
        store = rng.choice(("f32", "f32", "f16"))
        if pick == "ising":
            c = _batch("", "ising", str(_log(rng, 12, 300)), rng.randrange(8, 49), rng.randrange(20, 200))
        elif pick == "honeycomb":
            c = _batch("", "honeycomb", str(_log(rng, 12, 72)), rng.randrange(8, 65), rng.randrange(10, 50),
                       store=store)
        elif pick == "triangular":
            c = _batch("", "triangular", str(_log(rng, 24, 128)), rng.randrange(8, 33), rng.randrange(3, 10),
                       store=store, fields=rng.randrange(2, 33), charge=True)
        else:
            c = _batch("", "cubic", str(_log(rng, 10, 64)), rng.randrange(8, 97), rng.randrange(4, 9), store=store)
        c["thermal"] = rng.choice((0, 0, c["sweeps"] // 2))
        c["per_frame"] = rng.choice((1, 1, 2))
    if c["kind"] == "batch" and not c["wolff"]:  # at most the largest listed batch
        cap = {"ising": 1.2e8, "xy": 2.1e8, "honeycomb": 2.6e7, "triangular": 8e7, "cubic": 2.6e8}[c["model"]]
        most = int(cap / max(1, _sites(c)))
        c["sweeps"] = max(2, min(c["sweeps"], most))
        c["thermal"] = min(c["thermal"], c["sweeps"] // 2)
        c["per_frame"] = min(c["per_frame"], c["sweeps"] - c["thermal"])
    del c["name"]
    return c


# --------------------------------------------------------------------------
# what a program has in hand: lattices compiled once, then one batch
# --------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _lattice(model, edge):
    if model == "ising":
        return lat.square(edge, J=-1.0, ising=True)
    if model == "xy":
        return lat.square(edge, J=-1.0)
    if model == "honeycomb":
        return W.honeycomb_full_tensor(edge)
    if model == "triangular":
        return W.triangular_neel_dmi(edge)
    return lat.cubic(edge, J=-1.0)


@functools.lru_cache(maxsize=None)
def _graph(model, edge):
    x = _lattice(model, edge)
    nc = COMPONENTS[model]
    return compile_graph(nc, x.nbr, x.J if nc > 1 else x.J[:, :, :1], x.S, x.D, pairs=x.corr_pairs,
                         circuits=x.circuits if nc == 3 and len(x.circuits) else None)


def _edges(case):
    return [int(v) for v in case["edges"].split()]


def _volume(model, edge):
    return edge ** 3 if model == "cubic" else edge * edge * (2 if model == "honeycomb" else 1)


def _sites(case):
    return sum(_volume(case["model"], e) for e in _edges(case)) * case["temps"] * case["fields"]


def _rows(case):
    """(edge index, temperature, field) of every replica."""
    ts = np.linspace(*RANGES[case["model"]], case["temps"])
    if case["wolff"]:
        ts = np.full(case["temps"], 1.44)  # the critical temperature of this lattice is near 1.443
    hs = np.linspace(0.0, 1.0, case["fields"]) if case["fields"] > 1 else np.zeros(1)
    return [(e, t, h) for e in range(len(_edges(case))) for h in hs for t in ts]


def _spins(model, count, gen):
    """[components, count] spins spread around the ordered state."""
    nc = COMPONENTS[model]
    if nc == 1:
        return torch.where(torch.rand(1, count, generator=gen, device="cuda") < 0.85, 1.0, -1.0)
    v = torch.randn(nc, count, generator=gen, device="cuda") * 0.5
    v[0] += 1.0
    return v / v.norm(dim=0, keepdim=True)


def prepare(case, seed):
    model = case["model"]
    if case["kind"] == "point":
        # the temperature of the point comes from the seed: the drop-in
        # modules take no random seed
        t = float(np.random.default_rng(seed).uniform(*RANGES[model]))
        x = _lattice(model, case["edge"])
        make = lat.ising_args if model == "ising" else lat.on_args
        return {"main": isinglib.MCMainFunction if model == "ising" else heisenberglib.MCMainFunction,
                "args": make(x, t, 0.0, case["thermal"], case["frames"])}
    nc = COMPONENTS[model]
    graphs = [_graph(model, e) for e in _edges(case)]
    rows = _rows(case)
    per = case["temps"]
    reps, start = [], []
    for k, (e, _, _) in enumerate(rows):
        if case["swap"]:
            reps.append(ReplicaSpec(e, k // per * per, nrung=per, ladder=k // per, rung=k % per))
        else:
            reps.append(ReplicaSpec(e, k))
        start.append(np.zeros((graphs[e].n, nc), np.float32))
    meas = (L.MEAS_PAIRS if case["pairs"] else 0) | (L.MEAS_Q if case["charge"] else 0)
    b = Batch(nc, graphs, reps, [1.0 / max(t, 0.1) for _, t, _ in rows], [h for _, _, h in rows], start,
              store="f32" if nc == 1 else case["store"], meas=meas, nbins=NBINS, nframes=_frames(case), seed=seed,
              wolff=case["wolff"] > 0, recompute_every=L.RECOMPUTE_EVERY)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    for k, (e, _, _) in enumerate(rows):
        n = graphs[e].n
        b.spins[b.spin_off[k]:b.spin_off[k] + nc * n] = _spins(model, n, gen).reshape(-1).to(b.dtype)
    b.init()
    if case["wolff"]:
        b.sweeps(None, 200)
        b.init()
    return {"batch": b, "case": case}


def _frames(case):
    return case["sweeps"] if case["wolff"] else (case["sweeps"] - case["thermal"]) // case["per_frame"]


def run(state):
    if "args" in state:
        return [v for v in state["main"](*state["args"]) if not math.isnan(v)]
    b, case = state["batch"], state["case"]
    if case["wolff"]:
        b.run(0, _frames(case), 1, algorithm=L.WOLFF, clusters_per_sweep=case["wolff"])
    else:
        b.run(case["thermal"], _frames(case), case["per_frame"], pt_every=case["swap"])
    return {"spins": b.spins, "state": b.state, "acc": b.acc, "bins": b.bins, "rung": b.rung, "who": b.who,
            "swaps": b.pt_acc, "err": b.err}


def work(case):
    """Bytes: every spin in and out once, and each row's sums.  Operations of
    an update: the field over the links, the proposal, the energy change and
    the acceptance, and its share of a counter-based random draw."""
    model = case["model"]
    nc, z = COMPONENTS[model], LINKS[model]
    if case["kind"] == "point":
        n = _volume(model, case["edge"])
        sweeps = case["thermal"] + case["frames"]
        return {"bytes": float(n * (z * (1 if nc == 1 else 9) * 8 + z * 8 + 2 * nc * 4)),
                "flops": float(n * sweeps * _operations(nc, z, model != "ising"))}
    size = {"f32": 4, "f16": 2, "i8": 1}[case["store"]]
    n = _sites(case)
    rows = len(_rows(case))
    if case["wolff"]:
        # a cluster of the critical lattice holds a few thousand sites
        updates = case["temps"] * _frames(case) * case["wolff"] * min(n / case["temps"] / 50.0, 5000.0)
    else:
        updates = float(n) * (case["thermal"] + _frames(case) * case["per_frame"])
    flops = updates * _operations(nc, z, model in ("honeycomb", "triangular"))
    if case["charge"]:
        flops += 2.0 * n * _frames(case) * 60
    return {"bytes": float(2 * n * nc * size + rows * 8 * (L.NACC + L.NSTATE + NBINS * L.NBINQ)), "flops": flops}


def _operations(nc, z, tensors):
    draw = 10 * 8 + 20  # ten rounds of two products and the mixing
    if nc == 1:
        return draw / 4 + z + 6
    field = z * (2 * nc * nc if tensors else nc)
    return draw / (2 if nc == 2 else 1) + field + (55 if nc == 2 else 75)


# --------------------------------------------------------------------------
# 64-bit values
# --------------------------------------------------------------------------
# A Metropolis trajectory of continuous spins has no 64-bit value: one
# acceptance decided in the last bit of a 32-bit sum sends the rest of the
# lattice elsewhere, in any precision.  The Ising batches have one, because
# their flips compare integers: a flip that costs energy is accepted when a
# 32-bit random word is below floor(2^32 exp(-beta dE)).
def exact(case, seed):
    if case["kind"] != "batch" or case["model"] != "ising" or int(case["edges"]) % 2 or _sites(case) * case["sweeps"] > 3e8:
        return None
    edge = int(case["edges"])
    n, rows = edge * edge, _rows(case)
    beta = torch.tensor([np.float32(1.0 / max(t, 0.1)) for _, t, _ in rows], dtype=torch.float64, device="cuda")
    gen = torch.Generator(device="cuda").manual_seed(seed)
    # positions are sites grouped by the checkerboard's two colours
    site = torch.arange(n, device="cuda")
    x, y = site // edge, site % edge
    colour = (x + y) % 2
    order = torch.cat([site[colour == 0], site[colour == 1]])
    spin = torch.empty(len(rows), n, dtype=torch.int64, device="cuda")
    for k in range(len(rows)):
        spin[k, order] = _spins("ising", n, gen).reshape(-1).to(torch.int64)
    near = [((x + 1) % edge) * edge + y, ((x - 1) % edge) * edge + y, x * edge + (y + 1) % edge,
            x * edge + (y - 1) % edge]

    def field():
        return sum(spin[:, j] for j in near)

    energy = lambda: -0.5 * (spin * field()).sum(1).double()  # noqa: E731
    acc = torch.zeros(len(rows), L.NACC, dtype=torch.float64, device="cuda")
    bins = torch.zeros(len(rows), NBINS, L.NBINQ, dtype=torch.float64, device="cuda")
    start, frames = energy(), _frames(case)
    ref = start
    key = (torch.tensor(seed & 0xFFFFFFFF, device="cuda"),
           ((seed >> 32) & 0xFFFFFFFF) ^ torch.arange(len(rows), device="cuda").unsqueeze(1))
    limit = torch.floor(torch.exp(-beta.unsqueeze(1) * torch.arange(0, 9, device="cuda").double()) * 2.0 ** 32)
    limit = limit.clamp(max=2.0 ** 32 - 1).to(torch.int64)
    for k in range(case["thermal"] + frames * case["per_frame"]):
        for c in (0, 1):
            at = site[colour == c]
            word = _philox(torch.arange((len(at) + 3) // 4, device="cuda").unsqueeze(0), k, c << 8, *key)
            word = torch.stack(word, 2).reshape(len(rows), -1)[:, :len(at)]
            cost = 2 * spin[:, at] * field()[:, at]
            flip = (cost <= 0) | (word < torch.gather(limit, 1, cost.clamp(min=0)))
            spin[:, at] = torch.where(flip, -spin[:, at], spin[:, at])
        if k + 1 == case["thermal"]:
            ref = energy()
        f = k + 1 - case["thermal"]
        if f <= 0 or f % case["per_frame"]:
            continue
        f = f // case["per_frame"] - 1
        e, tot = energy() / n, spin.sum(1).double()
        m = tot / n
        for q, v in ((L.A_E, e), (L.A_E2, e * e), (L.A_M, m), (L.A_M2, m ** 2), (L.A_M4, m ** 4),
                     (L.A_MM, m * acc[:, L.A_MPREV]), (L.A_SI, m.abs()), (L.A_SJ, m.abs()),
                     (L.A_SIJ, torch.ones_like(m)), (L.A_COUNT, torch.ones_like(m)),
                     (L.A_LAST, spin[:, n - 1].double()), (L.A_TOT, tot), (L.A_ABSM, m.abs())):
            acc[:, q] += v
        acc[:, L.A_MPREV] = m
        bins[:, f * NBINS // frames] += torch.stack([e, e * e, m, m ** 2, m ** 4], 1)
    zero = torch.zeros_like(ref)
    state = torch.stack([energy(), spin.sum(1).double(), zero, zero, ref, zero, zero, zero], 1)
    return {"spins": None, "state": state.reshape(-1), "acc": acc.reshape(-1), "bins": bins.reshape(-1), "rung": None,
            "who": None, "swaps": None, "err": None}


def _philox(counter, sweep, tag, key0, key1):
    """Philox4x32-10 (Salmon et al., SC'11) words of the counters (counter,
    sweep, 0, tag), in 64-bit integers."""
    low = 0xFFFFFFFF
    a, b = counter + 0 * key1, torch.full_like(counter + 0 * key1, sweep & low)
    c, d = torch.full_like(a, sweep >> 32), torch.full_like(a, tag)
    for _ in range(10):
        p, q = a * 0xD2511F53, c * 0xCD9E8D57
        a, b, c, d = ((q >> 32) & low) ^ b ^ key0, q & low, ((p >> 32) & low) ^ d ^ key1, p & low
        key0, key1 = (key0 + 0x9E3779B9) & low, (key1 + 0xBB67AE85) & low
    return a, b, c, d
