"""The work that programs give this engine, as cases that can be timed.

Every case is one or more maximal biclique enumerations through the package's
public entry points. Graphs come from the package's own generators with a
random seed, at the sizes of its configurations, tests and benchmark:

  kind "solve"    cumbe_amd.solve: one graph per call, host graph in, count
                  and hash out (what the `mbe` command does)
  kind "noalloc"  cumbe_amd.solve_noalloc: the graph packed in device memory
  kind "list"     cumbe_amd.solve_list: every biclique as vertex lists
  kind "batch"    cumbe_amd.batch_solve: many graphs in one call
  kind "plan"     cumbe_amd.BatchPlan.run: a batch kept on the device
  kind "serve"    cumbe_amd.Server: a burst of concurrent requests

The graphs are `cl` (Chung-Lu: n_u, n_v, m edges, one exponent per side,
max_deg or 0), `er` (random plus planted bicliques) and `mix` (n graphs of
the batched workload's size distribution, those whose enumeration is known to
be feasible). A few graph seeds change the number of bicliques by some ten
per cent; the sizes, not the seed, set the cost of a case.
"""
import math
import os
import random

import numpy as np
import torch

import cumbe_amd as M
from cumbe_amd import autotune, serve_bench

SEEDS_CSV = os.path.join("tests", "golden", "batch_c3.csv")
MIX_MAX_WORK = 10 ** 11    # adjacency entries the serial algorithm scans per mixed graph
MIX_EDGES = 3300           # mean edges of a mixed graph
MIX_VERTICES = 1540        # mean vertices of a mixed graph


def _cl(name, kind, n_u, n_v, m, gamma_u, gamma_v, max_deg, variant="cuMBE", begin=0, end=0,
        tuned=""):
    c = {"kind": kind, "graph": "cl", "n_u": n_u, "n_v": n_v, "m": m, "gamma_u": gamma_u,
         "gamma_v": gamma_v, "max_deg": max_deg, "variant": variant, "begin": begin, "end": end,
         "tuned": tuned}
    return dict(c, name=name) if name else c


def _er(name, n_u, n_v, planted, begin, end, variant="cuMBE"):
    c = {"kind": "solve", "graph": "er", "n_u": n_u, "n_v": n_v, "p": 0.008, "planted": planted,
         "variant": variant, "begin": begin, "end": end, "tuned": ""}
    return dict(c, name=name) if name else c


def _mix(name, kind, n):
    c = {"kind": kind, "graph": "mix", "n": n, "variant": "cuMBE"}
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest calls: an interactive query on a small graph, where
        # latency, launches and the tail of a nearly empty chip count
        _cl("solve_small", "solve", 200, 100, 600, 2.1, 2.1, 0),
        # configuration 0: an ordinary graph, one call (the command-line use)
        _cl("solve_medium", "solve", 2000, 1000, 10000, 2.1, 2.1, 0),
        # odd sizes in the other search variants the command offers
        _cl("solve_medium_noRS", "solve", 1777, 1203, 9001, 2.1, 2.1, 0, "noRS"),
        _cl("solve_medium_noES", "solve", 1311, 907, 7003, 2.1, 2.2, 0, "noES"),
        # the headline workload: skewed degrees, thousands of candidates per
        # root, every root below the hub core, launch parameters from the
        # tuning cache
        _cl("solve_skewed", "solve", 94000, 30000, 293000, 2.0, 1.8, 7600, begin=400,
            tuned="c1_roots400"),
        # the largest graph: many roots, small subtrees; upload and
        # preparation are part of the call
        _cl("solve_large", "solve", 200000, 100000, 1500000, 2.0, 2.0, 128),
        # random graph with planted bicliques: the background roots, and the
        # planted core (few roots, deep trees that have to be split)
        _er("solve_planted", 6500, 1900, 60, 95, 0),
        _er("solve_planted_core", 6500, 1900, 60, 0, 15),
        # the allocation-free call on a packed device graph
        _cl("noalloc_medium", "noalloc", 1500, 801, 7003, 2.1, 2.1, 0),
        # every biclique as vertex lists
        _cl("list_medium", "list", 600, 400, 2500, 2.1, 2.1, 0),
        # batches: resident and replayed; from host graphs served as a burst
        _mix("plan_256", "plan", 256),
        _mix("serve_48", "serve", 48),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    variant = rng.choice(["cuMBE", "cuMBE", "cuMBE", "noRS", "noES", "noWS"])
    kind = rng.choice(["solve", "solve", "noalloc", "list", "skewed", "large", "planted", "core",
                       "batch", "plan", "serve"])
    if kind in ("solve", "noalloc", "list"):
        n_u = log(100, 800 if kind == "list" else 2500)
        n_v = max(50, int(n_u * rng.uniform(0.4, 1.2)))
        g = round(rng.uniform(2.1, 2.5), 2)
        return _cl("", kind, n_u, n_v, int(n_u * rng.uniform(2.5, 5.0)), g, g,
                   rng.choice([0, 0, 100]), variant)
    if kind == "skewed":
        return _cl("", "solve", 94000, 30000, 293000, 2.0, 1.8, 7600,
                   begin=rng.randint(500, 3000), tuned=rng.choice(["", "c1_roots400"]))
    if kind == "large":
        n_u = log(10000, 200000)
        return _cl("", "solve", n_u, int(n_u * rng.uniform(0.3, 0.8)),
                   int(n_u * rng.uniform(4.0, 7.5)), 2.0, 2.0, rng.randint(48, 128),
                   rng.choice(["cuMBE", "noRS", "noES"]))
    if kind in ("planted", "core"):
        n_v = log(600, 1900)
        n_u = int(n_v * rng.uniform(2.0, 3.4))
        top = int(math.ceil(0.05 * n_v))
        if kind == "planted":
            return _er("", n_u, n_v, rng.randint(20, 60), top, 0, variant)
        return _er("", n_u, n_v, rng.randint(20, 60), 0, rng.randint(6, 15))
    return _mix("", kind, log(8, 48) if kind == "serve" else log(8, 250))


def _graph(case, seed):
    if case["graph"] == "cl":
        return M.Graph.chung_lu(case["n_u"], case["n_v"], case["m"], case["gamma_u"],
                                case["gamma_v"], case["max_deg"], seed)
    return M.Graph.er_planted(case["n_u"], case["n_v"], case["p"], case["planted"], 8, 40, 0.05,
                              seed)


def _mixed(case, seed):
    known = serve_bench.seeds_from_csv(SEEDS_CSV, MIX_MAX_WORK)
    return [M.Graph.batch_graph(s) for s in random.Random(seed).sample(known, case["n"])]


def prepare(case, seed):
    M.init()
    s = {"kind": case["kind"], "variant": case["variant"]}
    if case["graph"] == "mix":
        gs = _mixed(case, seed)
        if case["kind"] == "plan":
            s["plan"] = M.BatchPlan(gs)
        else:
            s["graphs"] = gs
        return s
    g = _graph(case, seed)
    tuning = dict((autotune.cached(case["tuned"]) or {}) if case["tuned"] else {})
    if case["begin"]:
        tuning["root_begin"] = case["begin"]
    if case["end"]:
        tuning["root_end"] = case["end"]
    s["tuning"] = tuning or None
    s["room"] = _room(case) if case["kind"] == "list" else None
    if case["kind"] == "noalloc":
        packed, s["info"] = g.pack()
        s["packed"] = torch.from_numpy(packed).cuda()
    else:
        s["graph"] = g
    return s


def _numbers(results):
    return {"count": np.array([r.count for r in results], dtype=np.uint64).view(np.int64),
            "hash": np.array([r.hash for r in results], dtype=np.uint64).view(np.int64)}


def run(state):
    kind = state["kind"]
    if kind == "solve":
        return _numbers([M.solve(state["graph"], state["variant"], state["tuning"])])
    if kind == "noalloc":
        return _numbers([M.solve_noalloc(state["packed"].data_ptr(), state["info"],
                                         state["variant"], state["tuning"])])
    if kind == "list":
        r, bicliques = M.solve_list(state["graph"], state["variant"], state["tuning"])
        return dict(_numbers([r]), **_flat(bicliques, state["room"]))
    if kind == "batch":
        return _numbers(M.batch_solve(state["graphs"], state["variant"])[0])
    if kind == "plan":
        return _numbers(state["plan"].run()[0])
    # a burst of requests to a server of its own, sized for small graphs
    with M.Server(table_cap=4096, data_bytes=256 << 20, staging_bytes=64 << 20) as server:
        tickets = [server.submit(g, state["variant"]) for g in state["graphs"]]
        return _numbers([server.poll(t, wait_ms=-1) for t in tickets])


def _flat(bicliques, room):
    """[(A, B), ...] as arrays of the program's fixed sizes, -1 in unused
    places: the sizes of each pair, and all ids in order."""
    sizes = [n for a, b in bicliques for n in (len(a), len(b))]
    ids = [i for a, b in bicliques for s in (a, b) for i in s]
    out = {"sizes": np.full(room[0], -1, dtype=np.int64), "ids": np.full(room[1], -1, dtype=np.int64)}
    out["sizes"][:len(sizes)] = sizes
    out["ids"][:len(ids)] = ids
    return out


def _room(case):
    return 32 * case["m"], 256 * case["m"]


def work(case):
    """The graph's adjacency (32-bit ids, both directions are one input) and
    offsets read once, and the results written."""
    if case["graph"] == "mix":
        return {"bytes": case["n"] * (4 * (MIX_EDGES + MIX_VERTICES) + 16), "flops": 0}
    edges = case["m"] if case["graph"] == "cl" else (
        case["n_u"] * case["n_v"] * case["p"] + case["planted"] * 24 * 24)
    return {"bytes": int(4 * (edges + case["n_u"] + case["n_v"]) + 16), "flops": 0}


def tolerance(case):
    """Counts, hashes and vertex lists are whole numbers."""
    return "exact"


def _mix64(z):
    z &= (1 << 64) - 1
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & ((1 << 64) - 1)
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & ((1 << 64) - 1)
    return z ^ (z >> 31)


def exact(case, seed):
    """By closure: the column sides of the maximal bicliques are the nonempty
    intersections of row neighbourhoods."""
    if case["graph"] != "cl" or case["n_u"] > 700 or case["begin"] or case["end"]:
        return None
    n_u, n_v, off, adj = _graph(case, seed).csr()
    rows = [sum(1 << int(v) for v in adj[off[u]:off[u + 1]]) for u in range(n_u)]
    cols = set()
    for r in set(rows):
        if r:
            cols |= {c & r for c in cols} | {r}
    cols.discard(0)
    full = (1 << 64) - 1
    total, pairs = 0, []
    for c in cols:
        a = tuple(u for u in range(n_u) if c & rows[u] == c)
        b = tuple(v for v in range(n_v) if (c >> v) & 1)
        s_u = sum(_mix64(u ^ 0x9E3779B97F4A7C15) for u in a) & full
        s_v = sum(_mix64(v ^ 0xC2B2AE3D27D4EB4F) for v in b) & full
        rot = ((s_v << 29) | (s_v >> 35)) & full
        size = (len(a) * 0x165667B19E3779F9 + len(b) * 0xD6E8FEB86659FD93) & full
        total += _mix64(s_u ^ rot ^ size)
        pairs.append((a, b))
    out = {"count": np.array([len(pairs)], dtype=np.int64),
           "hash": np.array([total & full], dtype=np.uint64).view(np.int64)}
    if case["kind"] == "list":
        out.update(_flat(sorted(pairs), _room(case)))
    return out
