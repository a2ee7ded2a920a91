"""What a program that uses this library has it do, as cases that can be timed.

A case is one call (or one loop of calls) of the public entry points on seeded
synthetic graphs:

  eval    ODP_Set_aspl on a graph the evaluator has not just seen: the whole
          table is handed over every call.  From a graph of 1024 vertices, where
          launches and latency count, to 100000 vertices, where the default
          kind becomes MATRIX_SAVING; even and odd sizes and degrees, sizes that
          no block or tile divides, few levels (large degree) and many (degree 4).
  grid    the same for symmetric and plain grid graphs with short edges, whose
          diameter is many times a random graph's.
  anneal  ODPX_Anneal: a simulated-annealing chain, one 2-opt move and one exact
          evaluation a step.
  batch   ODPX_Batch_eval: a set of candidate graphs of uneven size in one call.
  serve   ODPX_Serve_*: chains whose graphs stay on the device, moves submitted
          for every chain and taken back (a rejected candidate), until all
          results are there.

The library keeps one active evaluator (ODP_Init_* / ODP_Finalize), as the API
it implements does, and one server; a state notes which one it belongs to.
"""
import math
import os

import numpy as np
import torch

import odp_amd as odp


def listed():
    return [
        # a small graph of the order/degree problem, a new one every call: latency
        {"name": "eval n1024 d6", "family": "eval", "nodes": 1024, "degree": 6},
        # ordinary sizes; nothing divides 5001
        {"name": "eval n5001 d10", "family": "eval", "nodes": 5001, "degree": 10},
        {"name": "eval n16384 d16", "family": "eval", "nodes": 16384, "degree": 16},
        # odd degree, past the sizes where a block of 64 sources fits a CU
        {"name": "eval n30002 d7", "family": "eval", "nodes": 30002, "degree": 7},
        # the headline graph as a program gets to it: another graph every call
        {"name": "eval n65536 d16", "family": "eval", "nodes": 65536, "degree": 16},
        # a sparse graph: many levels, and an odd size
        {"name": "eval n49999 d4", "family": "eval", "nodes": 49999, "degree": 4},
        # past the size where the default kind is MATRIX_SAVING
        {"name": "eval n100000 d8", "family": "eval", "nodes": 100000, "degree": 8},
        # the 4-fold symmetric grid of the benchmark, 128 levels
        {"name": "grid 256x256 s4 d8 L4", "family": "grid", "width": 256, "height": 256, "degree": 8, "length": 4,
         "symmetries": 4, "kind": "MATRIX_SAVING"},
        # the annealing loops: small (many steps a second) and the headline size
        {"name": "anneal n1024 d6", "family": "anneal", "nodes": 1024, "degree": 6, "steps": 1000},
        {"name": "anneal n65536 d16", "family": "anneal", "nodes": 65536, "degree": 16, "steps": 8},
        # candidates of uneven size and degree in one call
        {"name": "batch 256 n1024-16384", "family": "batch", "graphs": 256, "low": 1024, "high": 16384},
        # chains of all the benchmark's sizes and degrees, small and large together
        {"name": "serve 9 chains", "family": "serve", "chains": 9, "large": 65536},
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    family = rng.choice(["eval", "eval", "eval", "eval", "grid", "anneal", "batch", "serve"])
    if family == "eval":
        n = _log(rng, 1000, 100000)
        d = rng.choice([3, 4, 5, 6, 7, 8, 10, 12, 16, 20, 24, 32] if n <= 65536 else [4, 5, 6, 8, 10])
        if n * d % 2:
            n += 1
        return {"family": family, "nodes": n, "degree": d}
    if family == "grid":
        s = rng.choice([1, 2, 4])
        w = 4 * (_log(rng, 24, 160 if s == 1 else 256) // 4)
        h = w if s == 4 else 4 * (_log(rng, 24, 160 if s == 1 else 256) // 4)
        length = rng.choice([3, 4, 5, 6])
        return {"family": family, "width": w, "height": h, "degree": rng.choice([4, 5, 6, 8]), "length": length,
                "symmetries": s, "kind": rng.choice(["MATRIX", "MATRIX_SAVING"])}
    if family == "anneal":
        n = 2 * (_log(rng, 512, 65536) // 2)
        d = rng.choice([4, 5, 6, 8, 10, 12, 16])
        return {"family": family, "nodes": n, "degree": d, "steps": max(4, min(500, int(4e5 / n)))}
    if family == "batch":
        low = _log(rng, 256, 4096)
        return {"family": family, "graphs": _log(rng, 16, 256), "low": low, "high": min(16384, low * rng.choice([2, 4, 16]))}
    return {"family": family, "chains": rng.randrange(3, 10), "large": 2 * (_log(rng, 24000, 65536) // 2)}


# ---- the one evaluator and the one server ------------------------------------

_now = {"key": None, "server": None}


def _key(case):
    f = case["family"]
    if f == "eval" or f == "anneal":
        return ("general", case["nodes"], case["degree"])
    if f == "grid":
        return ("grid", case["width"], case["height"], case["degree"], case["symmetries"], case["kind"])
    return (f, case.get("chains"), case.get("large"))


def _activate(case):
    """The evaluator or server that the case's states belong to, made if it is not the current one."""
    key = _key(case)
    if _now["key"] == key:
        return
    if _now["key"] is not None:
        if _now["key"][0] in ("general", "grid"):
            odp.finalize_aspl()
        elif _now["key"][0] == "batch":
            odp.batch_release()
        else:
            _now["server"].stop()
            _now["server"] = None
    _now["key"] = key
    if key[0] == "general":
        odp.init_aspl_general(case["nodes"], case["degree"])
    elif key[0] == "grid":
        before = os.environ.get("ODP_ASPL")
        os.environ["ODP_ASPL"] = case["kind"]
        odp.init_aspl_grid_s(case["width"], case["height"], case["degree"], None, case["symmetries"])
        if before is None:
            del os.environ["ODP_ASPL"]
        else:
            os.environ["ODP_ASPL"] = before
    elif key[0] == "serve":
        _now["server"] = odp.Server(small_slots=1, large_slots=2)


# ---- inputs --------------------------------------------------------------------

def _inputs(case, seed):
    """The case's graphs, from the seed alone."""
    f, at = case["family"], 1000 * (int(seed) % (1 << 40)) + 1
    if f in ("eval", "anneal"):
        return {"full": odp.generate_regular(case["nodes"], case["degree"], at)}
    if f == "grid":
        w, h, d, s = case["width"], case["height"], case["degree"], case["symmetries"]
        full = odp.generate_grid(w, h, d, case["length"], s, at)
        return {"full": full, "base": odp.grid_base_table(w, h, d, s, full) if s > 1 else full}
    rng, move = np.random.default_rng(at), odp.Rng(at)
    graphs, moves = [], []
    if f == "batch":
        for g in range(case["graphs"]):
            n = 2 * int(rng.integers(case["low"] // 2, case["high"] // 2 + 1))
            graphs.append(odp.generate_regular(n, int(rng.choice([4, 8, 12, 16, 24])), at + g))
            odp.two_opt(graphs[-1], move)
        return {"graphs": graphs}
    for c in range(case["chains"]):
        n, d = (4096, 16384, case["large"])[c % 3], (8, 16, 32)[c // 3 % 3]
        graphs.append(odp.generate_regular(n, d, at + c))
        after = graphs[-1].copy()
        moves.append((odp.two_opt(after, move), after))
    return {"graphs": graphs, "moves": moves}


def prepare(case, seed):
    f, got = case["family"], _inputs(case, seed)
    _activate(case)
    state = {"case": case}
    if f == "eval":
        state["adjacency"] = got["full"]
    elif f == "grid":
        state["adjacency"] = got["base"]
    elif f == "anneal":
        state["adjacency"], state["seed"] = got["full"], int(seed) % (1 << 31) + 1
    elif f == "batch":
        state["packed"] = odp.pack(got["graphs"])
    else:
        state["chains"] = [_now["server"].add_chain(g) for g in got["graphs"]]
        state["moves"] = [m for m, _ in got["moves"]]
    return state


def run(state):
    case = state["case"]
    f = case["family"]
    if f == "batch":
        return odp.batch_eval(state["packed"])
    if f == "serve":
        server, ids = _now["server"], []
        for chain, (a, b, c, d) in zip(state["chains"], state["moves"]):
            ids.append(server.submit(chain, [(a, b, c, d)]))      # the candidate
            ids.append(server.submit(chain, [(a, c, b, d)]))      # taken back
        server.drain()
        got = {r["id"]: r for r in server.poll()}
        got = [got[i] for i in ids]
        return (np.array([r["status"] for r in got]), np.array([r["diameter"] for r in got]),
                np.array([r["sum"] for r in got]), np.array([r["ASPL"] for r in got]))
    if f == "anneal":
        best, r = odp.anneal(state["adjacency"], case["steps"], seed=state["seed"])
        return (best, r["steps"], r["accepted"], r["best_diameter"], r["best_sum"], r["best_ASPL"], r["diameter"], r["ASPL"])
    return odp.set_aspl(state["adjacency"])


def work(case):
    """The tables read once and the results written once.  (The bit matrix between
    them is the method's own; its floor depends on the levels and is not counted.)"""
    f = case["family"]
    if f == "grid":
        b = 4 * case["width"] * case["height"] // case["symmetries"] * case["degree"] + 20
    elif f == "eval":
        b = 4 * case["nodes"] * case["degree"] + 20
    elif f == "anneal":
        b = 2 * 4 * case["nodes"] * case["degree"] + 44
    elif f == "batch":
        b = case["graphs"] * (int(4 * 12.8 * (case["low"] + case["high"]) / 2) + 36)
    else:
        b = sum((16 + 20) * 2 for _ in range(case["chains"]))
    return {"bytes": b, "flops": 0}


# ---- the same values in plain torch ---------------------------------------------

def _distances(full, sources):
    """(diameter, sum over unordered pairs, ASPL) of a connected graph given by its table,
    from the distances out of the first `sources` rows times rows/sources."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    adj = torch.from_numpy(np.ascontiguousarray(full)).to(dev).long()
    n, d = adj.shape
    ones = torch.tensor([bin(i).count("1") for i in range(256)], dtype=torch.int64, device=dev)
    total, diameter = 0, 0
    for lo in range(0, len(sources), 4096):
        src = torch.as_tensor(sources[lo:lo + 4096], device=dev)
        m = len(src)
        cur = torch.zeros((n, (m + 7) // 8), dtype=torch.uint8, device=dev)
        for bit in range(8):
            own = src[bit::8]
            cur[own, torch.arange(len(own), device=dev)] |= 1 << bit
        level = 0
        reached = m
        while reached < n * m:
            total += n * m - reached
            level += 1
            nxt = cur.clone()
            for j in range(d):
                nxt |= cur[adj[:, j]]
            cur = nxt
            reached = 0
            for part in cur.split(8192):
                reached += int(ones[part.long()].sum())
        diameter = max(diameter, level)
    pairs = total * (n // len(sources))
    return diameter, pairs // 2, pairs / ((n - 1.0) * n)


def exact(case, seed):
    f = case["family"]
    if f == "anneal":
        return None                     # a chain of decisions, not a value
    got = _inputs(case, seed)
    if f == "eval":
        return _distances(got["full"], np.arange(case["nodes"]))
    if f == "grid":
        w, h, s = case["width"], case["height"], case["symmetries"]
        cells = np.arange(w * h).reshape(w, h)
        cells = cells if s == 1 else cells[: w // 2] if s == 2 else cells[: w // 2, : h // 2]
        return _distances(got["full"], cells.reshape(-1).copy())
    if f == "batch":
        r = [_distances(g, np.arange(len(g))) for g in got["graphs"]]
    else:
        r = []
        for g, (_, after) in zip(got["graphs"], got["moves"]):
            r += [_distances(after, np.arange(len(g))), _distances(g, np.arange(len(g)))]
    d, s, x = (np.array(v) for v in zip(*r))
    return (d, s, x) if f == "batch" else (None, d, s, x)
