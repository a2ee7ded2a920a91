"""The paths that results alone do not show are taken: folded and thin levels,
thin levels whose guess is wrong or whose lists are short, batches sent in
chunks.  Every result against the oracle: equality, no tolerance."""
import functools

import numpy as np
import pytest

import odp_amd as odp
import oracle

pytestmark = pytest.mark.gpu


def plan(direct=-1, group=0):
    return dict(plan=odp.PLAN_LEVEL, kw=16, upw=8, seg_major=0, xcd=1, direct=direct, parts=4, group=group)


def ring(n, d):
    """circulant graph of many levels"""
    k = np.array(list(range(1, d // 2)) + [n // 40])
    return ((np.arange(n)[:, None] + np.concatenate([k, -k])[None, :]) % n).astype(np.int32)


@functools.lru_cache(maxsize=None)
def graphs(n, d):
    half = odp.generate_regular(n // 2, d, 53)
    one_way = np.random.default_rng(33).integers(0, n, size=(n, d)).astype(np.int32)
    one_way[:, 0] = (np.arange(n) + 1) % n                       # not symmetric, strongly connected
    g = dict(a=odp.generate_regular(n, d, 51), b=odp.generate_regular(n, d, 52), o=one_way)
    if d % 2 == 0 and n % 2 == 0:
        g.update(r=ring(n, d), h=np.concatenate([half, half + n // 2]).astype(np.int32))
    return g, {k: oracle.evaluate(t, nodes=n) for k, t in g.items()}


def gained(before):
    return {k: v - before[k] for k, v in odp.routes().items()}


# one block, one row past two blocks, an odd number, partial last blocks; tables
# of 12, 20 and 36 ids (k_thin looks at 16 at a time, k_thin2 at 64 pairs)
@pytest.mark.parametrize("n,d", [(1024, 6), (2049, 8), (2300, 11), (1300, 20), (4000, 33), (4096, 5), (5001, 4), (9217, 6)])
@pytest.mark.parametrize("direct", [-1, 0])
def test_folded_and_thin(n, d, direct, monkeypatch):
    monkeypatch.setenv("ODP_HIP_LIST_FRAC", "1000")              # lists whatever share is left
    g, want = graphs(n, d)
    odp.init_aspl_general(n, d)
    try:
        odp.set_plan(**plan(direct))
        at = odp.routes()
        for name in "aaaabba":
            assert odp.set_aspl(g[name]) == want[name], name
        got = gained(at)
        assert got["folded"] == 7 and got["thin"] >= 3 and got["thin_whole"] == 0, got
        at = odp.routes()
        for name in "oooo":                                      # not symmetric: thin levels of every unit
            assert odp.set_aspl(g[name]) == want[name], name
        assert gained(at)["folded"] == 0
    finally:
        odp.finalize_aspl()


# lists that hold everything, nothing, one entry a sub-list, ten; groups of two blocks of three (not folded)
@pytest.mark.parametrize("cap", [None, "0", "64", "640"])
@pytest.mark.parametrize("group", [0, 2])
def test_thin_wrong_guess(cap, group, monkeypatch):
    monkeypatch.setenv("ODP_HIP_LIST_FRAC", "1000")
    if cap is not None:
        monkeypatch.setenv("ODP_HIP_LIST_CAP", cap)
    n, d = 3000, 8
    g, want = graphs(n, d)
    odp.init_aspl_general(n, d)
    try:
        odp.set_plan(**plan(group=group))
        at = odp.routes()
        for i, name in enumerate("aaabbahaaraabroaarhab"):
            assert odp.set_aspl(g[name]) == want[name], (i, name)
        got = gained(at)
        assert got["thin"] > 0, got
        assert (got["thin_whole"] > 0) == (cap is not None), got
        if cap is None:
            assert got["thin_late"] > 0, got
        assert (got["folded"] > 0) == (group == 0), got
    finally:
        odp.finalize_aspl()


@pytest.mark.parametrize("order,chunked", [("packed", 1), ("gaps", 1), ("reversed", 0), ("small", 0)])
def test_chunks_sent(order, chunked):
    gs = [odp.generate_regular(n, 10, 3 + n) for n in ([5000] * 22 if order != "small" else [300] * 22)]
    want = [oracle.evaluate(gs[0], nodes=len(gs[0]))] * len(gs)
    nodes, degrees, offsets, packed = odp.pack(gs)
    if order == "reversed":
        offsets = offsets[::-1].copy()
    elif order == "gaps":
        at = gs[0].size + 5
        offsets = np.arange(len(gs), dtype=np.int64) * at
        packed = np.full(at * len(gs), -7, np.int32)
        for o, g in zip(offsets, gs):
            packed[o:o + g.size] = g.ravel()
    try:
        at = odp.routes()
        got = odp.batch_eval((nodes, degrees, offsets, packed))
        assert [(int(d), int(s), float(a)) for d, s, a in zip(*got)] == want
        assert gained(at)["chunked"] == chunked
    finally:
        odp.batch_release()
