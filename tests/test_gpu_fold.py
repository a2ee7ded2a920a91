"""Folded and thin gather levels (k_pgather, k_thin, k_thin2) against the oracle.

Folded levels run one unit of each pair across the bit matrix's diagonal and
store both; they hold for symmetric tables only, so tables that are not must
take every unit.  Thin levels take part of the neighbours of the level before
the expected last one, so graphs whose level count differs from the last
evaluation's, and lists too short for what is left, must fall back.  Every
result is an integer (or a double from integers): equality, no tolerance.
"""
import functools

import numpy as np
import pytest

import odp_amd as odp
import oracle

pytestmark = pytest.mark.gpu

LEV = odp.PLAN_LEVEL


def plan(parts=4, direct=-1, group=0):
    return dict(plan=LEV, kw=16, upw=8, seg_major=0, xcd=1, direct=direct, parts=parts, group=group)


def ring(n, d):
    """circulant graph of many levels: vertex v next to v +- 1 .. d/2 - 1 and v +- n/40"""
    k = np.array(list(range(1, d // 2)) + [n // 40])
    return ((np.arange(n)[:, None] + np.concatenate([k, -k])[None, :]) % n).astype(np.int32)


@functools.lru_cache(maxsize=None)
def fold_graphs(n, d):
    a, b = odp.generate_regular(n, d, 31), odp.generate_regular(n, d, 32)
    c = np.random.default_rng(33).integers(0, n, size=(n, d)).astype(np.int32)
    c[:, 0] = (np.arange(n) + 1) % n                             # not symmetric, strongly connected
    e = a.copy()
    e[n // 2, 0] = e[n // 2, 1]                                  # one entry: no longer symmetric
    graphs = dict(a=a, b=b, c=c, e=e)
    return graphs, {k: oracle.evaluate(t, nodes=n) for k, t in graphs.items()}


@functools.lru_cache(maxsize=None)
def guess_graphs(n, d):
    graphs = [odp.generate_regular(n, d, 51), odp.generate_regular(n, d, 52), ring(n, d)]
    near, rng = graphs[0].copy(), odp.Rng(54)                    # a few moves away
    for _ in range(40):
        odp.two_opt(near, rng)
    half = odp.generate_regular(n // 2, d, 53)
    graphs += [near, np.concatenate([half, half + n // 2]).astype(np.int32)]       # the last: two components
    return graphs, [oracle.evaluate(g, nodes=n) for g in graphs]


# rows: one block, an even and an odd number of blocks, one row past a block,
# a partial last block, sizes that leave pieces of the last round without rows
@pytest.mark.parametrize("n,d", [(1024, 6), (2048, 8), (2049, 8), (3000, 11), (4096, 5), (5001, 4), (9217, 6)])
@pytest.mark.parametrize("parts,direct", [(4, -1), (2, 0)])
def test_folded_levels(n, d, parts, direct):
    graphs, want = fold_graphs(n, d)
    a = graphs["a"]
    odp.init_aspl_general(n, d)
    try:
        odp.set_plan(**plan(parts, direct))
        for name in "aaaabbeaeeccca":
            assert odp.set_aspl(graphs[name]) == want[name], name
        # swaps on the device keep a symmetric table so
        odp.upload_adjacency(a)
        host, rng = a.copy(), odp.Rng(5)
        for _ in range(3):
            assert odp.swap_device(*odp.two_opt(host, rng)) == 0
            assert odp.set_aspl_resident() == oracle.evaluate(host, nodes=n)
    finally:
        odp.finalize_aspl()


def test_folded_levels_num_degrees():
    """Entries past num_degrees: device swaps that touch them change the
    adjacency alone, and the table is checked again."""
    n, d = 3000, 8
    a = odp.generate_regular(n, d, 41)
    nd = np.full(n, d, np.int32)
    for v in range(0, n, 7):                                     # cut edges on one side or on both
        nd[v] = d - 1
    want = oracle.evaluate(a, nodes=n, num_degrees=nd)
    odp.init_aspl_general(n, d, nd)
    try:
        odp.set_plan(**plan())
        for _ in range(4):
            assert odp.set_aspl(a) == want
        host, rng = a.copy(), odp.Rng(6)
        for _ in range(6):
            assert odp.swap_device(*odp.two_opt(host, rng)) == 0
            assert odp.set_aspl_resident() == oracle.evaluate(host, nodes=n, num_degrees=nd)
    finally:
        odp.finalize_aspl()


@pytest.mark.parametrize("cap", [None, "0", "70"])
@pytest.mark.parametrize("group", [0, 2])
def test_thin_levels_wrong_guess(cap, group, monkeypatch):
    """Graphs of few and of many levels on one evaluator, the guess wrong both
    ways, with lists that hold everything, nothing, or one entry a sub-list."""
    if cap is not None:
        monkeypatch.setenv("ODP_HIP_LIST_CAP", cap)
    n, d = 3000, 8
    graphs, want = guess_graphs(n, d)
    odp.init_aspl_general(n, d)
    try:
        odp.set_plan(**plan(group=group))
        for i in (0, 0, 0, 0, 1, 1, 3, 3, 4, 0, 0, 0, 2, 0, 0, 4, 1, 1, 1):
            assert odp.set_aspl(graphs[i]) == want[i], i
    finally:
        odp.finalize_aspl()
