"""A batch handed over and run in one call is sent in chunks of whole graphs
(from 4 MB, graphs in the packed array's order): its results, those of later
runs of the same batch (one chunk, ordered lists, replayed) and of a whole load
must be the oracle's integers, whatever lies between the graphs."""
import numpy as np
import pytest

import odp_amd as odp
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", ["packed", "gaps", "reversed"])
def test_chunks(order):
    # one graph fills several chunks and is past LDS, several are tiny
    sizes = [(4, 3), (700, 5), (41000, 8), (4096, 16), (12000, 24), (9, 4), (2500, 6), (16384, 8), (64, 3), (3000, 9)]
    gs = [odp.generate_regular(n, d, 3 + i) for i, (n, d) in enumerate(sizes + [(5000, 10)] * 20)]
    want = [oracle.evaluate(g, nodes=len(g)) for g in gs]
    nodes, degrees, offsets, packed = odp.pack(gs)
    if order != "packed":
        gap = 37 if order == "gaps" else 0
        at, offsets = gap, np.zeros(len(gs), np.int64)
        for k in range(len(gs)) if order == "gaps" else reversed(range(len(gs))):
            offsets[k] = at
            at += gs[k].size + gap
        packed = np.full(at, -7, np.int32)                       # what lies between belongs to no graph
        for k, g in enumerate(gs):
            packed[offsets[k]:offsets[k] + g.size] = g.ravel()
    assert packed.nbytes > 4 << 20

    def check(got):
        assert [(int(d), int(s), float(a)) for d, s, a in zip(*got)] == want

    p = (nodes, degrees, offsets, packed)
    try:
        check(odp.batch_eval(p))
        for _ in range(3):                                       # one chunk and balanced lists, then replayed
            check(odp.batch_run(len(gs)))
        check(odp.loop_run(len(gs), odp.PLAN_AUTO))
        check(odp.batch_eval(p))
        odp.batch_load(p)
        check(odp.batch_run(len(gs)))
    finally:
        odp.batch_release()
