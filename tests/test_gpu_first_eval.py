"""The first evaluation of an Init under a plan with row parts: its own levels
first, frontier levels past the sixteenth.  Every result against the oracle."""
from functools import lru_cache

import numpy as np
import pytest

import odp_amd as odp
import oracle

pytestmark = pytest.mark.gpu

PARTS = dict(plan=odp.PLAN_LEVEL, kw=16, upw=8, seg_major=0, xcd=1, direct=-1, parts=4)


def same(a, b):
    return a[0] == b[0] and a[1] == b[1] and np.float64(a[2]).tobytes() == np.float64(b[2]).tobytes()


@lru_cache(None)
def graph(kind):
    if kind == "random":
        a = odp.generate_regular(2100, 4, 3)
    elif kind == "two components":
        n = 1400
        v = np.arange(n)[:, None]
        half = n // 2
        a = (v // half) * half + (v % half + np.array([[1, -1, 2, -2]])) % half
    elif kind == "one way":            # the last entry leads on only
        n = 1300
        a = (np.arange(n)[:, None] + np.array([[1, -1, 9]])) % n
    else:                              # ring: n // 4 levels of 1, 2
        n = int(kind)
        a = (np.arange(n)[:, None] + np.array([[1, -1, 2, -2]])) % n
    a = np.ascontiguousarray(a, np.int32)
    return a, oracle.evaluate(a, nodes=len(a))


# 64 levels end on a batch's edge; 16, 17 and 18 around the change; 300 past the counter ring
@pytest.mark.parametrize("kind", ["random", "two components", "one way", "64", "68", "72", "76", "256", "1100", "1200"])
@pytest.mark.parametrize("group", [0, 1])
def test_first_evaluation(kind, group):
    a, want = graph(kind)
    odp.init_aspl_general(len(a), a.shape[1])
    try:
        odp.set_plan(**dict(PARTS, group=group))
        for rep in range(3):
            assert same(odp.set_aspl(a), want), (kind, rep)
    finally:
        odp.finalize_aspl()


def test_first_evaluation_timed():
    """Per-launch timing of a first evaluation: levels of both kinds (64, of
    which k_direct runs at most 8)."""
    a, want = graph("256")
    odp.init_aspl_general(len(a), a.shape[1])
    try:
        odp.set_plan(**PARTS)
        odp.stats_enable(True)
        odp.stats_reset()
        assert same(odp.set_aspl(a), want)
        st = odp.stats()
        assert st["level_launches"] + st["idle_launches"] >= 64 - 8 and st["level_bytes"] > 0
    finally:
        odp.stats_enable(False)
        odp.finalize_aspl()
