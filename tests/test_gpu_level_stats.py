"""The bytes ODPX_Stats reports for gather levels are those of the work they did:
a folded level gathers for one unit of each pair across the diagonal (of T
blocks, T (T + 1) / 2 units of T^2) and writes every row."""
import numpy as np
import pytest

import odp_amd as odp
import oracle

pytestmark = pytest.mark.gpu

PARTS = dict(plan=odp.PLAN_LEVEL, kw=16, upw=8, seg_major=0, xcd=1, direct=-1, parts=4)


# every block of these graphs ends at the same level, so each launch that did work did all of it
@pytest.mark.parametrize("n,d,symmetric", [(2048, 6, True), (2048, 6, False), (3072, 8, True), (4096, 8, True)])
@pytest.mark.parametrize("fold", [1, 0])
def test_level_bytes(n, d, symmetric, fold, monkeypatch):
    if not fold:
        monkeypatch.setenv("ODP_HIP_FOLD", "0")
    a = odp.generate_regular(n, d, 61)
    if not symmetric:
        a = np.random.default_rng(33).integers(0, n, size=(n, d)).astype(np.int32)
        a[:, 0] = (np.arange(n) + 1) % n
    blocks = n // 1024
    share = (blocks + 1) / (2 * blocks) if symmetric and fold else 1
    want = oracle.evaluate(a, nodes=n)
    odp.init_aspl_general(n, d)
    try:
        odp.set_plan(**PARTS)
        odp.stats_enable(True)
        odp.stats_reset()
        for _ in range(3):
            assert odp.set_aspl(a) == want
        st = odp.stats()
        row = 1024 // 8
        level = blocks * n * (share * ((d + 1) * row + 4 * d) + row)
        assert st["level_launches"] > 0
        assert st["level_bytes"] == pytest.approx(st["level_launches"] * level, rel=1e-12)
        assert st["level_min_bytes"] == pytest.approx(st["level_launches"] * (blocks * n * 2 * row + n * d * 4), rel=1e-12)
    finally:
        odp.stats_enable(False)
        odp.finalize_aspl()
