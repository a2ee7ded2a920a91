"""Device annealing with more workgroups than a wave has lanes, and several
words a block: the same chain as the host-stepped loop, step counts around the
end of a launch."""
import numpy as np
import pytest

import odp_amd as odp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,d,steps", [
    (2080, 3, 70),      # 65 blocks: one slot past a wave's lanes
    (512, 70, 40),      # rows of more than 64 entries (searched in two looks)
    (4100, 6, 530),     # 129 blocks, a tag that wraps past 511
    (64, 3, 520),       # two blocks
])
def test_device_chain_equals_host_chain(monkeypatch, n, d, steps):
    base = odp.generate_regular(n, d, 9)
    got = {}
    for where in ("host", "device"):
        monkeypatch.setenv("ODP_HIP_ANNEAL", where)
        odp.init_aspl_general(n, d)
        try:
            got[where] = odp.anneal(base, steps, 20.0, 0.2, False, False, 4)
        finally:
            odp.finalize_aspl()
    assert np.array_equal(got["host"][0], got["device"][0])
    for key in ("steps", "accepted", "best_diameter", "best_sum", "best_ASPL", "diameter", "ASPL", "optimum"):
        assert got["host"][1][key] == got["device"][1][key], key
