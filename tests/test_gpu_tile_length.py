"""The longest entry of a large grid table, measured on the device before the
evaluation that needs it: results equal the oracle's and the tiles run the
levels per launch that the length allows, also after uploads that
change it."""
import numpy as np
import pytest

import odp_amd as odp
import oracle
from test_gpu_tile import TILE_PLAN, lmax_of, same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,d,s,lengths", [
    (130, 130, 4, 1, (3, 9, 2)),       # odd halves; 67600 entries
    (100, 100, 8, 4, (6, 3, 12)),      # 20000 entries of a first quadrant
    (98, 86, 6, 2, (3, 20, 4)),        # 25284; 20 is past the halo (one level a launch)
])
def test_length_follows_uploads(w, h, d, s, lengths):
    if s == 1:
        odp.init_aspl_grid(w, h, d)
    else:
        odp.init_aspl_grid_s(w, h, d, None, s)
    try:
        odp.set_plan(**TILE_PLAN)
        for i, length in enumerate(lengths):
            full = odp.generate_grid(w, h, d, length, s, 3 + i)
            base = full if s == 1 else odp.grid_base_table(w, h, d, s, full)
            want = oracle.evaluate(base, width=w, height=h, symmetries=s)
            for rep in range(3):
                if rep == 2:
                    odp.stats_enable(True)
                    odp.stats_reset()
                assert same(odp.set_aspl(base), want), (length, rep)
            st = odp.stats()
            odp.stats_enable(False)
            k = min(8, 16 // lmax_of(full, h))
            launches = st["level_launches"] + st["idle_launches"]
            if k:
                assert launches <= (want[0] - 1) // k + 2, (length, launches)
            else:
                assert launches >= want[0] - 6, (length, launches)
    finally:
        odp.stats_enable(False)
        odp.finalize_aspl()
