"""A table shorter than the active Init's is refused by the Python binding: the
library would read past its end."""
import numpy as np
import pytest

import odp_amd as odp
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["general", "general_s", "grid", "grid_s"])
def test_short_table(kind):
    if kind == "general":
        full, kw, init = odp.generate_regular(128, 4, 3), dict(nodes=128), lambda: odp.init_aspl_general(128, 4)
    elif kind == "general_s":
        full = odp.generate_general_s(128, 4, 2, 3)
        kw, init = dict(nodes=128, symmetries=2), lambda: odp.init_aspl_general_s(128, 4, None, 2)
    elif kind == "grid":
        full = odp.generate_grid(12, 8, 4, 3, 1, 3)
        kw, init = dict(width=12, height=8), lambda: odp.init_aspl_grid(12, 8, 4)
    else:
        full = odp.grid_base_table(12, 8, 4, 2, odp.generate_grid(12, 8, 4, 3, 2, 3))
        kw = dict(width=12, height=8, symmetries=2)
        init = lambda: odp.init_aspl_grid_s(12, 8, 4, None, 2)
    want = oracle.evaluate(full, **kw)
    init()
    try:
        assert odp.set_aspl(full) == want
        for short in (full[:-1], full[:, :3], np.zeros((0, 4), np.int32)):
            for call in (odp.set_aspl, odp.upload_adjacency, odp.autotune, lambda t: odp.anneal(t, 1)):
                with pytest.raises(ValueError):
                    call(short)
        assert odp.set_aspl_resident() == want                   # nothing was uploaded
        assert odp.set_aspl(np.concatenate([full, full])) == want    # a longer one is read as far as it is needed
    finally:
        odp.finalize_aspl()
    odp.init_aspl_general(16, 3)                                 # a smaller Init takes smaller tables
    try:
        small = odp.generate_regular(16, 3, 1)
        assert odp.set_aspl(small) == oracle.evaluate(small, nodes=16)
    finally:
        odp.finalize_aspl()


def test_library_init():
    """An Init made on the library itself is judged by the library's size."""
    odp.init_aspl_general(64, 4)
    odp.load().ODP_Finalize_aspl()
    odp.load().ODP_Init_aspl_general(16, 3, None)
    try:
        small = odp.generate_regular(16, 3, 1)
        assert odp.set_aspl(small) == oracle.evaluate(small, nodes=16)
    finally:
        odp.finalize_aspl()
