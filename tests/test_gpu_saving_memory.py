"""MATRIX_SAVING bounds device memory where ODP_ASPL asks for it (32 blocks of 1024
sources at a time) and keeps every block where the size alone chose the kind and
the card has room; the results are the same."""
import ctypes

import pytest

import odp_amd as odp

pytestmark = pytest.mark.gpu

N, D = 100000, 4
BLOCK = 2 * N * 128                                              # both levels of a block's rows
OTHERS = 300 << 20                                               # table, pair lists, chunk lists (90 MB), and room


def free_bytes():
    hip = ctypes.CDLL("/opt/rocm/lib/libamdhip64.so")
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def evaluate(a):
    odp.init_aspl_general(64, 3)                                 # whatever the runtime takes by itself
    odp.finalize_aspl()
    before = free_bytes()
    odp.init_aspl_general(N, D)
    try:
        return odp.get_plan()["group"], odp.set_aspl(a), before - free_bytes()
    finally:
        odp.finalize_aspl()


def test_saving_group(monkeypatch):
    monkeypatch.delenv("ODP_ASPL", raising=False)
    a = odp.generate_regular(N, D, 5)
    assert odp.get_kind(N, D) == 2
    room = free_bytes() > 8 * 98 * BLOCK
    group, want, used = evaluate(a)
    assert group == (0 if room else 32)
    if room:
        assert used >= 98 * BLOCK
    monkeypatch.setenv("ODP_ASPL", "MATRIX_SAVING")
    assert odp.get_kind(N, D) == 2
    group, got, used = evaluate(a)
    assert group == 32 and got == want
    assert 32 * BLOCK <= used <= 32 * BLOCK + OTHERS
    monkeypatch.setenv("ODP_ASPL", "MATRIX")
    group, got, _ = evaluate(a)
    assert group == 0 and got == want
