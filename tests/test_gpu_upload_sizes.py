"""Tables read from host memory by the kernel that builds the neighbour table:
both sides of the size limits, with symmetry, with rows of uneven degree (the
device copy holds the entries past num_degrees too), and moves afterwards."""
import numpy as np
import pytest

import odp_amd as odp
import oracle

pytestmark = pytest.mark.gpu


def same(a, b):
    return a[0] == b[0] and a[1] == b[1] and np.float64(a[2]).tobytes() == np.float64(b[2]).tobytes()


def ring(n, d):
    """+-1, +-3, +-9 ...: a few levels; entry order differs from row to row."""
    steps = np.array([s * (3 ** k) for k in range(d // 2) for s in (1, -1)])
    a = (np.arange(n)[:, None] + steps[None, :]) % n
    return np.ascontiguousarray(np.take_along_axis(a, (np.arange(d)[None, :] + np.arange(n)[:, None]) % d, 1), np.int32)


@pytest.mark.parametrize("n,d", [(5460, 12), (5462, 12), (9000, 14)])      # 256 KiB and a row more; 492 KiB
def test_upload_sizes(n, d):
    a = ring(n, d)
    b = np.ascontiguousarray(a[:, ::-1])
    want = oracle.evaluate(a, nodes=n)
    odp.init_aspl_general(n, d)
    try:
        for t in (a, b, a):
            assert same(odp.set_aspl(t), want)
        assert same(odp.set_aspl_resident(), want)
    finally:
        odp.finalize_aspl()


def test_upload_uneven_rows():
    n, d = 6000, 12
    a = ring(n, d)
    nd = np.full(n, d, np.int32)
    for r in range(0, n - 1, 14):      # without the edge r, r + 1: both rows end with it, past num_degrees
        for x, y in ((r, r + 1), (r + 1, r)):
            k = int(np.nonzero(a[x] == y)[0][0])
            a[x, k], a[x, d - 1] = a[x, d - 1], y
            nd[x] = d - 1
    want = oracle.evaluate(a, nodes=n, num_degrees=nd)
    odp.init_aspl_general(n, d, nd)
    try:
        for _ in range(2):
            assert same(odp.set_aspl(a), want)
        assert same(odp.set_aspl_resident(), want)
    finally:
        odp.finalize_aspl()


@pytest.mark.parametrize("s", [2, 4])
def test_upload_symmetric(s):
    n, d = 12000 * 2, 8                # base tables of 375 and 187 KiB
    base = odp.generate_general_s(n, d, s, 3)
    want = oracle.evaluate(base, nodes=n, symmetries=s)
    odp.init_aspl_general_s(n, d, None, s)
    try:
        for _ in range(2):
            assert same(odp.set_aspl(base), want)
    finally:
        odp.finalize_aspl()
