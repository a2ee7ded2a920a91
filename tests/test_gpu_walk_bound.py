"""The walked levels of the resident plan with their cost rule turned down
(ODP_HIP_RES_WALK_COST): a level with more walks than the kernel's 24-bit decoding
holds is pulled, whatever the rule says."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# circulant, 125 levels: its walks would go on to the eighth step; 32 * 16^5
# prefixes (the sixth level's) are past 2^24, 32 * 16^4 are not
CODE = """
import numpy as np, odp_amd as odp, oracle
n = 2000
k = np.arange(1, 9)
a = ((np.arange(n)[:, None] + np.concatenate([k, -k])[None, :]) % n).astype(np.int32)
odp.init_aspl_general(n, 16)
assert odp.get_plan()["plan"] == odp.PLAN_RESIDENT and odp.get_plan()["wb"] == 1
got = [odp.set_aspl(a) for _ in range(2)]
odp.finalize_aspl()
want = oracle.evaluate(a, nodes=n)
assert got == [want, want], (got, want)
print("equal")
"""


@pytest.mark.parametrize("cost", ["1", "1e-9"])
def test_cheap_walks(cost):
    env = dict(os.environ, ODP_HIP_RES_WALK_COST=cost,
               PYTHONPATH=os.pathsep.join([ROOT, os.path.join(ROOT, "oracle")]))
    r = subprocess.run([sys.executable, "-c", CODE], capture_output=True, text=True, timeout=100, env=env)
    assert r.returncode == 0 and "equal" in r.stdout, (r.stdout, r.stderr)
