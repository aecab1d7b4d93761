"""The read-outs' helper threads and pinned slots go with the last run, also
where a mpic_create has failed for lack of memory in between."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

CODE = """
import os, numpy as np, mandor3_amd as ma
def threads():
    return len(os.listdir("/proc/self/task"))
def run():
    r = ma.Run((60, 60, 60), (.05,) * 3, (3.,) * 3, .012, (0,) * 6)
    z = np.ones(3 * r.nodes)
    r.set_fields(z, z)
    assert r.fields()[0].sum() == z.size
    return r
r = run()
r.close()
base = threads()
r = run()
with_helpers = threads()
assert with_helpers == base + 5, (base, with_helpers)     # six chunks of one slot
try:
    ma.Run((2000, 2000, 1100), (.05,) * 3, (100., 100., 55.), .012, (0,) * 6)   # 528 GB
    raise SystemExit("created")
except ma.MpicError:
    pass
r.close()
assert threads() == base, (base, threads())
run().close()
assert threads() == base, (base, threads())
"""


def test_helpers_go_with_the_last_run():
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    p = subprocess.run([sys.executable, "-c", CODE], cwd=root, timeout=60, capture_output=True, text=True)
    assert p.returncode == 0, p.stderr
