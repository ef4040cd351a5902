"""XPUHIP_JIT_AUTO on small chunks: no call waits for the compiler.  A plan that
has run a million rows in small chunks is interpreted until a thread of the
library has compiled it, then specialised; a process may end meanwhile."""
import os
import subprocess
import sys
import time

import numpy as np
import pytest

from conftest import ROOT
from pgstrom import codegen as cg, datagen, kds, workloads as W, xpuhip
from helpers import assert_groups_equal, run_oracle_groupby, run_oracle_projection
from test_gpu_batch import ACTIONS

pytestmark = pytest.mark.gpu


def _until_specialised(call):
    """Runs the call until it ran specialised kernels (60 s at most)."""
    end = time.monotonic() + 60
    while time.monotonic() < end:
        call()
        if xpuhip.last_task_stats()["jit"]:
            return True
        time.sleep(0.05)
    return False


def test_scan_chunks(gpu):
    """k = 432,101 is no other test's constant: the plan is new here."""
    n = 300_000
    cols = datagen.scan_table(n)
    src = kds.build_arrow_kds(cols)
    blob = W.scan_query(cols, k=432_101)
    exp, _ = run_oracle_projection(blob, src, 32 << 20)

    def call():
        rc, dst, _, _ = s.exec(src, dst_length=32 << 20)
        assert rc == 0 and np.array_equal(dst, exp)

    s = xpuhip.Session(blob)
    for i in range(4):
        call()
        assert xpuhip.last_task_stats()["jit"] == 0, i      # the fourth has run a million rows
    assert _until_specialised(call)
    s.close()


def test_groupby_chunks(gpu):
    n = 600_000
    cols = datagen.preagg_table(n)
    src = kds.build_arrow_kds(cols)
    plan = cg.Plan([(c.name, c.typname) for c in cols])
    key, v, w, x = (plan.scan_var(k) for k in ("key", "v", "w", "x"))
    plan.scan_quals = cg.Func("int4gt", x, cg.Const("int4", -2_147_432_107))
    plan.set_groupby(W.preagg_tlist(plan, key, v, w, x))
    blob = plan.build(final_nrows=10_000)
    s = xpuhip.Session(blob)
    count = 0

    def call():
        nonlocal count
        assert s.exec(src)[0] == 0
        count += 1

    for i in range(2):
        call()
        assert xpuhip.last_task_stats()["jit"] == 0, i
    assert _until_specialised(call)
    s.reset()
    call()
    assert xpuhip.last_task_stats()["jit"] == 1
    assert_groups_equal(s.final(), run_oracle_groupby(blob, [src]), ACTIONS)
    s.close()


def test_large_chunk_is_specialised_at_once(gpu):
    n = 1_000_000
    cols = datagen.scan_table(n)
    s = xpuhip.Session(W.scan_query(cols, k=432_103))
    assert s.exec(kds.build_arrow_kds(cols), dst_length=96 << 20)[0] == 0
    assert xpuhip.last_task_stats()["jit"] == 1
    s.close()


@pytest.mark.parametrize("shutdown", [False, True])
def test_process_ends_while_compiling(gpu, shutdown):
    code = """
import sys
sys.path.insert(0, %r)
from pgstrom import datagen, kds, workloads as W, xpuhip
xpuhip.init(0)
cols = datagen.scan_table(300_000)
src = kds.build_arrow_kds(cols)
s = xpuhip.Session(W.scan_query(cols, k=432_105))
for _ in range(4):
    assert s.exec(src, dst_length=32 << 20)[0] == 0
assert xpuhip.last_task_stats()["jit"] == 0
if %r:
    s.close()
    xpuhip.lib().xpuhip_shutdown()
print("ended", flush=True)
""" % (os.path.join(ROOT, "pg-strom_amd"), shutdown)
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "ended" in r.stdout, (r.returncode, r.stderr[-2000:])
