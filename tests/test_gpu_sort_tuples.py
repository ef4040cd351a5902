"""GPU-Sort over group tuples that end within, at and beyond the 128 bytes a
wave stages of each: text keys of 0 to 60 characters in one buffer, waves with
short tuples only and waves with a long one, item counts around a wave and a
tile.  The order equals the oracle's."""
import numpy as np
import pytest

from pgstrom import abi, codegen as cg, kds
from helpers import run_gpu_groupby, run_oracle_groupby

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("maxlen", [6, 60])
@pytest.mark.parametrize("ngroups", [2, 64, 65, 257, 5000])
def test_order_over_text_keyed_groups(gpu, jit, ngroups, maxlen):
    r = np.random.default_rng(ngroups + maxlen)
    n = 3 * ngroups
    texts = [b"%05d" % i + b"x" * int(k) for i, k in enumerate(r.integers(0, maxlen - 4, size=ngroups))]
    pick = np.concatenate([np.arange(ngroups), r.integers(0, ngroups, size=n - ngroups)])
    cols = [kds.Column("key", "text", [texts[i] for i in pick]),
            kds.Column("v", "int8", r.integers(-10**9, 10**9, size=n, dtype=np.int64)),
            kds.Column("x", "int4", r.integers(-50, 50, size=n, dtype=np.int32), r.random(n) < 0.3)]
    plan = cg.Plan([(c.name, c.typname) for c in cols])
    key, v, x = (plan.scan_var(k) for k in ("key", "v", "x"))
    plan.set_groupby([(abi.KAGG_ACTION__NROWS_ANY, None, ("n", "int8")),
                      (abi.KAGG_ACTION__PMAX_INT32, x, ("mx", "bytea")),
                      (abi.KAGG_ACTION__PSUM_INT64, v, ("sv", "bytea")),
                      (abi.KAGG_ACTION__VREF, key, ("key", "text"))])
    # max(x) has ties and NULLs, sum(v) breaks them
    blob = plan.build(final_nrows=5000,
                      sort_keys=[(abi.KSORT_KEY_KIND__PMINMAX_INT64, 2, None, True, False),
                                 (abi.KSORT_KEY_KIND__PSUM_NUMERIC, 3, None, False, True)])
    src = kds.build_arrow_kds(cols)
    got = [row[0][3] for row in kds.parse_row_kds(run_gpu_groupby(blob, [src], tuning=dict(jit=jit)))]
    exp = [row[0][3] for row in kds.parse_row_kds(run_oracle_groupby(blob, [src]))]
    assert got == exp
