"""Projected tuples are written as 8-byte words gathered from the columns:
texts of every length and alignment, between fixed-width columns, with NULLs.
kds_dst equals the oracle's byte for byte."""
import numpy as np
import pytest

from pgstrom import datagen, kds, xpuhip
from helpers import project_all_query, run_oracle_projection

pytestmark = pytest.mark.gpu


def _columns(n, maxlen, null_frac):
    r = np.random.default_rng(1000 * maxlen + n)
    null = lambda: r.random(n) < null_frac      # noqa: E731
    text = lambda: [bytes(r.integers(65, 91, size=k, dtype=np.uint8))     # noqa: E731
                    for k in r.integers(0, maxlen + 1, size=n)]
    return [kds.Column("a", "int2", r.integers(-9, 9, size=n).astype(np.int16), null()),
            kds.Column("t", "text", text(), null()),
            kds.Column("b", "bool", r.random(n) < 0.5, null()),
            kds.Column("u", "text", text(), null()),
            kds.Column("c", "int4", r.integers(-2**31, 2**31 - 1, size=n, dtype=np.int32), null()),
            kds.Column("d", "float8", r.standard_normal(n), null())]


def _compare(src, cols, jit, tuples=False):
    blob = project_all_query(cols)
    s = xpuhip.Session(blob)
    s.set_tuning(jit=jit)
    rc, dst, res, _ = s.exec(src, dst_length=8 << 20)
    s.close()
    assert rc == 0
    exp, ores = run_oracle_projection(blob, src, 8 << 20)
    assert np.array_equal(dst, exp)
    assert (res.nitems_in, res.nitems_out) == (ores.nitems_in, ores.nitems_out)


@pytest.mark.parametrize("null_frac", [0.0, 0.2])
@pytest.mark.parametrize("n,maxlen", [(1, 5), (63, 8), (65, 33), (257, 64), (1500, 130)])
def test_arrow_texts(gpu, jit, n, maxlen, null_frac):
    cols = _columns(n, maxlen, null_frac)
    _compare(kds.build_arrow_kds(cols), cols, jit)


def test_heap_texts(gpu, jit):
    cols = datagen.heap_table(700)
    _compare(kds.build_block_kds(cols), cols, jit)
