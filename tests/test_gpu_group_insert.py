"""Insertion of groups into kds_final: group counts around the 64 entries a
wave merges at a time and around one LDS table, and text keys whose bytes
end at every offset of the 8-byte words their tuple is written in.  Groups
equal the oracle's, each once, with row ids 0..n-1."""
import numpy as np
import pytest

from pgstrom import abi, codegen as cg, datagen, kds, workloads as W, xpuhip
from helpers import assert_groups_equal, run_gpu_groupby, run_oracle_groupby

pytestmark = pytest.mark.gpu


def _check(cols, keys, jit):
    plan = cg.Plan([(c.name, c.typname) for c in cols])
    kv = [plan.scan_var(k) for k in keys]
    tlist = W.preagg_tlist(plan, kv[0], plan.scan_var("v"), plan.scan_var("w"), plan.scan_var("x"))
    tlist += [(abi.KAGG_ACTION__VREF, k, (n, k.typname)) for n, k in zip(keys[1:], kv[1:])]
    plan.set_groupby(tlist)
    blob = plan.build(final_nrows=5000)
    src = kds.build_arrow_kds(cols)
    fin = run_gpu_groupby(blob, [src, src], tuning=dict(jit=jit))
    exp = run_oracle_groupby(blob, [src, src])
    got = assert_groups_equal(fin, exp, [a for a, _, _ in tlist])
    assert sorted(r for _, r in kds.parse_row_kds(fin)) == list(range(len(got)))


def _args(n, r):
    return [kds.Column("v", "int8", r.integers(-1000, 1_000_000, size=n, dtype=np.int64)),
            kds.Column("w", "float8", r.random(n)),
            kds.Column("x", "int4", r.integers(-2**31, 2**31 - 1, size=n, dtype=np.int32))]


@pytest.mark.parametrize("ngroups", [1, 63, 64, 65, 127, 129, 512, 3993, 9001])
def test_group_counts(gpu, jit, ngroups):
    r = np.random.default_rng(ngroups)
    n = 3 * ngroups + 5
    key = np.concatenate([np.arange(ngroups), r.integers(0, ngroups, size=n - ngroups)])
    _check([kds.Column("key", "int4", key.astype(np.int32))] + _args(n, r), ["key"], jit)


@pytest.mark.parametrize("second", [None, "int2"])
def test_text_keys_of_every_length(gpu, jit, second):
    r = np.random.default_rng(5)
    n = 6000
    texts = [bytes(97 + (i + j) % 26 for j in range(i % 41)) for i in range(300)]
    null = r.random(n) < 0.05
    cols = [kds.Column("key", "text", [texts[i] for i in r.integers(0, 300, size=n)], null)]
    keys = ["key"]
    if second:
        cols.append(kds.Column("k2", "int2", r.integers(-2, 3, size=n).astype(np.int16),
                               r.random(n) < 0.1))
        keys.append("k2")
    _check(cols + _args(n, r), keys, jit)


@pytest.mark.parametrize("lds_nents", [64, 1024, 2000])
def test_partitions_with_more_groups_than_a_table(gpu, jit, lds_nents):
    """Spilled rows and dumps of 150,000 groups: a dump partition holds about
    600 of them, fewer or more than the table it is folded in."""
    r = np.random.default_rng(lds_nents)
    n = 300_000
    key = np.concatenate([np.arange(150_000), r.integers(0, 150_000, size=n - 150_000)])
    cols = [kds.Column("key", "int4", r.permutation(key).astype(np.int32))] + _args(n, r)
    plan = cg.Plan([(c.name, c.typname) for c in cols])
    tlist = W.preagg_tlist(plan, *[plan.scan_var(k) for k in ("key", "v", "w", "x")])
    plan.set_groupby(tlist)
    blob = plan.build(final_nrows=150_000)
    src = kds.build_arrow_kds(cols)
    fin = run_gpu_groupby(blob, [src], tuning=dict(jit=jit, lds_nents=lds_nents))
    assert_groups_equal(fin, run_oracle_groupby(blob, [src]), [a for a, _, _ in tlist])


@pytest.mark.parametrize("graph", [False, True])
def test_batch_of_uneven_fragments(gpu, jit, graph):
    """Fragments of 1 to 200,000 rows and 1 to 10,000 groups in one launch,
    run twice: each equals its session alone."""
    r = np.random.default_rng(8)
    sizes = [(1, 3), (64, 1), (4097, 9000), (70_001, 17), (200_000, 100_000)]
    base = 200_000
    cols = datagen.preagg_table(base)
    cols = [kds.Column("a", "int4", r.integers(0, 1_000_000, size=base, dtype=np.int32))] + cols
    chunk = kds.build_arrow_kds(cols)
    hdrs = kds.window_headers(chunk, [(0, n) for n, _ in sizes], len(sizes) * 1024, 1024)
    dev = xpuhip.DeviceBuffer(len(hdrs) + len(chunk), np.concatenate([hdrs, chunk]))
    acts = [a for a, _, _ in W.preagg_tlist(None, cols[1], None, None, None)]
    tasks, alone = [], []
    for i, (n, m) in enumerate(sizes):
        blob = W.fragment_query(cols, k=700_000, m=m)
        s = xpuhip.Session(blob)
        s.set_tuning(jit=jit, lds_nents=1024)
        tasks.append((s, dev.ptr + i * 1024, n))
        part = kds.build_arrow_kds(datagen.take_rows(cols, np.arange(base) < n))
        alone.append(run_oracle_groupby(blob, [part, part]))
    for _ in range(2):
        xpuhip.batch_exec(tasks, graph=graph)
    for (s, _, _), exp in zip(tasks, alone):
        assert_groups_equal(s.final(), exp, acts)
        s.close()
    dev.free()


@pytest.mark.parametrize("lds_nents", [96, 1500])
def test_text_groups_beyond_a_table(gpu, jit, lds_nents):
    """Text keys name their group by a row of the chunk through spill records
    and dumps: 20,000 texts that share prefixes, some of one byte, and an int4
    key beside them, over heap pages and an Arrow chunk."""
    r = np.random.default_rng(lds_nents)
    n = 60_000
    pick = r.integers(0, 20_000, size=n)
    cols = [kds.Column("key", "text", [b"prefix-of-many-%d" % i if i > 200 else b"%c" % (32 + i % 90)
                                       for i in pick], r.random(n) < 0.01),
            kds.Column("k2", "int4", (pick % 3).astype(np.int32), r.random(n) < 0.01)] + _args(n, r)
    plan = cg.Plan([(c.name, c.typname) for c in cols])
    kv = [plan.scan_var("key"), plan.scan_var("k2")]
    tlist = W.preagg_tlist(plan, kv[0], *[plan.scan_var(k) for k in ("v", "w", "x")])
    tlist.append((abi.KAGG_ACTION__VREF, kv[1], ("k2", "int4")))
    plan.set_groupby(tlist)
    blob = plan.build(final_nrows=20_000)
    src = kds.build_arrow_kds(cols)
    exp = run_oracle_groupby(blob, [src])
    for chunk in (src, kds.build_block_kds(cols)):
        fin = run_gpu_groupby(blob, [chunk], tuning=dict(jit=jit, lds_nents=lds_nents))
        assert_groups_equal(fin, exp, [a for a, _, _ in tlist])


@pytest.mark.parametrize("lds_nents", [64, 1200])
@pytest.mark.parametrize("null_frac", [0.05, 0.9])
def test_null_arguments_through_the_tables(gpu, jit, lds_nents, null_frac):
    """Arguments with validity bitmaps: NULLs are counted per entry in the
    tables, spill records and dumps (every action that skips a NULL), and one
    column of the chunk is NULL throughout."""
    r = np.random.default_rng(int(100 * null_frac) + lds_nents)
    n = 40_000
    a = _args(n, r)
    for c in a[:2]:
        c.nulls = r.random(n) < null_frac
    a[2].nulls = np.ones(n, dtype=bool)
    cols = [kds.Column("key", "int4", r.integers(0, 3000, size=n).astype(np.int32),
                       r.random(n) < 0.05)] + a
    plan = cg.Plan([(c.name, c.typname) for c in cols])
    key, v, w, x = (plan.scan_var(k) for k in ("key", "v", "w", "x"))
    tlist = [(abi.KAGG_ACTION__NROWS_ANY, None, ("n", "int8")),
             (abi.KAGG_ACTION__NROWS_COND, v, ("nv", "int8")),
             (abi.KAGG_ACTION__PSUM_INT64, v, ("sv", "bytea")),
             (abi.KAGG_ACTION__PMIN_INT64, v, ("mv", "bytea")),
             (abi.KAGG_ACTION__STDDEV, w, ("dw", "bytea")),
             (abi.KAGG_ACTION__PMAX_FP64, w, ("xw", "bytea")),
             (abi.KAGG_ACTION__PSUM_INT, x, ("sx", "bytea")),
             (abi.KAGG_ACTION__PMAX_INT32, x, ("xx", "bytea")),
             (abi.KAGG_ACTION__VREF, key, ("key", "int4"))]
    plan.set_groupby(tlist)
    blob = plan.build(final_nrows=3000)
    src = kds.build_arrow_kds(cols)
    fin = run_gpu_groupby(blob, [src], tuning=dict(jit=jit, lds_nents=lds_nents))
    # sums of squares of uniform [0, 1) values: addends of one sign
    assert_groups_equal(fin, run_oracle_groupby(blob, [src]), [t[0] for t in tlist])


def test_batch_of_text_keys(gpu, jit):
    """Fragments grouped by a text column in one launch: entries name rows of
    their own fragment's window."""
    r = np.random.default_rng(4)
    n = 30_000
    cols = [kds.Column("key", "text", [b"k%d" % i for i in r.integers(0, 4000, size=n)],
                       r.random(n) < 0.02)] + _args(n, r)
    cols[2].nulls = r.random(n) < 0.1
    blob = W.preagg_query(cols)
    acts = [a for a, _, _ in W.preagg_tlist(None, cols[0], None, None, None)]
    wins = [(0, 30_000), (64, 1), (8_000, 9_999)]
    chunk = kds.build_arrow_kds(cols)
    hdrs = kds.window_headers(chunk, wins, len(wins) * 1024, 1024)
    dev = xpuhip.DeviceBuffer(len(hdrs) + len(chunk), np.concatenate([hdrs, chunk]))
    sess = [xpuhip.Session(blob) for _ in wins]
    for s in sess:
        s.set_tuning(jit=jit, lds_nents=1024)
    xpuhip.batch_exec([(s, dev.ptr + i * 1024, w[1]) for i, (s, w) in enumerate(zip(sess, wins))],
                      graph=False)
    for s, (r0, m) in zip(sess, wins):
        keep = (np.arange(n) >= r0) & (np.arange(n) < r0 + m)
        part = kds.build_arrow_kds(datagen.take_rows(cols, keep))
        assert_groups_equal(s.final(), run_oracle_groupby(blob, [part]), acts)
        s.close()
    dev.free()


@pytest.mark.parametrize("third", ["text", "numeric"])
def test_null_keys_before_variable_length_keys(gpu, jit, third):
    """Groups that differ in which of their int8 keys is NULL hash alike (NULLs
    stay out of the hash) and share a chain: a walk compares each with the
    others' tuples, whose texts and numerics lie behind different bytes.  The
    int8 values are timestamps in microseconds, whose bytes would be lengths of
    hundreds of MB.  Each group is there once, over heap pages and (no
    numeric) an Arrow chunk."""
    r = np.random.default_rng(6)
    n = 20_000
    base = 1_733_400_000_000_000 + r.integers(0, 12, size=n)
    which = r.integers(0, 4, size=n)
    pick = r.integers(0, 9, size=n)
    short = third == "numeric"
    var = [kds.numeric_image(str(i % 3) + ".25", short_varlena=True) if short else b"x" * (i % 3)
           for i in pick]
    cols = [kds.Column("a", "int8", base, (which & 1) != 0),
            kds.Column("d", "int8", base, (which & 2) != 0),
            kds.Column("t", third, var, r.random(n) < 0.1),
            kds.Column("u", "text", [b"y" * (i // 3) for i in pick], r.random(n) < 0.1),
            kds.Column("e", "int8", base + which, r.random(n) < 0.5)] + _args(n, r)
    names = ["a", "d", "t", "u", "e"]
    plan = cg.Plan([(c.name, c.typname) for c in cols])
    tlist = [(abi.KAGG_ACTION__NROWS_ANY, None, ("n", "int8")),
             (abi.KAGG_ACTION__PSUM_INT64, plan.scan_var("v"), ("sv", "bytea"))]
    tlist += [(abi.KAGG_ACTION__VREF, plan.scan_var(k), (k, third if k == "t" else c.typname))
              for k, c in zip(names, cols)]
    plan.set_groupby(tlist)
    blob = plan.build(final_nrows=5000)
    chunks = [kds.build_block_kds(cols)] + ([] if short else [kds.build_arrow_kds(cols)])
    for src in chunks:
        fin = run_gpu_groupby(blob, [src, src], tuning=dict(jit=jit))
        got = assert_groups_equal(fin, run_oracle_groupby(blob, [src, src]), [t[0] for t in tlist])
        assert len(got) > 1000
