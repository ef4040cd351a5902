"""Timed cases of the MI355X xPU library: what a backend has the GPU service do.

Each case drives the library through its public entry points (the Python
binding of include/xpuhip.h) on chunks as the backend hands them over:

  scan    GpuScan of an Arrow chunk in device memory, projecting (c, d)
  heap    the same scan of 8 KB heap pages, in device memory or (host = True)
          in host memory, as the service receives a chunk over its socket
  preagg  GROUP BY key: count(*), sum(v), avg(w), min(x), max(x), with the
          result read back and the session cleared for the next query; int4
          Zipf keys or text keys, with or without NULL arguments
  topn    the same aggregates over about a million groups, ORDER BY sum(v)
          DESC, key LIMIT n
  join    star join of a fact chunk with three dimensions and a GROUP BY;
          the session keeps its dimension hash tables across queries
  query   the whole star query of a backend that keeps nothing: dimensions
          scanned into pinned inner buffers, attached, joined, read back,
          every session closed
  batch   many scan + group-by fragments in one launch (xpuhip_batch_exec)

Tables have the distributions of pgstrom.datagen, made on the GPU.
"""
import ctypes as C
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "pg-strom_amd"))

from pgstrom import abi, codegen as cg, datagen, kds, workloads as W, xpuhip  # noqa: E402

DIMS = (2_000_000, 200_000, 2_556)
NKEYS = 10_000          # int4 Zipf keys 1..NKEYS
NTEXTS = 2_556          # text keys
DEV = "cuda"


# ----------------------------------------------------------------------
# the cases
# ----------------------------------------------------------------------
def listed():
    return [
        # a small table's only chunk: launches and host work count
        {"name": "scan_4k", "kind": "scan", "rows": 4_001, "k": 500_000},
        # an ordinary columnar chunk
        {"name": "scan_1m", "kind": "scan", "rows": 1_000_000, "k": 500_000},
        # a large slice of a table resident in HBM
        {"name": "scan_24m", "kind": "scan", "rows": 24_000_000, "k": 500_000},
        # heap pages cached in device memory
        {"name": "heap_1m", "kind": "heap", "rows": 1_000_000, "k": 500_000, "host": False},
        # a 64 MB chunk of heap pages as the service receives it
        {"name": "heap_host_850k", "kind": "heap", "rows": 850_000, "k": 500_000, "host": True},
        # a small group-by with NULLs among the arguments
        {"name": "preagg_60k", "kind": "preagg", "rows": 60_001, "key": "int", "null_pct": 5},
        # the headline group-by: 100M rows, 10,000 Zipf keys
        {"name": "preagg_100m", "kind": "preagg", "rows": 100_000_000, "key": "int",
         "null_pct": 0},
        # GROUP BY a text column
        {"name": "preagg_text_4m", "kind": "preagg", "rows": 4_000_000, "key": "text",
         "null_pct": 0},
        # a top-N report over about a million groups
        {"name": "topn_6m", "kind": "topn", "rows": 6_000_000, "limit": 1000},
        # the large star join over resident dimensions
        {"name": "join_200m", "kind": "join", "rows": 200_000_000},
        # a backend's whole star query from session open to close
        {"name": "query_2m", "kind": "query", "rows": 2_000_000},
        # fragments of many backends coalesced into one launch
        {"name": "batch_24", "kind": "batch", "frags": 24, "max_rows": 16_000_000},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["scan", "scan", "heap", "preagg", "preagg", "topn", "join", "query",
                       "batch"])
    if kind == "scan":
        return {"kind": kind, "rows": _log(rng, 1_000, 24_000_000),
                "k": rng.randrange(100_000, 900_001)}
    if kind == "heap":
        host = rng.random() < 0.5
        return {"kind": kind, "rows": _log(rng, 2_000, 850_000 if host else 1_000_000),
                "k": rng.randrange(100_000, 900_001), "host": host}
    if kind == "preagg":
        key = rng.choice(["int", "int", "text"])
        return {"kind": kind, "rows": _log(rng, 2_000, 4_000_000 if key == "text" else 100_000_000),
                "key": key, "null_pct": rng.choice([0, 5])}
    if kind == "topn":
        return {"kind": kind, "rows": _log(rng, 100_000, 6_000_000), "limit": _log(rng, 10, 10_000)}
    if kind == "join":
        return {"kind": kind, "rows": _log(rng, 100_000, 200_000_000)}
    if kind == "query":
        return {"kind": kind, "rows": _log(rng, 50_000, 2_000_000)}
    return {"kind": kind, "frags": rng.randrange(4, 25), "max_rows": _log(rng, 200_000, 16_000_000)}


# ----------------------------------------------------------------------
# tables on the GPU
# ----------------------------------------------------------------------
class _Buf:
    """A torch buffer where the session API takes a device buffer."""

    def __init__(self, t):
        self.t = t
        self.ptr = t.data_ptr()
        self.nbytes = t.numel()


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _ints(g, lo, hi, n, dtype):
    return torch.randint(lo, hi, (n,), generator=g, device=DEV, dtype=dtype)


def _rand(g, n):
    return torch.rand(n, generator=g, device=DEV, dtype=torch.float64)


def _text(g, lens):
    """int32 offsets and bytes of random [A-Za-z0-9] strings of these lengths."""
    offs = torch.zeros(len(lens) + 1, device=DEV, dtype=torch.int64)
    torch.cumsum(lens, 0, out=offs[1:])
    abc = torch.from_numpy(datagen.ALNUM.copy()).to(DEV)
    data = abc[_ints(g, 0, len(abc), int(offs[-1]), torch.int64)]
    return offs.to(torch.int32), data


def _scan_columns(seed, n):
    """a int4, b float8, c int8, d text of 8-24 characters, 5% NULLs each."""
    g = _gen(seed)
    null = [_rand(g, n) < 0.05 for _ in range(4)]
    lens = torch.where(null[3], 0, _ints(g, 8, 25, n, torch.int64))
    return [("a", "int4", _ints(g, 0, 1_000_000, n, torch.int32), null[0]),
            ("b", "float8", torch.randn(n, generator=g, device=DEV, dtype=torch.float64), null[1]),
            ("c", "int8", _ints(g, -10**12, 10**12 + 1, n, torch.int64), null[2]),
            ("d", "text", _text(g, lens), null[3])]


def _zipf(g, n, nkeys=NKEYS, s=1.1):
    p = torch.arange(1, nkeys + 1, device=DEV, dtype=torch.float64) ** (-s)
    cdf = torch.cumsum(p, 0)
    return (torch.searchsorted(cdf / cdf[-1], _rand(g, n), right=True) + 1).clamp_(max=nkeys)


def _preagg_columns(seed, n, key="zipf", null_pct=0):
    """key, v int8, w float8, x int4; key int4 Zipf over 10,000 or uniform
    over a million values, or one of 2,556 texts of 8-24 characters."""
    g = _gen(seed)
    if key == "text":
        lens = _ints(g, 8, 25, NTEXTS, torch.int64)
        offs, data = _text(g, lens)
        pick = _ints(g, 0, len(lens), n, torch.int64)
        o = torch.zeros(n + 1, device=DEV, dtype=torch.int64)
        torch.cumsum(lens[pick], 0, out=o[1:])
        at = torch.repeat_interleave(offs[:-1].long()[pick] - o[:-1], lens[pick])
        col = ("key", "text", (o.to(torch.int32), data[at + torch.arange(len(at), device=DEV)]), None)
    elif key == "uniform":
        col = ("key", "int4", _ints(g, 0, 1_000_000, n, torch.int32), None)
    else:
        col = ("key", "int4", _zipf(g, n).to(torch.int32), None)
    null = [(_rand(g, n) < null_pct / 100.0) if null_pct else None for _ in range(3)]
    return [col, ("v", "int8", _ints(g, 0, 1_000_000, n, torch.int64), null[0]),
            ("w", "float8", _rand(g, n) * 1000.0, null[1]),
            ("x", "int4", _ints(g, -2**31, 2**31, n, torch.int64).to(torch.int32), null[2])]


def _fact_columns(seed, n):
    g = _gen(seed)
    return [("fk%d" % (i + 1), "int4", _ints(g, 1, sz + 1, n, torch.int32), None)
            for i, sz in enumerate(DIMS)] + \
           [("quantity", "int8", _ints(g, 1, 51, n, torch.int64), None),
            ("price", "int8", _ints(g, 1000, 10_000_001, n, torch.int64), None)]


def _dim_columns(seed):
    """The three dimensions: pk 1..size, category 0-24, a 16-character text."""
    out = []
    for i, sz in enumerate(DIMS):
        g = _gen(seed * 4 + 1 + i)
        out.append([("pk", "int4", torch.arange(1, sz + 1, device=DEV, dtype=torch.int32), None),
                    ("category", "int2", _ints(g, 0, 25, sz, torch.int16), None),
                    ("txt", "text", _text(g, torch.full((sz,), 16, device=DEV)), None)])
    return out


class _Schema:
    """What the workloads read of a column: its name and type."""

    def __init__(self, name, typname):
        self.name = name
        self.typname = typname


def _schema(cols):
    return [_Schema(c[0], c[1]) for c in cols]


def _bytes(t):
    return t.contiguous().view(torch.uint8)


def _bitmap(null):
    n = len(null)
    v = torch.zeros((n + 7) // 8 * 8, device=DEV, dtype=torch.uint8)
    v[:n] = ~null
    w = torch.tensor([1 << i for i in range(8)], device=DEV, dtype=torch.uint8)
    return (v.view(-1, 8) * w).sum(1, dtype=torch.uint8)


def _arrow_chunk(cols):
    """The columns as a KDS_FORMAT_ARROW chunk in device memory."""
    proto = [kds.Column(nm, ty, [b"x"] if ty == "text" else [0]) for nm, ty, _, _ in cols]
    n = len(cols[0][2][0]) - 1 if cols[0][1] == "text" else len(cols[0][2])
    head = kds.build_arrow_kds(proto)[:abi.kds_head_length(len(cols))].copy()
    parts, pos = [], (len(head) + 63) & ~63
    for j, (_, ty, vals, null) in enumerate(cols):
        cm = abi.kern_colmeta.from_buffer(head, abi.KDS_COLMETA_OFFSET + j * C.sizeof(abi.kern_colmeta))
        pieces = [("values", _bytes(vals[0])), ("extra", vals[1])] if ty == "text" else \
            [("values", _bytes(vals))]
        if null is not None:
            pieces.insert(0, ("nullmap", _bitmap(null)))
        for what, t in pieces:
            setattr(cm, what + "_offset", pos)
            setattr(cm, what + "_length", len(t))
            parts.append((pos, t))
            pos = (pos + len(t) + 63) & ~63
    hd = abi.kern_data_store_head.from_buffer(head)
    hd.length = pos
    hd.nitems = n
    out = torch.zeros(pos, device=DEV, dtype=torch.uint8)
    out[:len(head)] = torch.from_numpy(head).to(DEV)
    for at, t in parts:
        out[at:at + len(t)] = t
    return _Buf(out), n


ROWS_PER_PAGE = 108     # of at most 80 bytes each; 66 on average


def _heap_chunk(cols, seed):
    """The scan table's rows as heap tuples on 8 KB pages (KDS_FORMAT_BLOCK in
    device memory); one row in a hundred is invisible (LP_UNUSED).  Returns
    the chunk and its header."""
    (_, _, a, na), (_, _, b, nb), (_, _, c, nc), (_, _, (offs, data), nd) = cols
    n = len(a)
    npages = (n + ROWS_PER_PAGE - 1) // ROWS_PER_PAGE
    lens = (offs[1:] - offs[:-1]).long()
    # payload after the 24-byte tuple header: NULLs take no space
    pa = torch.zeros(n, device=DEV, dtype=torch.int64)
    end = torch.where(na, 0, 4)
    pb = (end + 7) & ~7
    end = torch.where(nb, end, pb + 8)
    pc = (end + 7) & ~7
    end = torch.where(nc, end, pc + 8)
    pd = end
    end = torch.where(nd, end, pd + 1 + lens)
    size = 24 + end
    asize = (size + 7) & ~7
    page = torch.arange(n, device=DEV) // ROWS_PER_PAGE
    cum = torch.cumsum(asize, 0)
    before = torch.cat([cum.new_zeros(1), cum])[page * ROWS_PER_PAGE]
    off = kds.BLCKSZ - (cum - before)           # tuples down from the page's end
    slot = torch.arange(n, device=DEV) - page * ROWS_PER_PAGE
    live = _rand(_gen(seed + 77), n) >= 0.01
    pages = torch.zeros(npages * kds.BLCKSZ, device=DEV, dtype=torch.uint8)
    at = page * kds.BLCKSZ + off

    def put(pos, vals, keep=None):
        raw = _bytes(vals).view(len(vals), -1)
        if keep is not None:
            pos, raw = pos[keep], raw[keep]
        for k in range(raw.shape[1]):
            pages[pos + k] = raw[:, k]

    anynull = na | nb | nc | nd
    bits = (~na).to(torch.uint8) | (~nb).to(torch.uint8) << 1 | (~nc).to(torch.uint8) << 2 | \
        (~nd).to(torch.uint8) << 3
    put(at, torch.full((n,), kds.FROZEN_XID, device=DEV, dtype=torch.int32))
    put(at + 16, (slot + 1).to(torch.int16))
    put(at + 18, torch.full((n,), 4, device=DEV, dtype=torch.int16))
    put(at + 20, (0x0900 + (~nd).int() * abi.HEAP_HASVARWIDTH +
                  anynull.int() * abi.HEAP_HASNULL).to(torch.int16))
    put(at + 22, torch.full((n,), 24, device=DEV, dtype=torch.uint8))
    put(at + 23, torch.where(anynull, bits, 0).to(torch.uint8))
    put(at + 24 + pa, a, ~na)
    put(at + 24 + pb, b, ~nb)
    put(at + 24 + pc, c, ~nc)
    put(at + 24 + pd, ((lens + 1) << 1 | 1).to(torch.uint8), ~nd)
    pages[torch.repeat_interleave(at + 25 + pd - offs[:-1].long(), lens) +
          torch.arange(len(data), device=DEV)] = data
    lp = torch.where(live, off | kds.LP_NORMAL << 15 | size << 17, 0).to(torch.int32)
    put(page * kds.BLCKSZ + kds.PAGE_HEADER_SIZE + 4 * slot, lp)
    last = torch.full((npages,), n - 1, device=DEV)
    last[:-1] = torch.arange(1, npages, device=DEV) * ROWS_PER_PAGE - 1
    p0 = torch.arange(npages, device=DEV) * kds.BLCKSZ
    put(p0 + 10, torch.full((npages,), kds.PD_ALL_VISIBLE, device=DEV, dtype=torch.int16))
    put(p0 + 12, (kds.PAGE_HEADER_SIZE + 4 * (slot[last] + 1)).to(torch.int16))
    put(p0 + 14, off[last].to(torch.int16))
    put(p0 + 16, torch.full((npages,), kds.BLCKSZ, device=DEV, dtype=torch.int16))
    put(p0 + 18, torch.full((npages,), kds.BLCKSZ | 4, device=DEV, dtype=torch.int16))
    head = np.frombuffer(bytes(kds.kds_header(abi.KDS_FORMAT_BLOCK, [c[:2] for c in cols])),
                         dtype=np.uint8).copy()
    hd = abi.kern_data_store_head.from_buffer(head)
    hd.block_offset = abi.maxalign(len(head) + 4 * npages)
    hd.length = hd.block_offset + len(pages)
    hd.nitems = hd.block_nloaded = npages
    out = torch.zeros(hd.length, device=DEV, dtype=torch.uint8)
    out[:len(head)] = torch.from_numpy(head).to(DEV)
    out[len(head):len(head) + 4 * npages] = _bytes(torch.arange(1000, 1000 + npages, device=DEV,
                                                                dtype=torch.int32))
    out[hd.block_offset:] = pages
    return _Buf(out), head


def _selected(case):
    """Rows that WHERE a < k AND b > 0.0 is expected to keep."""
    return 0.95 * case["k"] / 1e6 * 0.475 * case["rows"]


def _dst_length(case):
    """A kds_dst for them: 58 bytes a row on average, 72 at most, and room
    for eight standard deviations more rows."""
    n = _selected(case)
    return 4096 + 8 * int((64 * n + 72 * 8 * math.sqrt(n)) / 8)


def _inner_tables(dims):
    """kern_multirels of the filtered dimensions (pk % 10 = i), as the
    backend's inner preload builds it from MinimalTuples."""
    coldefs = [("pk", "int4"), ("category", "int2"), ("txt", "text")]
    mark = kds.form_minimal_tuple(coldefs, (0x01020304, 0x0506, b"~" * 16))
    p_pk, p_cat, p_txt = (mark.index(x) for x in (b"\4\3\2\1", b"\6\5", b"~" * 16))
    inners = []
    for i, (pk, cat, txt) in enumerate(dims):
        mod, rem = W.dim_filter_mod(i)
        pkv, catv = pk[2].cpu().numpy(), cat[2].cpu().numpy()
        text = txt[2][1].cpu().numpy().reshape(-1, 16)
        sel = np.nonzero(pkv % mod == rem)[0]
        rows = np.tile(np.frombuffer(mark, dtype=np.uint8), (len(sel), 1))
        rows[:, p_pk:p_pk + 4] = pkv[sel].astype("<i4").view(np.uint8).reshape(-1, 4)
        rows[:, p_cat:p_cat + 2] = catv[sel].astype("<i2").view(np.uint8).reshape(-1, 2)
        rows[:, p_txt:p_txt + 16] = text[sel]
        inners.append((xpuhip.inner_hash_setup(coldefs, [r.tobytes() for r in rows], [1]), False))
    return kds.build_multirels(inners)


def _topn_query(cols, limit):
    plan = cg.Plan([(c.name, c.typname) for c in cols])
    key, v, w, x = (plan.scan_var(nm) for nm in ("key", "v", "w", "x"))
    plan.set_groupby(W.preagg_tlist(plan, key, v, w, x))
    return plan.build(final_nrows=1_000_000, sort_limit=limit,
                      sort_keys=[(abi.KSORT_KEY_KIND__PSUM_NUMERIC, 2, None, False, False),
                                 (abi.KSORT_KEY_KIND__VREF, 6, "int4", True, False)])


def _fragments(case):
    """(rows, k, m) of each fragment: rows log-uniform from 64K up, its own
    predicate constant a < k and GROUP BY key % m."""
    r = random.Random(case["frags"] * 1_000_003 + case["max_rows"])
    lo = 65_536
    out = []
    for i in range(case["frags"]):
        n = int(lo * (case["max_rows"] / lo) ** ((i + 0.5) / case["frags"]))
        out.append((n, r.randrange(100_000, 900_001), int(round(math.exp(
            r.uniform(math.log(16), math.log(100_000)))))))
    r.shuffle(out)
    return out


def _batch_columns(case, seed):
    cols = _preagg_columns(seed, case["max_rows"])
    return [("a", "int4", _ints(_gen(seed + 91), 0, 1_000_000, case["max_rows"], torch.int32),
             None)] + cols


def _windows(case, seed):
    r = random.Random(seed)
    return [(r.randrange(0, (case["max_rows"] - n) // 64 + 1) * 64, n)
            for n, _, _ in _fragments(case)]


# ----------------------------------------------------------------------
# what the program has in hand, and one pass
# ----------------------------------------------------------------------
def prepare(case, seed):
    kind = case["kind"]
    xpuhip.init(0)
    st = {"case": case}
    if kind in ("scan", "heap"):
        cols = _scan_columns(seed, case["rows"])
        st["sess"] = xpuhip.Session(W.scan_query(_schema(cols), k=case["k"]))
        if kind == "scan":
            st["src"], st["n"] = _arrow_chunk(cols)
        else:
            st["src"], st["head"] = _heap_chunk(cols, seed)
        st["len"] = _dst_length(case)
        if case.get("host"):
            st["host"] = st.pop("src").t.cpu().numpy()
        else:
            st["dst"] = _Buf(torch.zeros(st["len"], device=DEV, dtype=torch.uint8))
    elif kind == "preagg":
        cols = _preagg_columns(seed, case["rows"], "zipf" if case["key"] == "int" else "text",
                               case["null_pct"])
        st["sess"] = xpuhip.Session(W.preagg_query(_schema(cols)))
        st["src"], st["n"] = _arrow_chunk(cols)
    elif kind == "topn":
        cols = _preagg_columns(seed, case["rows"], "uniform")
        st["sess"] = xpuhip.Session(_topn_query(_schema(cols), case["limit"]))
        st["src"], st["n"] = _arrow_chunk(cols)
    elif kind == "join":
        cols = _fact_columns(seed, case["rows"])
        st["sess"] = xpuhip.Session(W.star_query(_schema(cols)))
        st["sess"].attach_inner(_inner_tables(_dim_columns(seed)))
        st["src"], st["n"] = _arrow_chunk(cols)
    elif kind == "query":
        cols = _fact_columns(seed, case["rows"])
        dims = _dim_columns(seed)
        st["dims"] = [_arrow_chunk(d) for d in dims]
        st["dim_blobs"] = [W.dim_scan_pinned(_schema(d), i) for i, d in enumerate(dims)]
        st["blob"] = W.star_query(_schema(cols))
        st["kmrels"] = W.star_inner_pinned()
        st["src"], st["n"] = _arrow_chunk(cols)
    else:
        cols = _batch_columns(case, seed)
        base, _ = _arrow_chunk(cols)
        stride = 1024
        nfrag = case["frags"]
        hdrs = kds.window_headers(base.t[:abi.kds_head_length(len(cols))].cpu().numpy(),
                                  _windows(case, seed), nfrag * stride, stride)
        st["src"] = _Buf(torch.cat([torch.from_numpy(hdrs).to(DEV), base.t]))
        st["tasks"] = []
        for i, (n, k, m) in enumerate(_fragments(case)):
            s = xpuhip.Session(W.fragment_query(_schema(cols), k=k, m=m))
            st["tasks"].append((s, st["src"].ptr + i * stride, n))
    torch.cuda.synchronize()
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "scan":
        rc, _, _ = st["sess"].exec_device(st["src"], st["n"], st["dst"], st["len"])
        assert rc == 0
        return st["dst"].t
    if kind == "heap":
        if case["host"]:
            rc, dst, _, _ = st["sess"].exec(st["host"], dst_length=st["len"])
            assert rc == 0
            return dst
        rc, _, _ = st["sess"].exec_device_tuples(st["src"], st["head"], st["dst"], st["len"])
        assert rc == 0
        return st["dst"].t
    if kind == "batch":
        xpuhip.batch_exec(st["tasks"], graph=True)
        parts = []
        for (s, _, _), (_, _, m) in zip(st["tasks"], _fragments(case)):
            parts.append(_groups(s.final(), min(m, NKEYS + 1)))
            s.reset()
        return {k: np.concatenate([p[k] for p in parts]) for k in parts[0]}
    if kind == "query":
        sess = [xpuhip.Session(b) for b in st["dim_blobs"]]
        for s, (buf, n) in zip(sess, st["dims"]):
            s.exec_device(buf, n)
        j = xpuhip.Session(st["blob"])
        j.attach_inner(st["kmrels"])
        j.exec_device(st["src"], st["n"])
        out = _star_groups(j.final())
        j.close()
        for s in sess:
            s.close()
        return out
    s = st["sess"]
    s.exec_device(st["src"], st["n"])
    fin = s.final()
    s.reset()
    if kind == "join":
        return _star_groups(fin)
    if kind == "topn":
        return _groups(fin, None)
    return _text_groups(fin) if case["key"] == "text" else _groups(fin, NKEYS + 1)


def _words(fin):
    """A kds_final as 8-byte words, and the word each group tuple starts at:
    the tuples have fixed offsets (partial states first, then the key)."""
    hd = abi.kern_data_store_head.from_buffer_copy(fin[:C.sizeof(abi.kern_data_store_head)])
    ridx = fin[abi.kds_head_length(hd.nr_colmeta):][:8 * hd.nitems].view(np.int64)
    return fin[:hd.length >> 3 << 3].view(np.int64), (hd.length - ridx) >> 3


def _states(words, at):
    return {"rows": words[at + 2], "v_n": words[at + 4], "v_lo": words[at + 5],
            "v_hi": words[at + 6], "w_n": words[at + 8], "w": words[at + 9].view(np.float64),
            "min": words[at + 11], "max": words[at + 13]}


def _dense(cols, key, nkeys):
    """The columns by key 0..nkeys - 1, zero where there is no group."""
    out = {}
    for name, v in cols.items():
        out[name] = np.zeros(nkeys, dtype=v.dtype)
        out[name][key] = v
    return out


def _groups(fin, nkeys):
    """The groups of an int4 key: by key, or (nkeys None) in the order they came."""
    words, at = _words(fin)
    key = words[at + 14] & 0xffffffff
    cols = _states(words, at)
    return dict(cols, key=key) if nkeys is None else _dense(cols, key, nkeys)


def _star_groups(fin):
    words, at = _words(fin)
    key = words[at + 6]
    return _dense({"n": words[at + 3], "lo": words[at + 4], "hi": words[at + 5]},
                  (key & 0xffff) * 25 + (key >> 16 & 0xffff), 625)


def _text_groups(fin):
    """The groups of a text key in the keys' byte order."""
    words, at = _words(fin)
    # a 4-byte length word, the characters, then the row id
    raw = np.stack([words[at + 14 + i] for i in range(4)], axis=1).view(np.uint8)
    size = (raw[:, :4].copy().view(np.uint32) >> 2).astype(np.int64)
    text = np.where(np.arange(32) < size, raw, 0).astype(np.uint8)[:, 4:].copy()
    order = np.argsort(text.view("S28")[:, 0])
    cols = dict(_states(words, at), key=text)
    out = {}
    for name, v in cols.items():
        out[name] = np.zeros((NTEXTS,) + v.shape[1:], dtype=v.dtype)
        out[name][:len(order)] = v[order]
    return out


# ----------------------------------------------------------------------
# work, tolerance, exact results
# ----------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "batch":
        return {"bytes": sum(28 * n + 128 * min(m, 10_000) for n, _, m in _fragments(case)), "flops": 0}
    n = case["rows"]
    nsel = _selected(case) if "k" in case else 0
    if kind == "scan":
        # a, b, c, text offsets, text, validity bits; rows out
        return {"bytes": n * (4 + 8 + 8 + 4 + 15.2 + 0.5) + nsel * 58, "flops": 0}
    if kind == "heap":
        return {"bytes": (n // ROWS_PER_PAGE + 1) * kds.BLCKSZ + nsel * 58, "flops": 0}
    if kind == "preagg":
        return {"bytes": n * (24 if case["key"] == "int" else 20 + 4 + 16) + 1_280_000, "flops": 0}
    if kind == "topn":
        return {"bytes": n * 24 + 128 * case["limit"], "flops": 0}
    if kind == "join":
        return {"bytes": n * 28, "flops": 0}
    return {"bytes": n * 28 + sum(DIMS) * (4 + 2 + 20), "flops": 0}


def tolerance(case):
    if case["kind"] in ("preagg", "topn", "batch"):
        # counts, integer sums, min and max are whole; float8 sums of up to
        # 13M addends: 5e-15 off a sum in another order, 6e-16 run to run
        return {"rel": 2e-14, "max": 1e-12}
    return "exact"


def _sums(key, w, nkeys):
    """Rows and float64 sum of w per key, summed a million rows at a time."""
    key, w = key.cpu().numpy(), w.cpu().numpy()
    rows, sums = np.zeros(nkeys, dtype=np.int64), np.zeros(nkeys)
    for i in range(0, len(key), 1_000_000):
        k = key[i:i + 1_000_000]
        rows += np.bincount(k, minlength=nkeys)
        sums += np.bincount(k, weights=w[i:i + 1_000_000], minlength=nkeys)
    return rows, sums


def exact(case, seed):
    """The float8 sums per group; whole values are compared as they are."""
    kind = case["kind"]
    none = {k: None for k in ("rows", "v_n", "v_lo", "v_hi", "w_n", "min", "max")}
    if kind == "batch":
        cols = _batch_columns(case, seed)
        got = []
        for (n, k, m), (r0, _) in zip(_fragments(case), _windows(case, seed)):
            a, key, w = (cols[i][2][r0:r0 + n] for i in (0, 1, 3))
            keep = a < k
            got.append(_sums(key[keep] % m, w[keep], min(m, NKEYS + 1))[1])
        return dict(none, w=np.concatenate(got))
    if kind not in ("preagg", "topn"):
        return None
    if kind == "preagg" and case["key"] == "text":
        return None
    cols = _preagg_columns(seed, case["rows"], "zipf" if kind == "preagg" else "uniform",
                           case.get("null_pct", 0))
    key, v, w = (c[2] for c in cols[:3])
    if case.get("null_pct"):
        w = torch.where(cols[2][3], 0.0, w)
    if kind == "preagg":
        return dict(none, w=_sums(key, w, NKEYS + 1)[1])
    rows, sums = _sums(key, w, 1_000_000)
    tot = _sums(key, v, 1_000_000)[1]       # whole numbers below 2^53
    tot[rows == 0] = -1
    return dict(none, key=None, w=sums[np.lexsort((np.arange(1_000_000), -tot))[:case["limit"]]])
