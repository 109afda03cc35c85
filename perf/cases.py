"""The work that users have this package do, as cases that can be timed.

A case is a dict of plain values.  `listed()` names twelve of them, `draw(rng)`
gives another of the same ranges, `prepare(case, seed)` makes what a program
holds before the call (columns on the device, result buffers, an index to
query), `run(state)` is one pass through the public entry points,
`work(case)` the bytes that pass cannot do without, and `exact(case, seed)`
the same results from plain torch.

Kinds of case:
  build    Context.build_device of one column that is resident in HBM
  batch    Context.build_batch_device of many ragged columns, replayed from a
           graph in buffers that the program keeps
  host     Context.build of a host array: the per-column drop-in
  range    Context.query_range_device on a built index
  codec    Context.encode_device of a row bitmap and decode_device of its words
  combine  Context.combine_device of two keys' words
  stages   the staged pipeline, one entry point per stage
  prims    compaction, exclusive scan and segmented scan
"""
import math

import numpy as np
import torch

import indexing_amd as ia

DEV = "cuda:0"
OPS = ("and", "or", "xor", "andnot")
COUNT_WORDS = 10  # a wahgpu_counts record in 32-bit words

_context = None


def shared_context():
    """One context for the whole process, as a program keeps it."""
    global _context
    if _context is None:
        _context = ia.Context(0)
    return _context


# -- the cases -----------------------------------------------------------------
def listed():
    return [
        # the smallest call: a column of a few rows, bound by launches
        {"name": "build-1000", "kind": "build", "n": 1000, "dist": "uniform", "card": 1000,
         "rid_base": 0},
        # 2^20 uniform 16-bit values: one column of an ordinary table
        {"name": "build-2p20", "kind": "build", "n": 1 << 20, "dist": "uniform", "card": 65536,
         "rid_base": 0},
        # 2^28 uniform 16-bit values: the headline column of the benchmark
        {"name": "build-2p28", "kind": "build", "n": 1 << 28, "dist": "uniform", "card": 65536,
         "rid_base": 0},
        # 2^28 values in long runs (a sorted or clustered column), 20-bit keys
        {"name": "build-runs-2p28", "kind": "build", "n": 1 << 28, "dist": "runs",
         "card": 1 << 20, "rid_base": 0},
        # a slice of a column of 32-bit identifiers, ragged, with global rows
        {"name": "build-ids-5m", "kind": "build", "n": 5_000_011, "dist": "uniform",
         "card": 1 << 32, "rid_base": 1_000_003},
        # a table's columns of uneven length and cardinality, in one launch set
        {"name": "batch-128", "kind": "batch", "cols": 128, "lo_log": 12.0, "hi_log": 20.0},
        # a column handed over in host memory and its index handed back
        {"name": "host-300k", "kind": "host", "n": 300_007, "dist": "zipf", "card": 4096,
         "rid_base": 0},
        # a range predicate over a tenth of the keys of a 2^26-row index
        {"name": "range-2p26", "kind": "range", "n": 1 << 26, "card": 4096, "part": 0.1},
        # a query's result bitmap stored as WAH words and read back
        {"name": "codec-2p27", "kind": "codec", "n": (1 << 27) + 3, "density": 0.01},
        # two predicates of a small table combined, bound by launches and waits
        {"name": "combine-300k", "kind": "combine", "n": 300_007, "card": 50, "op": "and"},
        # the pipeline stage by stage, as the phases program runs it
        {"name": "stages-4m", "kind": "stages", "n": (1 << 22) + 13, "dist": "uniform",
         "card": 65536},
        # the scan and compaction primitives
        {"name": "prims-16m", "kind": "prims", "n": (1 << 24) + 5},
    ]


def _log_size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _column(rng, lo, hi):
    dist = rng.choice(("uniform", "uniform", "zipf", "runs"))
    n = _log_size(rng, lo, hi)
    if dist == "uniform":
        card = rng.choice((_log_size(rng, 2, 65536), 65536, 1 << 32))
    elif dist == "zipf":
        card = _log_size(rng, 2, 65536)
    else:
        card = _log_size(rng, 1 << 10, 1 << 20)
    return {"n": n, "dist": dist, "card": card}


def draw(rng):
    kind = rng.choice(("build", "build", "build", "build", "batch", "host", "range", "codec",
                       "combine", "stages", "prims"))
    if kind == "build":
        return {"kind": kind, **_column(rng, 500, 1 << 27),
                "rid_base": rng.choice((0, 0, rng.randrange(1 << 20)))}
    if kind == "batch":
        return {"kind": kind, "cols": _log_size(rng, 4, 200), "lo_log": rng.choice((9.0, 12.0)),
                "hi_log": rng.uniform(14.0, 20.0)}
    if kind == "host":
        return {"kind": kind, **_column(rng, 500, 1 << 22), "rid_base": 0}
    if kind == "range":
        return {"kind": kind, "n": _log_size(rng, 10_000, 1 << 26), "card": _log_size(rng, 16, 65536),
                "part": rng.uniform(0.01, 0.5)}
    if kind == "codec":
        return {"kind": kind, "n": _log_size(rng, 10_000, 1 << 28),
                "density": 10.0 ** rng.uniform(-4.0, -0.3)}
    if kind == "combine":
        return {"kind": kind, "n": _log_size(rng, 10_000, 1 << 26), "card": _log_size(rng, 4, 1000),
                "op": rng.choice(OPS)}
    if kind == "stages":
        return {"kind": kind, **_column(rng, 1000, 1 << 24)}
    return {"kind": kind, "n": _log_size(rng, 1000, 1 << 27)}


# -- inputs --------------------------------------------------------------------
def _generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _as_i32(x):
    """int64 values in [0, 2^32) as int32 bit patterns."""
    return torch.where(x >= 1 << 31, x - (1 << 32), x).to(torch.int32)


def _zipf(n, card, s, g):
    cdf = torch.cumsum(torch.arange(1, card + 1, device=DEV, dtype=torch.float64) ** -s, 0)
    u = torch.rand(n, device=DEV, dtype=torch.float64, generator=g) * cdf[-1]
    return torch.searchsorted(cdf, u).clamp_(max=card - 1).to(torch.int32)


RUN_MEAN = 4096.0


def values_of(dist, n, card, seed):
    """A column as an int32 tensor of uint32 bit patterns."""
    g = _generator(seed)
    if dist == "uniform":
        if card == 1 << 32:
            return torch.randint(-(1 << 31), 1 << 31, (n,), device=DEV, dtype=torch.int32,
                                 generator=g)
        return torch.randint(0, card, (n,), device=DEV, dtype=torch.int32, generator=g)
    if dist == "zipf":
        return _zipf(n, card, 1.0, g)
    # runs: Zipf(1.2) values, each for a geometric number of rows
    m = int(n / RUN_MEAN * 1.5) + 64
    u = torch.rand(m, device=DEV, dtype=torch.float64, generator=g)
    length = torch.floor(torch.log1p(-u) / math.log1p(-1.0 / RUN_MEAN)).to(torch.int64) + 1
    length[-1] += n  # the last run reaches past the column
    ends = torch.cumsum(length, 0).clamp_(max=n)
    starts = torch.cat([ends.new_zeros(1), ends[:-1]])
    return torch.repeat_interleave(_zipf(m, card, 1.2, g), ends - starts)


# Results such as a stage's entries or a bitmap's words are returned at their own
# length, which the inputs decide.  The inputs below are one arrangement of rows
# per case, varied by the seed in ways that keep those lengths: other values for
# the same rows, other places of the same rows inside their 31-row chunks.
LAYOUT = 20250


def relabelled(case, seed):
    """A column whose equal rows are the case's and whose values are the seed's."""
    v = values_of(case["dist"], case["n"], case["card"], LAYOUT)
    g = _generator(seed)
    if case["card"] == 1 << 32:
        return v ^ torch.randint(-(1 << 31), 1 << 31, (1,), device=DEV, dtype=torch.int32,
                                 generator=g)
    return torch.randperm(case["card"], device=DEV, generator=g).to(torch.int32)[v.long()]


def rotated(rows, seed):
    """The rows (any dtype) of each whole 31-row chunk rotated by a random step."""
    chunks = rows.numel() // 31
    if not chunks:
        return rows
    step = torch.randint(0, 31, (chunks, 1), device=DEV, generator=_generator(seed))
    at = (torch.arange(31, device=DEV) + step) % 31
    out = rows.clone()
    out[:31 * chunks] = rows[:31 * chunks].view(chunks, 31).gather(1, at).view(-1)
    return out


def batch_columns(case):
    """(offset, n, cardinality, distribution) of each column, and their extent."""
    rng = np.random.default_rng(case["cols"])
    cols, at = [], 0
    for i in range(case["cols"]):
        n = int(2.0 ** rng.uniform(case["lo_log"], case["hi_log"]))
        card = max(2, int(2.0 ** rng.uniform(1, 16)))
        cols.append((at, n, card, "uniform" if i % 2 == 0 else "zipf"))
        at += (n + 63) // 64 * 64
    return cols, at


def batch_values(case, seed):
    cols, total = batch_columns(case)
    values = torch.zeros(total, device=DEV, dtype=torch.int32)
    for i, (at, n, card, dist) in enumerate(cols):
        values[at:at + n] = values_of(dist, n, card, seed * 1009 + i)
    return cols, total, values


def bitmap_of(mask):
    """Row bitmap (32 rows a word, row r in bit r % 32) of a bool tensor."""
    n = mask.numel()
    pad = torch.zeros((n + 31) // 32 * 32, device=mask.device, dtype=torch.uint8)
    pad[:n] = mask
    weight = torch.tensor([1 << b for b in range(8)], device=mask.device, dtype=torch.uint8)
    return (pad.view(-1, 8) * weight).sum(1, dtype=torch.uint8).view(torch.int32)


def codec_mask(case, seed):
    base = torch.rand(case["n"], device=DEV, generator=_generator(LAYOUT)) < case["density"]
    return rotated(base, seed)


def combine_columns(case, seed):
    """Two columns of one table: a predicate selects a key of each."""
    return [rotated(values_of("uniform", case["n"], case["card"], LAYOUT + i), seed)
            for i in range(2)]


def range_bounds(case):
    width = max(1, int(case["card"] * case["part"]))
    lo = (case["card"] - width) // 2
    return lo, lo + width - 1


def prims_inputs(case, seed):
    g, n = _generator(seed), case["n"]
    data = torch.randint(0, 1000, (n,), device=DEV, dtype=torch.int32, generator=g)
    valid = torch.randint(0, 2, (n,), device=DEV, dtype=torch.int32, generator=_generator(LAYOUT))
    valid = torch.roll(valid, seed % n)
    heads = (torch.rand(n, device=DEV, generator=g) < 0.01).to(torch.int32)
    return data, valid, heads


def _out(n, counts=1):
    """The result buffers of a build, as a program that builds often keeps them."""
    def z(m):
        return torch.zeros(m, device=DEV, dtype=torch.int32)
    return z(n), z(n), z(n), z(2 * n), z(counts * COUNT_WORDS)


def _built(ctx, values):
    """A column's index, in tensors of its size."""
    out = ctx.build_device(values)
    c = ctx.read_counts(out[4])
    sizes = (int(c.keycnt),) * 3 + (int(c.length),)
    return [t[:m].clone() for t, m in zip(out, sizes)]


def prepare(case, seed):
    kind, ctx = case["kind"], shared_context()
    state = {"kind": kind, "ctx": ctx, "case": case}
    if kind == "build":
        state["values"] = values_of(case["dist"], case["n"], case["card"], seed)
        state["out"] = _out(case["n"])
    elif kind == "batch":
        # the graph holds the buffers' addresses: a program keeps a context for it
        cols, total, values = batch_values(case, seed)
        state["ctx"] = ia.Context(0)
        state["ctx"].batch_reserve(total, len(cols))
        state["values"] = values
        state["cols"] = [(at, n) for at, n, _, _ in cols]
        state["out"] = _out(total, len(cols))
    elif kind == "host":
        state["values"] = relabelled(case, seed).cpu().numpy().view(np.uint32)
    elif kind == "range":
        state["index"] = _built(ctx, values_of("uniform", case["n"], case["card"], seed))
        state["bounds"] = range_bounds(case)
    elif kind == "combine":  # the words of each column's first key
        for name, v in zip("ab", combine_columns(case, seed)):
            _, _, lens, words = _built(ctx, v)
            state[name] = words[:int(lens[0])]
    elif kind == "codec":
        state["bitmap"] = bitmap_of(codec_mask(case, seed))
    elif kind == "stages":
        state["values"] = relabelled(case, seed)
    else:
        state["data"], state["valid"], state["heads"] = prims_inputs(case, seed)
    return state


def run(state):
    kind, ctx = state["kind"], state["ctx"]
    if kind == "build":
        return ctx.build_device(state["values"], state["case"]["rid_base"], state["out"])
    if kind == "batch":
        return ctx.build_batch_device(state["values"], state["cols"], state["out"])
    if kind == "host":
        x = ctx.build(state["values"], state["case"]["rid_base"])
        return [a.view(np.int32) for a in (x.keys, x.offsets, x.lengths, x.words)] + \
            [x.k, x.length, x.keycnt, x.bound, x.passes, x.mode]
    if kind == "range":
        return ctx.query_range_device(*state["index"], *state["bounds"], state["case"]["n"])
    if kind == "codec":
        n = state["case"]["n"]
        words = ctx.encode_device(state["bitmap"], n)
        bitmap, last = ctx.decode_device(words, n)
        return words, bitmap, last
    if kind == "combine":
        return ctx.combine_device(state["case"]["op"], state["a"], state["b"], state["case"]["n"])
    if kind == "stages":
        keys, rids = ctx.sort_rids_by_value(state["values"])
        chids, lits = ctx.produce_chunk_id_literals(rids)
        mv, mc, ml = ctx.merge_lit_by_val_chids(keys, chids, lits)
        fills = ctx.produce_fills(mv, mc)
        words = ctx.fuse_fill_literals(fills, ml)
        out = ctx.compute_column_length(mv, fills)
        return [keys, rids, chids, lits, mv, mc, ml, fills, words, *out]
    return (ctx.stream_compaction(state["data"], state["valid"]),
            ctx.exclusive_scan(state["data"]),
            ctx.segmented_inclusive_scan(state["data"], state["heads"]))


# -- what a pass cannot do without ------------------------------------------------
def _index_size(dist, n, card):
    """Expected (entries, words, keys) of a column's index."""
    if dist == "runs":
        runs = n / RUN_MEAN
        return n / 31 + runs, n / 31 + 2 * runs, min(card, runs)
    if dist == "zipf":
        p = np.arange(1, card + 1, dtype=np.float64) ** -1.0
        p /= p.sum()
        times = np.ones(card)
    else:
        p, times = np.array([1.0 / card]), np.array([float(card)])
    absent = np.exp(31 * np.log1p(-p)) if card > 1 else np.zeros(1)
    chunks = max(1.0, n / 31)
    entries = chunks * float((times * (1 - absent)).sum())
    words = chunks * float((times * (1 - absent) * (1 + absent)).sum())
    keys = float((times * -np.expm1(n * np.log1p(-p))).sum()) if card > 1 else 1.0
    return entries, words, keys


def work(case):
    kind, n = case["kind"], case.get("n", 0)
    if kind in ("build", "host"):
        _, L, K = _index_size(case["dist"], n, case["card"])
        b = 4 * n + 4 * L + 12 * K
    elif kind == "batch":
        cols, _ = batch_columns(case)
        b = 0.0
        for _, m, card, dist in cols:
            _, L, K = _index_size(dist, m, card)
            b += 4 * m + 4 * L + 12 * K
    elif kind == "range":
        lo, hi = range_bounds(case)
        _, L, _ = _index_size("uniform", n, case["card"])
        b = 4 * L * (hi - lo + 1) / case["card"] + n / 8
    elif kind in ("codec", "combine"):
        p = case["density"] if kind == "codec" else 1.0 / case["card"]
        absent = (1 - p) ** 31
        L = n / 31 * (1 - absent) * (1 + absent)
        if kind == "codec":
            b = 2 * (n / 8 + 4 * L)
        else:
            q = {"and": p * p, "or": 2 * p - p * p, "xor": 2 * p - 2 * p * p,
                 "andnot": p - p * p}[case["op"]]
            none = (1 - q) ** 31
            b = 8 * L + 4 * n / 31 * (1 - none) * (1 + none)
    elif kind == "stages":
        k, L, K = _index_size(case["dist"], n, case["card"])
        b = 12 * n + 12 * n + (12 * n + 12 * k) + 12 * k + (8 * k + 4 * L) + (8 * k + 12 * K)
    else:
        b = 10 * n + 8 * n + 12 * n
    return {"bytes": float(b), "flops": 0.0}


# -- the same results from plain torch ---------------------------------------------
def _words_of(chunk, lit, first):
    """Fill and literal of each entry (its chunk, its bits, whether it is its
    key's first), zero fills dropped -> (words, word count per entry, fills)."""
    before = torch.cat([chunk.new_full((1,), -1), chunk[:-1]])
    fill = torch.where(first, chunk, chunk - before - 1)
    pairs = torch.stack([fill, lit | (1 << 31)], 1).view(-1)
    return pairs[pairs != 0], 1 + (fill != 0).to(torch.int64), fill


def _index(v32, rid_base):
    """Every array of a column's index in 64 bits."""
    v = v32.to(torch.int64) & 0xFFFFFFFF
    n = v.numel()
    keys, order = torch.sort(v, stable=True)
    rid = order + rid_base
    chunk = rid // 31
    bit = torch.ones_like(rid) << (rid % 31)
    new_key = torch.ones(n, device=DEV, dtype=torch.bool)
    new_key[1:] = keys[1:] != keys[:-1]
    new_entry = new_key.clone()
    new_entry[1:] |= chunk[1:] != chunk[:-1]
    at = torch.nonzero(new_entry).view(-1)
    upto = torch.cumsum(bit, 0)  # rows of one entry are different bits: their sum is their OR
    ends = torch.cat([at[1:], at.new_full((1,), n)]) - 1
    lit = upto[ends] - upto[at] + bit[at]
    del upto
    entry_key, entry_chunk, first = keys[at], chunk[at], new_key[at]
    words, per_entry, fill = _words_of(entry_chunk, lit, first)
    pos = torch.cumsum(per_entry, 0) - per_entry
    offsets = pos[first]
    lengths = torch.cat([offsets[1:], offsets.new_full((1,), words.numel())]) - offsets
    repeat = torch.zeros(n, device=DEV, dtype=torch.bool)
    rows = torch.arange(n, device=DEV) + rid_base
    repeat[1:] = (v[1:] == v[:-1]) & (rows[1:] % 31 != 0)
    items = n - int(repeat.sum())
    bits = int(v.max()), [bool(((v >> (8 * p)) & 255 != (v[0] >> (8 * p)) & 255).any())
                          for p in range(4)]
    return {"sorted": keys, "rids": rid, "chids": chunk, "lits": bit | (1 << 31),
            "mv": entry_key, "mc": entry_chunk, "ml": lit | (1 << 31), "fills": fill,
            "words": words, "keys": entry_key[first], "offsets": offsets, "lengths": lengths,
            "bound": bits[0], "passes": sum(bits[1]), "mode": int(3 * items < 2 * n)}


def _counts(x):
    c = np.zeros(1, np.dtype([("s", "<u8", 3), ("w", "<u4", 4)]))
    c["s"] = (x["mv"].numel(), x["words"].numel(), x["keys"].numel())
    c["w"] = (x["bound"], x["passes"], 0, x["mode"])
    return torch.from_numpy(c.view(np.int32).copy()).to(DEV)


def _build_exact(v, rid_base, out, at, column):
    x = _index(v, rid_base)
    for buf, name in zip(out, ("keys", "offsets", "lengths")):
        buf[at:at + x[name].numel()] = _as_i32(x[name])
    out[3][2 * at:2 * at + x["words"].numel()] = _as_i32(x["words"])
    out[4][column * COUNT_WORDS:(column + 1) * COUNT_WORDS] = _counts(x)


def _mask_words(mask):
    """WAH words of a bool tensor's rows."""
    rows = torch.nonzero(mask).view(-1)
    if not rows.numel():
        return torch.zeros(0, device=DEV, dtype=torch.int32)
    chunk, which = torch.unique_consecutive(rows // 31, return_inverse=True)
    lit = torch.zeros_like(chunk).index_add_(0, which, torch.ones_like(rows) << (rows % 31))
    first = torch.zeros(chunk.numel(), device=DEV, dtype=torch.bool)
    first[0] = True
    return _as_i32(_words_of(chunk, lit, first)[0])


def exact(case, seed):
    kind, n = case["kind"], case.get("n", 0)
    if kind == "build":
        out = _out(n)
        _build_exact(values_of(case["dist"], n, case["card"], seed), case["rid_base"], out, 0, 0)
        return out
    if kind == "batch":
        cols, total, values = batch_values(case, seed)
        out = _out(total, len(cols))
        for i, (at, m, _, _) in enumerate(cols):
            _build_exact(values[at:at + m], 0, out, at, i)
        return out
    if kind == "host":
        x = _index(relabelled(case, seed), case["rid_base"])
        return [_as_i32(x[k]) for k in ("keys", "offsets", "lengths", "words")] + \
            [x["mv"].numel(), x["words"].numel(), x["keys"].numel(), x["bound"], x["passes"],
             x["mode"]]
    if kind == "range":
        v = values_of("uniform", n, case["card"], seed)
        lo, hi = range_bounds(case)
        mask = (v >= lo) & (v <= hi)
        return bitmap_of(mask), int(torch.unique(v[mask]).numel())
    if kind == "codec":
        mask = codec_mask(case, seed)
        rows = torch.nonzero(mask).view(-1)
        return _mask_words(mask), bitmap_of(mask), int(rows[-1]) + 1 if rows.numel() else 0
    if kind == "combine":
        a, b = (v == v.min() for v in combine_columns(case, seed))
        return _mask_words({"and": a & b, "or": a | b, "xor": a ^ b, "andnot": a & ~b}[case["op"]])
    if kind == "stages":
        x = _index(relabelled(case, seed), 0)
        return [_as_i32(x[k]) for k in ("sorted", "rids", "chids", "lits", "mv", "mc", "ml",
                                        "fills", "words", "keys", "offsets", "lengths")]
    data, valid, heads = (t.to(torch.int64) for t in prims_inputs(case, seed))
    total = torch.cumsum(data, 0)
    head = heads != 0
    head[0] = True
    at = torch.nonzero(head).view(-1)
    before = (total - data)[at][torch.cumsum(head, 0) - 1]
    wrap = 0xFFFFFFFF
    return (data[valid != 0].to(torch.int32), _as_i32((total - data) & wrap),
            _as_i32((total - before) & wrap))
