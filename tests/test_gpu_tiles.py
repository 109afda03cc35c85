"""Short columns, which one workgroup builds, at the sizes where its rows per
thread change (1024, 4096, 8192, 16384), alone and in batches.  Radix and tail
tiles of longer ones where their number and their ends change: one tile and a row, fewer tiles than the eight counter lanes, a number the
lanes do not divide, as many tiles as blocks and one more, with last tiles of
one row and of all but one, over even and skewed digits, in both sort modes and
both rankings.  Against the oracle; whole numbers, so equal or wrong.
"""
import numpy as np
import pytest

import indexing_amd as ia
from oracle import oracle
from tests.test_gpu_parity import assert_same

pytestmark = pytest.mark.gpu

T = 16384  # rows of a radix tile (the tail's is 8192)
SIZES = [1, 2, 31, 63, 1023, 1024, 1025, 4095, 4096, 4097, 8191, 8192, 8193, T - 1, T, T + 1, 3 * T + 1, 9 * T - 1, 18 * T + 1, 65 * T - 1, 255 * T + 1,
         256 * T + 7]


def column(kind, n):
    rng = np.random.default_rng(n)
    if kind == "u16":
        return rng.integers(0, 65536, n).astype(np.uint32)
    if kind == "u32":
        return rng.integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32)
    if kind == "top":  # the highest key and digit 255 in most rows
        v = rng.integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32)
        return np.where(rng.random(n) < 0.9, np.uint32(0xFFFFFFFF), v)
    if kind == "skew":
        return np.minimum(rng.geometric(0.3, n), 300).astype(np.uint32)
    return np.repeat(rng.integers(0, 1 << 20, n // 40 + 1), 40)[:n].astype(np.uint32)


@pytest.mark.parametrize("kind", ["u16", "u32", "top", "skew", "runs"])
@pytest.mark.parametrize("n", SIZES)
def test_one_column(ctx, n, kind):
    v = column(kind, n)
    print(f"[tiles] n={n} {kind}", flush=True)
    assert_same(ctx.build(v, rid_base=n % 31), oracle.build(v, rid_base=n % 31), f"{n} {kind}")


@pytest.mark.parametrize("kind", ["u32", "top", "runs"])
def test_ballot_ranking(monkeypatch, kind):
    monkeypatch.setenv("WAHGPU_RANK", "match")
    with ia.Context(0) as c:
        assert c.rank_mode == 0
        for n in (1, 1000, 4097, 8193, T, T + 1, 9 * T - 1, 65 * T - 1):
            v = column(kind, n)
            print(f"[tiles] match n={n} {kind}", flush=True)
            assert_same(c.build(v), oracle.build(v), f"{n} {kind}")


@pytest.mark.parametrize("kind", ["u32", "top", "runs"])
def test_untuned_shape(ctx, kind):
    """A context without a tuning table takes its tile shape from the column's
    length: where it changes; and the shape that a table of zeros keeps."""
    from indexing_amd import _native as N
    for n in (2**20 - 1, 2**20, 2**21, 2**21 + 1):
        v = column(kind, n)
        print(f"[tiles] untuned n={n} {kind}", flush=True)
        assert_same(ctx.build(v), oracle.build(v, threads=8), f"{n} {kind}")
    with ia.Context(0) as c:
        c.set_tuning([0] * N.TUNE_BUCKETS)
        for n in (T + 1, 9 * T - 1, 18 * T + 1):
            v = column(kind, n)
            print(f"[tiles] table n={n} {kind}", flush=True)
            assert_same(c.build(v), oracle.build(v), f"{n} {kind}")


@pytest.mark.parametrize("reserve", [0, 2**22, 2**24], ids=["eager", "short", "long"])
def test_untuned_batch_shape(reserve):
    """A batch's one shape goes by the mean length of its columns, a graph's by
    that of the reservation."""
    import torch

    from tests.test_gpu_batch import per_column
    lens = [2**20 - 1, 2**20 + 1, 20001, 5] if reserve != 2**24 else [2**21 + 3, 17, T + 1, 40000]
    cols, refs, at = [], [], 0
    for i, n in enumerate(lens):
        cols.append((at, n, i))
        refs.append(oracle.build(column("u32", n), rid_base=i, threads=8))
        at += (n + 63) // 64 * 64
    buf = torch.zeros(at, dtype=torch.int32, device="cuda:0")
    for o, n, _ in cols:
        buf[o:o + n] = torch.from_numpy(column("u32", n).view(np.int32))
    with ia.Context(0) as c:
        if reserve:
            c.batch_reserve(reserve, 8)
        out = None
        for _ in range(3):
            out = c.build_batch_device(buf, cols) if out is None else \
                c.build_batch_device(buf, cols, out)
            counts = c.read_counts_batch(out[4], len(lens))
            got = per_column(out, counts, [(o, n) for o, n, _ in cols])
            for i, (g, r) in enumerate(zip(got, refs)):
                assert counts[i].fault == 0
                assert_same(g, r, f"reserve {reserve} column {i}")


@pytest.mark.parametrize("shape", [0, 1, 4])
@pytest.mark.parametrize("tiles", [4094, 4095, 4096])
def test_run_cut_units(shape, tiles):
    """The cut of a run-mode column goes by chunks below 4096 radix tiles and
    by tiles from there on; a last tile of one row and of all but one."""
    from indexing_amd import _native as N
    rows = {0: T, 1: T // 2, 4: T // 4}[shape]
    with ia.Context(0) as c:
        c.set_tuning([shape] * N.TUNE_BUCKETS)
        for n in (tiles * rows + 1, (tiles + 1) * rows - 1):
            v = column("runs", n)
            print(f"[tiles] cut shape={shape} n={n}", flush=True)
            assert_same(c.build(v, rid_base=7), oracle.build(v, rid_base=7, threads=8), f"{n}")


@pytest.mark.parametrize("reserved", [False, True], ids=["eager", "graph"])
def test_short_and_long_columns_in_one_batch(reserved):
    """Short columns take a workgroup each beside the launch set of the longer
    ones; a graph replays layouts with more, fewer and none of either."""
    import torch

    from tests.test_gpu_batch import per_column
    kinds = ["u16", "u32", "top", "skew", "runs"]
    layouts = [[1, 1000, 5000, 0, T, T + 1, 16000, 40000, 3], [7, 8192, 0, 1024] * 3,
               [T + 5, 60000], [T, 0, 20011]]
    total = max(sum(n + 3 for n in lay) for lay in layouts)
    with ia.Context(0) as c:
        if reserved:
            c.batch_reserve(total, 16)
        buf = torch.zeros(total, dtype=torch.int32, device="cuda:0")
        out = None
        for rep, lay in enumerate(layouts + layouts[:2]):
            cols, refs, at = [], [], rep % 2
            for i, n in enumerate(lay):
                v = column(kinds[(i + rep) % 5], n) if n else np.zeros(0, np.uint32)
                buf[at:at + n] = torch.from_numpy(v.view(np.int32))
                cols.append((at, n, 1000 * i))
                refs.append(oracle.build(v, rid_base=1000 * i))
                at += n + i % 3  # offsets off the 16-byte grid
            print(f"[batch] {lay} reserved={reserved}", flush=True)
            d = torch.zeros(16 * 10, dtype=torch.int32, device="cuda:0") if out is None else out[4]
            if out is None:
                out = tuple(torch.zeros(m, dtype=torch.int32, device="cuda:0")
                            for m in (total, total, total, 2 * total)) + (d,)
            c.build_batch_device(buf, cols, out)
            torch.cuda.synchronize()
            counts = c.read_counts_batch(out[4], len(lay))
            got = per_column(out, counts, [(o, n) for o, n, _ in cols])
            for i, (g, r) in enumerate(zip(got, refs)):
                assert counts[i].fault == 0
                assert_same(g, r, f"layout {rep} column {i}")
        if reserved:
            assert c.graph_stats()[0] == 1


def test_host_results_are_the_callers_own(monkeypatch):
    """Context.build hands out copies of what it keeps: an index stays as it was
    while the context builds others, longer than the kept memory's bound and
    shorter, from several threads, and after the context is closed."""
    from concurrent.futures import ThreadPoolExecutor
    monkeypatch.setattr(ia, "_STAGE_MAX", 30000)
    lens = [1, 20000, 16384, 0, 16385, 30000, 30001, 70001, 5]
    cols = [column("skew", n) for n in lens]
    with ia.Context(0) as c:
        got = [c.build(v) for v in cols]
        assert c._stage_lock.acquire(blocking=False)  # as if another call held the memory
        got.append(c.build(cols[1]))
        c._stage_lock.release()
    with ThreadPoolExecutor(3) as pool:
        def run(v):
            with ia.Context(0) as own:
                own.build(cols[-1])
                return own.build(v)
        got += pool.map(run, cols)
    for g, v in zip(got, cols + [cols[1]] + cols):
        assert_same(g, oracle.build(v), f"{v.size}")


@pytest.mark.parametrize("shape", [None, 3], ids=["untuned", "table"])
@pytest.mark.parametrize("reserved", [False, True], ids=["eager", "graph"])
def test_short_columns_join_the_long_ones(reserved, shape):
    """Few short columns beside long ones take part in their launch set, more
    of them or with less beside them do not; one graph replays all of these."""
    import torch

    from indexing_amd import _native as N
    from tests.test_gpu_batch import per_column
    layouts = [[5, 2**16, 0, 1], [5, 2**16 - 1, 1, 0], [16384, 7, 2**18, 0, 16383, 1, 1025],
               [3, 300000] + [4] * 8 + [9] * 200, [40] * 128 + [2**22], [40] * 129 + [2**22]]
    with ia.Context(0) as c:
        if shape is not None:
            c.set_tuning([shape] * N.TUNE_BUCKETS)
        total = 2**22 + 130 * 64
        if reserved:
            c.batch_reserve(total, 256)
        buf = torch.zeros(total, dtype=torch.int32, device="cuda:0")
        out = None
        for rep, lay in enumerate(layouts):
            cols, at = [], 0
            for i, n in enumerate(lay):
                v = column(("u16", "skew", "runs")[i % 3], n) if n else np.zeros(0, np.uint32)
                buf[at:at + n] = torch.from_numpy(v.view(np.int32))
                cols.append((at, n, i, v))
                at += (n + 63) // 64 * 64
            spec = [(o, n, r) for o, n, r, _ in cols]
            if out is None:
                out = tuple(torch.zeros(m, dtype=torch.int32, device="cuda:0")
                            for m in (total, total, total, 2 * total, 256 * 10))
            c.build_batch_device(buf, spec, out)
            torch.cuda.synchronize()
            counts = c.read_counts_batch(out[4], len(lay))
            got = per_column(out, counts, [(o, n) for o, n, _ in spec])
            for i, (g, col) in enumerate(zip(got, cols)):
                assert counts[i].fault == 0
                assert_same(g, oracle.build(col[3], rid_base=i), f"layout {rep} column {i}")
        if reserved:
            assert c.graph_stats()[0] == 1
