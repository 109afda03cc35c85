"""The single-pass scans at their edges: tiles of 4096, 8192 and 16384 elements
and the sizes where the tile changes, ragged ends, pointers off the 16-byte
grid, more tiles than resident blocks, segments and runs that span tiles, and
calls one after another (each launch leaves the scan state as it found it).
Whole numbers: results are equal or wrong.
"""
import numpy as np
import pytest

from oracle import oracle

pytestmark = pytest.mark.gpu

# rows of 256 per wave, tiles of 4096 / 8192 / 16384, the small-call limit 2^19,
# and more than 512 tiles of 16384
SIZES = [1, 3, 4, 5, 255, 257, 1023, 1025, 4095, 4096, 4097, 8191, 8193, 16385, (1 << 19) - 1,
         1 << 19, (1 << 19) + 1, 513 * 16384 + 7]


def u32(t):
    return t.detach().cpu().numpy().view(np.uint32)


def dev(a, shift=0):
    """On the device, `shift` words past an aligned address."""
    import torch
    a = np.ascontiguousarray(a, dtype=np.uint32).view(np.int32)
    buf = torch.zeros(a.size + shift, dtype=torch.int32, device="cuda:0")
    buf[shift:] = torch.from_numpy(a).to("cuda:0")
    return buf[shift:]


@pytest.mark.parametrize("n", SIZES)
def test_scans_and_compaction(ctx, n):
    rng = np.random.default_rng(n)
    data = rng.integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32)
    want_ex = oracle.exclusive_scan(data)
    for kind, shift in (("sparse", 0), ("none", 1), ("all", 2), ("dense", 3)):
        p = {"sparse": 0.0005, "none": 0.0, "all": 1.0, "dense": 0.5}[kind]
        flags = (rng.random(n) < p).astype(np.uint32) * rng.integers(1, 1 << 32, n, dtype=np.uint64).astype(np.uint32)
        print(f"[scan] n={n} {kind} shift={shift}", flush=True)
        assert np.array_equal(u32(ctx.exclusive_scan(dev(data, shift))), want_ex)
        got = ctx.segmented_inclusive_scan(dev(data, shift), dev(flags, 3 - shift))
        assert np.array_equal(u32(got), oracle.segmented_inclusive_scan(data, flags))
        got = ctx.stream_compaction(dev(data, shift), dev(flags, 3 - shift))
        assert np.array_equal(u32(got), data[flags != 0])


@pytest.mark.parametrize("n", SIZES)
def test_merge_fuse_and_column_length(ctx, n):
    rng = np.random.default_rng(n + 1)
    for mean, shift in ((1, 1), (3, 0), (20000, 2)):  # mean run length of (value, chunk)
        start = rng.random(n) < 1.0 / mean
        start[0] = True
        chunk = np.cumsum(start).astype(np.uint32)  # ascending, so runs never meet again
        value = (chunk // 7).astype(np.uint32)
        lits = (1 << rng.integers(0, 31, n)).astype(np.uint32) | np.uint32(0x80000000)
        print(f"[merge] n={n} mean={mean} shift={shift}", flush=True)
        mv, mc, ml = ctx.merge_lit_by_val_chids(dev(value, shift), dev(chunk, 1), dev(lits, shift))
        at = np.flatnonzero(start)
        assert np.array_equal(u32(mv), value[at])
        assert np.array_equal(u32(mc), chunk[at])
        assert np.array_equal(u32(ml), np.bitwise_or.reduceat(lits, at))
        fills = rng.integers(0, 3, at.size).astype(np.uint32)
        kept = u32(ml).copy()
        kept[rng.random(at.size) < 0.1] = 0  # zero words are dropped on either side
        words = np.stack([fills, kept], 1).reshape(-1)
        assert np.array_equal(u32(ctx.fuse_fill_literals(dev(fills, shift), dev(kept, 3))),
                              words[words != 0])
        keys, offs, lens = ctx.compute_column_length(dev(value[at], shift), dev(fills, 1))
        first = np.flatnonzero(np.concatenate([[True], value[at][1:] != value[at][:-1]]))
        per = 1 + (fills != 0).astype(np.int64)
        pos = np.concatenate([[0], np.cumsum(per)])
        assert np.array_equal(u32(keys), value[at][first])
        assert np.array_equal(u32(offs), pos[first])
        assert np.array_equal(u32(lens), np.diff(np.append(pos[first], pos[-1])))


def test_scan_replayed_from_a_graph(ctx):
    import torch
    n = 100_003
    rng = np.random.default_rng(7)
    src = dev(np.zeros(n))
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        ctx.exclusive_scan(src)  # binds the context to the stream before the capture
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            out = ctx.exclusive_scan(src)
        for _ in range(3):
            data = rng.integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32)
            src.copy_(dev(data))
            g.replay()
            torch.cuda.synchronize()
            assert np.array_equal(u32(out), oracle.exclusive_scan(data))
            # eager work between the replays, on the same scan state
            assert np.array_equal(u32(ctx.stream_compaction(dev(data), dev(data & 1))),
                                  data[(data & 1) != 0])
