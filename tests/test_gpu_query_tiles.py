"""Decode, encode and combine where their tiles end and where a literal meets
words the builds never write: streams of a decode tile's words (4096) give or
take one, bitmaps of an encode tile's chunks (4096) give or take a row, 1-fills
and fills of no chunks beside literals, rows past nrows, and outputs one word
short.  Whole numbers: results are equal or wrong.
"""
import numpy as np
import pytest

from indexing_amd import WahError
from tests.test_gpu_query import bitmap_rows, canonical_words, rows_to_bitmap
from tests.test_gpu_scan import dev, u32

pytestmark = pytest.mark.gpu


def decode_rows(words):
    """Rows of a word stream, from the word format alone."""
    rows, chunk = [], 0
    for w in np.asarray(words, np.uint64).tolist():
        if w & 0x80000000:
            rows += [31 * chunk + b for b in range(31) if (w >> b) & 1]
            chunk += 1
        else:
            n = w & 0x3FFFFFFF
            if w & 0x40000000:
                rows += range(31 * chunk, 31 * (chunk + n))
            chunk += n
    return np.array(rows, np.int64), chunk


def stream(n, seed, odd):
    """n words: literals in runs (their bitmap words are shared), 0-fills, and
    if odd 1-fills, fills of no chunks and empty literals among them."""
    rng = np.random.default_rng(seed)
    lit = (rng.integers(0, 1 << 31, n) | 0x80000000).astype(np.uint32)
    one = ((1 << rng.integers(0, 31, n)) | 0x80000000).astype(np.uint32)
    fill = rng.integers(1, 40, n).astype(np.uint32)
    pick = rng.random(n)
    w = np.where(pick < 0.4, lit, np.where(pick < 0.7, one, fill))
    if odd:
        kind = rng.random(n)
        w = np.where(kind < 0.05, fill | 0x40000000, w)
        w = np.where((kind >= 0.05) & (kind < 0.10), np.uint32(0), w)
        w = np.where((kind >= 0.10) & (kind < 0.15), np.uint32(0x80000000), w)
        w = np.where((kind >= 0.15) & (kind < 0.18), np.uint32(0x40000000), w)
    return w.astype(np.uint32)


@pytest.mark.parametrize("odd", [False, True], ids=["canonical", "odd"])
@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 511, 513, 4095, 4096, 4097, 12289])
def test_decode_streams(ctx, n, odd):
    words = stream(n, 10 * n + odd, odd)
    rows, chunks = decode_rows(words)
    for nrows in sorted({max(1, 31 * chunks), max(1, 31 * chunks - 17), max(1, 31 * chunks // 2),
                         31 * chunks + 100, 1}):
        print(f"[decode] n={n} odd={odd} nrows={nrows}", flush=True)
        bm, last = ctx.decode_device(dev(words, n % 4), nrows)
        assert np.array_equal(bitmap_rows(u32(bm), nrows), rows[rows < nrows])
        assert not bitmap_rows(u32(bm), u32(bm).size * 32)[rows[rows < nrows].size:].size
        assert last == (int(rows[-1]) + 1 if rows.size else 0)


def test_decode_drops_what_lies_past_every_row(ctx):
    """Fills that sum past 2^32 chunks: what follows them lies past nrows."""
    words = np.concatenate([[0x80000005], np.full(6, 0x3FFFFFFF), [0x80000003] * 5000])
    bm, _ = ctx.decode_device(dev(words.astype(np.uint32)), 100_000)
    assert bitmap_rows(u32(bm), 100_000).tolist() == [0, 2]


@pytest.mark.parametrize("chunks", [511, 512, 513, 4095, 4096, 4097, 8193])
@pytest.mark.parametrize("extra", [-30, -1, 0, 1])
def test_encode_at_tile_ends(ctx, chunks, extra):
    n = 31 * chunks + extra
    rng = np.random.default_rng(n)
    # nothing, the last row alone, the first chunk of the last tile alone, dense
    # up to the tile's end, scattered
    for rows in ([], [n - 1], [min(n - 1, 31 * (chunks // 4096 * 4096))], np.arange(n),
                 np.flatnonzero(rng.random(n) < 0.01), np.flatnonzero(rng.random(n) < 0.3)):
        want = canonical_words(rows)
        print(f"[encode] rows={n} set={len(rows)}", flush=True)
        got = ctx.encode_device(dev(rows_to_bitmap(rows, n), n % 3), n)
        assert np.array_equal(u32(got), want)
        if want.size > 1:
            with pytest.raises(WahError):
                ctx.encode_device(dev(rows_to_bitmap(rows, n)), n, cap=want.size - 1)


def test_encode_ignores_rows_past_the_end_and_writes_none_past_cap(ctx):
    import ctypes

    import torch

    from indexing_amd import _ptr
    n = 31 * 5000 + 7
    bits = np.full((n + 31) // 32, 0xFFFFFFFF, np.uint32)
    assert np.array_equal(u32(ctx.encode_device(dev(bits), n)), canonical_words(np.arange(n)))
    out = torch.full((6000,), 7, dtype=torch.int32, device="cuda:0")
    length = ctypes.c_uint64(0)
    ctx._bind_stream()
    rc = ctx._lib.wahgpu_encode_device(ctx._h, _ptr(dev(bits)), n, _ptr(out), 4990,
                                       ctypes.byref(length))
    assert rc != 0 and length.value == 5001
    assert bool((out[4990:] == 7).all()) and bool((out[:4990] != 7).all())


@pytest.mark.parametrize("op", ["and", "or", "xor", "andnot"])
def test_combine_of_unequal_streams(ctx, op):
    a, b = stream(4097, 1, True), stream(300, 2, False)
    for x, y in ((a, b), (b, a), (a, b[:0]), (b[:0], a)):
        (rx, cx), (ry, cy) = decode_rows(x), decode_rows(y)
        n = 31 * max(cx, cy) - 5
        sx, sy = (np.isin(np.arange(n), r) for r in (rx, ry))
        want = {"and": sx & sy, "or": sx | sy, "xor": sx ^ sy, "andnot": sx & ~sy}[op]
        got = ctx.combine_device(op, dev(x), dev(y), n, cap=2 * (n // 31 + 1))
        assert np.array_equal(u32(got), canonical_words(np.flatnonzero(want)))


@pytest.mark.parametrize("card", [2, 97, 5000])
def test_range_over_many_keys_per_tile(ctx, card):
    rng = np.random.default_rng(card)
    n = 200_003
    v = rng.integers(0, card, n).astype(np.uint32)
    idx = ctx.build(v)
    k, o, ln, w = (dev(x) for x in (idx.keys, idx.offsets, idx.lengths, idx.words))
    for lo, hi in ((0, card), (card // 3, card // 2), (card - 1, card - 1), (card, card + 9),
                   (1, 0xFFFFFFFF), (5, 4)):
        bm, m = ctx.query_range_device(k, o, ln, w, lo, hi, n)
        sel = (v >= lo) & (v <= hi)
        assert np.array_equal(bitmap_rows(u32(bm), n), np.flatnonzero(sel))
        assert m == np.unique(v[sel]).size


SLICED = 1 << 22  # rows from which a range may decode by slices of the bitmap


@pytest.mark.parametrize("arena", [0, 1 << 12, 1 << 30], ids=["grows", "no-room", "room"])
@pytest.mark.parametrize("n", [SLICED - 1, SLICED, SLICED + 31 * 1024 - 17, 2 * SLICED + 5,
                               31 * 8192 * 256 - 1, 31 * 8192 * 256 + 1])
def test_range_by_slices(n, arena):
    """Ranges of few and many words per key and slice, on either side of where
    the slices' size and the way of decoding change."""
    import torch

    import indexing_amd as ia
    with ia.Context(0) as c:
        g = torch.Generator(device="cuda:0").manual_seed(n)
        for card in (3, 100, 3000):
            v = torch.randint(0, card, (n,), device="cuda:0", generator=g, dtype=torch.int32)
            v[n // 3:n // 2] = 0  # slices that most keys skip
            v[-1] = card - 1
            with ia.Context(0, arena_bytes=arena) as q:
                k, o, ln, w, counts = c.build_device(v)
                m, L = c.read_counts(counts).keycnt, c.read_counts(counts).length
                for lo, hi in ((0, card), (card // 3, card // 2), (card - 1, card - 1), (1, 1)):
                    print(f"[range] n={n} card={card} [{lo}, {hi}]", flush=True)
                    try:
                        bm, keys = q.query_range_device(k[:m], o[:m], ln[:m], w[:L], lo, hi, n)
                    except WahError:
                        assert arena == 1 << 12  # the words' own limit
                        continue
                    sel = (v >= lo) & (v <= hi)
                    pad = torch.zeros((n + 31) // 32 * 32, dtype=torch.int64, device="cuda:0")
                    pad[:n] = sel
                    want = (pad.view(-1, 32) << torch.arange(32, device="cuda:0")).sum(1)
                    assert bool((bm.to(torch.int64) & 0xFFFFFFFF == want).all())
                    assert keys == int(torch.unique(v[sel]).numel())


@pytest.mark.parametrize("seed", [1, 2])
def test_range_by_slices_of_words_that_builds_never_write(ctx, seed):
    """1-fills and fills over several slices, fills of no chunks, empty
    literals and a key without words."""
    rng = np.random.default_rng(seed)
    n = SLICED + 1000
    chunks = (n + 30) // 31
    streams = []
    for k in range(40):
        w = stream(12000 + 517 * k, 100 * seed + k, True)
        if k % 5 == 1:  # a fill over several slices, of ones or not
            w[rng.integers(w.size)] = np.uint32(5000 | (0x40000000 if k % 2 else 0))
        if k == 7:
            w = w[:0]
        streams.append(w)
    words = np.concatenate(streams)
    lengths = np.array([s.size for s in streams], np.uint32)
    offsets = (np.cumsum(lengths) - lengths).astype(np.uint32)
    keys = np.arange(40, dtype=np.uint32) * 3
    rows = [decode_rows(s)[0] for s in streams]
    assert max(int(r[-1]) for r in rows if r.size) > n and chunks > 130 * 1024
    d = [dev(x) for x in (keys, offsets, lengths, words)]
    for lo, hi in ((0, 200), (20, 22), (21, 21), (30, 90)):
        bm, m = ctx.query_range_device(*d, lo, hi, n)
        take = [i for i in range(40) if lo <= 3 * i <= hi]
        want = np.unique(np.concatenate([rows[i] for i in take])) if take else np.zeros(0, np.int64)
        assert np.array_equal(bitmap_rows(u32(bm), n), want[want < n])
        assert m == len(take)


@pytest.mark.parametrize("n", [100_000, SLICED + 31], ids=["small", "sliced"])
@pytest.mark.parametrize("drop", [1, 2047, 5000, 1 << 31])
def test_range_whose_offsets_descend_is_refused(ctx, n, drop):
    """An index whose last key of the range ends before its first one begins:
    refused with an empty bitmap (nothing of it is decoded); the same index in
    order decodes."""
    import ctypes

    import torch

    from indexing_amd import _ptr
    words = dev(np.full(8000, 0x80000001, np.uint32))
    keys = dev(np.arange(3, dtype=np.uint32))
    lengths = dev(np.array([10, 10, 7], np.uint32))
    first = drop + 7  # the last key ends `drop` words before it
    good = [0, 10, 20]
    bitmap = torch.full(((n + 31) // 32,), -1, dtype=torch.int32, device="cuda:0")
    found = ctypes.c_uint64(0)
    for offsets in ([first, 5, 0], good):
        ctx._bind_stream()
        print(f"[descend] n={n} offsets={offsets}", flush=True)
        rc = ctx._lib.wahgpu_query_range_device(
            ctx._h, _ptr(keys), _ptr(dev(np.array(offsets, np.uint32))), _ptr(lengths), 3,
            _ptr(words), 0, 9, n, _ptr(bitmap), ctypes.byref(found))
        assert found.value == 3
        if offsets is good:
            assert rc == 0 and np.array_equal(bitmap_rows(u32(bitmap), n), 31 * np.arange(10))
        else:
            assert rc == -1 and not bool(bitmap.any())


def test_keys_that_descend_match_none(ctx):
    words = dev(np.full(100, 0x80000001, np.uint32))
    keys, offsets = dev(np.array([9, 5, 1], np.uint32)), dev(np.array([0, 1, 2], np.uint32))
    for lo, hi in ((6, 7), (2, 3), (0, 9)):
        bm, m = ctx.query_range_device(keys, offsets, dev(np.ones(3)), words, lo, hi, 1000)
        assert 0 <= m <= 3 and set(bitmap_rows(u32(bm), 1000).tolist()) <= {0}


@pytest.mark.parametrize("n", [2_000_003, SLICED + 31], ids=["small", "sliced"])
def test_range_on_a_fixed_arena_is_whole_or_untouched(ctx, n):
    """In an arena of the bytes that a range's words count as, it decodes; in one
    a step (2 MiB) short of them, or of a step, the call is refused with the
    bitmap empty and the keys counted."""
    import ctypes

    import torch

    import indexing_amd as ia
    from indexing_amd import _ptr
    step = 2 << 20
    rng = np.random.default_rng(n)
    v = rng.integers(0, 60, n).astype(np.uint32)
    idx = ctx.build(v)
    k, o, ln, w = (dev(x) for x in (idx.keys, idx.offsets, idx.lengths, idx.words))
    words = int(idx.lengths[5:41].sum())
    need = -(-(2080 + -(-words // 2048) * 8) // 256) * 256 + -(-4 * words // 256) * 256
    assert need > step
    for arena, room in ((need, True), (need // step * step, need % step == 0), (step, False)):
        with ia.Context(0, arena_bytes=arena) as q:
            bitmap = torch.full(((n + 31) // 32,), -1, dtype=torch.int32, device="cuda:0")
            found = ctypes.c_uint64(0)
            q._bind_stream()
            print(f"[fixed] n={n} need={need} arena={q.arena_bytes()}", flush=True)
            rc = q._lib.wahgpu_query_range_device(q._h, _ptr(k), _ptr(o), _ptr(ln), k.numel(),
                                                  _ptr(w), 5, 40, n, _ptr(bitmap),
                                                  ctypes.byref(found))
            assert found.value == 36 and (rc == 0) == room
            want = np.flatnonzero((v >= 5) & (v <= 40)) if room else np.zeros(0, np.int64)
            assert np.array_equal(bitmap_rows(u32(bitmap), n), want)


@pytest.mark.parametrize("arena", [0, 1 << 28], ids=["grows", "fixed"])
def test_range_of_more_keys_than_the_first_table_holds(arena):
    """5000 keys of 2^24 rows need 1.28 million entries, the first table has 2^20:
    the range comes back for its own; narrower ones before and after it."""
    import torch

    import indexing_amd as ia
    n, card = 1 << 24, 5003
    g = torch.Generator(device="cuda:0").manual_seed(5)
    v = torch.randint(0, card, (n,), device="cuda:0", generator=g, dtype=torch.int32)
    with ia.Context(0) as c, ia.Context(0, arena_bytes=arena) as q:
        k, o, ln, w, counts = c.build_device(v)
        m, L = c.read_counts(counts).keycnt, c.read_counts(counts).length
        for lo, hi in ((7, 300), (2, 5001), (2, 5001), (4000, 4800), (17, 17)):
            print(f"[range] card={card} arena={arena} [{lo}, {hi}]", flush=True)
            bm, keys = q.query_range_device(k[:m], o[:m], ln[:m], w[:L], lo, hi, n)
            sel = ((v >= lo) & (v <= hi)).to(torch.int64).view(-1, 32)
            want = (sel << torch.arange(32, device="cuda:0")).sum(1)
            assert bool((bm.to(torch.int64) & 0xFFFFFFFF == want).all())
            assert keys == hi - lo + 1


def test_streams_of_more_words_than_a_context_starts_with():
    """More than 2^29 words (0-fills of a chunk with literals among them): a decode
    and ranges on either side of the slices grow the context's status words; the
    scans before and after it are as ever."""
    import torch

    import indexing_amd as ia
    total, half = (1 << 29) + 3 * 4096 + 5, (1 << 28) + 777
    words = torch.ones(total, dtype=torch.int32, device="cuda:0")
    at = torch.cat([torch.arange(0, 4000, 7), torch.tensor([40_000, 135_290, total - 1])])
    lit = -0x80000000 + (1 << 30) + 1  # rows 0 and 30 of the chunk
    words[at.to("cuda:0")] = lit
    second = torch.tensor([3, 40_001, 135_299])  # of the second key
    words[(half + second).to("cuda:0")] = lit

    def rows(*chunks):
        r = torch.cat([torch.cat([31 * c, 31 * c + 30]) for c in chunks])
        return np.unique(r.numpy())
    small = dev(np.arange(5000))
    with ia.Context(0) as c:
        for nrows in (100_000, SLICED + 5):
            print(f"[long] decode and range, nrows={nrows}", flush=True)
            assert int(c.exclusive_scan(small)[-1]) == 4999 * 4998 // 2
            bm, last = c.decode_device(words, nrows)
            want = rows(at)
            assert np.array_equal(bitmap_rows(u32(bm), nrows), want[want < nrows])
            assert last == 31 * total
            keys, offsets = dev(np.array([4, 9])), dev(np.array([0, half]))
            bm, m = c.query_range_device(keys, offsets, dev(np.array([half, total - half])), words,
                                         0, 10, nrows)
            want = rows(at[at < half], second)
            assert m == 2 and np.array_equal(bitmap_rows(u32(bm), nrows), want[want < nrows])


def long_stream(n, seed, odd):
    """n words whose fills are short, so that their chunks fit a bit array."""
    rng = np.random.default_rng(seed)
    w = (rng.integers(0, 1 << 31, n) | 0x80000000).astype(np.uint32)
    kind = rng.random(n)
    w[kind < 0.3] = rng.integers(1, 4, n)[kind < 0.3]
    if odd:
        w[kind < 0.04] = 0x40000000 | rng.integers(0, 4, n)[kind < 0.04]  # 1-fills, some of nothing
        w[(kind >= 0.04) & (kind < 0.06)] = 0
        w[(kind >= 0.06) & (kind < 0.08)] = 0x80000000
    return w


def stream_bits(words):
    """Rows of a stream as an array of bits, 31 per chunk."""
    lit = (words >> 31) == 1
    chunks = np.where(lit, 1, words & 0x3FFFFFFF).astype(np.int64)
    start = np.cumsum(chunks) - chunks
    payload = np.zeros(int(chunks.sum()), np.uint32)
    payload[start[lit]] = words[lit] & 0x7FFFFFFF
    ones = (words >> 30) == 1
    edge = np.zeros(payload.size + 1, np.int64)
    np.add.at(edge, start[ones], 1)
    np.add.at(edge, (start + chunks)[ones], -1)
    payload[np.cumsum(edge)[:-1] > 0] = 0x7FFFFFFF
    bits = np.unpackbits(payload.view(np.uint8).reshape(-1, 4), axis=1, bitorder="little")
    return bits[:, :31].reshape(-1)


def pack(bits):
    out = np.zeros((bits.size + 31) // 32 * 4, np.uint8)
    out[:(bits.size + 7) // 8] = np.packbits(bits, bitorder="little")
    return out.view(np.uint32)


def canonical_of(bits):
    """The words of an array of bits: a fill where chunks were skipped, then the
    literal, per chunk with a row."""
    chunks = np.zeros((bits.size + 30) // 31 * 31, np.uint8)
    chunks[:bits.size] = bits
    payload = np.zeros((chunks.size // 31, 32), np.uint8)
    payload[:, :31] = chunks.reshape(-1, 31)
    payload = np.packbits(payload, axis=1, bitorder="little").view(np.uint32).reshape(-1)
    at = np.flatnonzero(payload)
    fill = np.diff(at, prepend=-1) - 1
    words = np.stack([fill.astype(np.uint32), payload[at] | np.uint32(0x80000000)], 1).reshape(-1)
    return words[words != 0]


@pytest.mark.parametrize("odd", [False, True], ids=["canonical", "odd"])
def test_decode_of_more_tiles_than_blocks(ctx, odd):
    """More tiles than a launch has blocks (512), so blocks draw theirs and the
    look-back goes over many windows; twice, on the state the first left."""
    words = long_stream(600 * 4096 + 77, 3 + odd, odd)
    bits = stream_bits(words)
    for nrows in (bits.size, bits.size // 2 + 5):
        want, last = pack(bits[:nrows]), int(np.flatnonzero(bits)[-1]) + 1
        for rep in range(2):
            print(f"[decode] odd={odd} nrows={nrows} {rep}", flush=True)
            bm, got = ctx.decode_device(dev(words, rep), nrows)
            assert np.array_equal(u32(bm), want) and got == last


@pytest.mark.parametrize("density", [0.0005, 0.02, 0.6])
def test_encode_of_more_tiles_than_blocks(ctx, density):
    n = 31 * 4096 * 1100 + 1234  # 1100 tiles and a part, 1024 blocks
    bits = (np.random.default_rng(9).random(n, dtype=np.float32) < density).astype(np.uint8)
    bits[n // 4:n // 4 + 31 * 4096 * 70] = 0  # more than a window of tiles without a row
    want, bitmap = canonical_of(bits), dev(pack(bits))
    for rep in range(2):
        print(f"[encode] density={density} {rep}", flush=True)
        assert np.array_equal(u32(ctx.encode_device(bitmap, n)), want)


@pytest.mark.parametrize("op", ["and", "xor"])
def test_combine_of_long_streams(ctx, op):
    """The second stream's tiles start past the first look-back window, and both
    streams' together are more than the blocks."""
    a, b = long_stream(300 * 4096 + 5, 21, True), long_stream(280 * 4096 + 900, 22, False)
    x, y = stream_bits(a), stream_bits(b)
    n = min(x.size, y.size) - 7
    want = canonical_of(x[:n] & y[:n] if op == "and" else x[:n] ^ y[:n])
    for rep in range(2):
        assert np.array_equal(u32(ctx.combine_device(op, dev(a), dev(b), n)), want)
