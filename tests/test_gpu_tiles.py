"""Radix and tail tiles of one column where their number and their ends change:
one tile and a row, fewer tiles than the eight counter lanes, a number the
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
SIZES = [8193, T - 1, T, T + 1, 3 * T + 1, 9 * T - 1, 18 * T + 1, 65 * T - 1, 255 * T + 1,
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
        for n in (T + 1, 9 * T - 1, 65 * T - 1):
            v = column(kind, n)
            print(f"[tiles] match n={n} {kind}", flush=True)
            assert_same(c.build(v), oracle.build(v), f"{n} {kind}")
