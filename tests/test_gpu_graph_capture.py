"""A caller captures the device-pointer builds into its own graph.

wahgpu_build_device returns nothing to the host, and
wahgpu_build_device_noalloc allocates nothing: both can be captured (torch's
CUDAGraph on a stream the context is bound to beforehand; the first, eager
build sizes the arena, so the captured call allocates nothing either).  The
graph is replayed over different inputs written into the captured input
buffer, with eager work and synchronizations between the replays, and every
replay is compared with the oracle (src/cpu.cpp:313-328).
"""
import numpy as np
import pytest

import indexing_amd as ia
from oracle import oracle
from tests.test_gpu_batch import per_column
from tests.test_gpu_parity import assert_same, dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("noalloc", [False, True], ids=["build_device", "noalloc"])
def test_build_captured_and_replayed(noalloc):
    import torch
    n = (1 << 20) + 77
    inputs = [ia.generate(n, "uniform", seed=90 + i, lo=0, hi=(1 << (8 + 3 * i)) - 1)
              for i in range(3)]
    c = ia.Context(0)
    s = torch.cuda.Stream()
    build = c.build_device_noalloc if noalloc else c.build_device
    try:
        d_in = dev(inputs[0])
        with torch.cuda.stream(s):
            out = build(d_in)     # binds the context to s and sizes its arena
            build(d_in, out=out)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        print(f"[capture] noalloc={noalloc}", flush=True)
        with torch.cuda.graph(g, stream=s):
            build(d_in, out=out)
        for rep, v in enumerate(inputs):
            d_in.copy_(dev(v))
            x = torch.ones(1 << 20, device="cuda:0").sum()  # eager work between replays
            g.replay()
            torch.cuda.synchronize()
            assert float(x) == float(1 << 20)
            cnt = c.read_counts(out[4])
            assert cnt.fault == 0
            got = per_column(out, [cnt], [(0, n)])[0]
            assert_same(got, oracle.build(v), f"replay {rep}")
    finally:
        c.close()


@pytest.mark.parametrize("segmented", [False, True], ids=["scan", "segmented"])
def test_scan_replayed_beside_the_contexts_own_work(ctx, segmented):
    """Replays on one stream while the context scans and compacts on another:
    every result is right, and so are those after it.  (Few tiles: all blocks of
    both have a place, so no wait depends on the order.)"""
    import torch
    n = 100_003
    rng = np.random.default_rng(11)
    data = rng.integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32)
    heads = (rng.random(n) < 0.001).astype(np.uint32)
    src, flags = dev(data), dev(heads)
    replayed, own = torch.cuda.Stream(), torch.cuda.Stream()

    def scan():
        return ctx.segmented_inclusive_scan(src, flags) if segmented else ctx.exclusive_scan(src)
    want = oracle.segmented_inclusive_scan(data, heads) if segmented else oracle.exclusive_scan(data)
    with torch.cuda.stream(replayed):
        scan()
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=replayed):
            out = scan()
    torch.cuda.synchronize()
    for rep in range(10):
        print(f"[replay] {rep} segmented={segmented}", flush=True)
        out.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(replayed):
            for _ in range(8):
                g.replay()
        with torch.cuda.stream(own):
            for _ in range(4):
                eager = scan()
                kept = ctx.stream_compaction(src, flags)
                assert np.array_equal(kept.cpu().numpy().view(np.uint32), data[heads != 0])
        torch.cuda.synchronize()
        for got in (out, eager):
            assert np.array_equal(got.cpu().numpy().view(np.uint32), want)


def test_a_short_column_warms_up_for_a_captured_longer_one():
    """The first call sizes the arena for some 80000 rows, also where it needs
    none itself."""
    import torch
    n = 50_000
    inputs = [ia.generate(n, "uniform", seed=i, lo=0, hi=5000) for i in range(3)]
    s = torch.cuda.Stream()
    with ia.Context(0) as c:
        d_in = dev(inputs[0])
        out = tuple(torch.zeros(m, dtype=torch.int32, device="cuda:0") for m in (n, n, n, 2 * n, 16))
        with torch.cuda.stream(s):
            c.build_device(d_in[:1000])
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            c.build_device(d_in, out=out)
        for rep, v in enumerate(inputs):
            d_in.copy_(dev(v))
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            cnt = c.read_counts(out[4])
            assert cnt.fault == 0
            assert_same(per_column(out, [cnt], [(0, n)])[0], oracle.build(v), f"replay {rep}")
