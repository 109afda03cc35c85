"""Host code of the C ABI (indexing_amd/csrc/wahgpu_api.hip) on the CPU: compiled
with g++ against tests/api_harness, whose launchers compute nothing but hand the
host what a test scripts, a given fault among it.  What the entry points do with
that, how much memory they take, and what they refuse.
"""
import ctypes
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HARNESS = os.path.join(ROOT, "tests", "api_harness")
CSRC = os.path.join(ROOT, "indexing_amd", "csrc")
OK, EINVAL, ENOMEM, EHIP = 0, -1, -2, -3
U64, VP = ctypes.c_uint64, ctypes.c_void_p


def u64(x):
    return U64(int(x))


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not installed")
    so = str(tmp_path_factory.mktemp("api") / "libapi.so")
    r = subprocess.run(["g++", "-shared", "-fPIC", "-std=c++17", "-O1", "-g", "-Wall", "-I" + HARNESS,
                        "-I" + os.path.join(ROOT, "include"), "-I" + CSRC,
                        "-x", "c++", os.path.join(CSRC, "wahgpu_api.hip"),
                        os.path.join(HARNESS, "fake_gpu.cpp"), os.path.join(CSRC, "wah_host.cpp"),
                        "-o", so], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    x = ctypes.CDLL(so)
    x.fake_log.restype = ctypes.c_char_p
    x.fake_device_bytes.restype = U64
    x.wahgpu_arena_bytes.restype = U64
    x.wahgpu_last_error.restype = ctypes.c_char_p
    x.wahgpu_stream.restype = VP
    return x


class Ctx:
    """A context and one buffer that stands for every device pointer."""

    def __init__(self, lib, arena=0):
        self.lib, self.h = lib, VP()
        self.buf = VP(256)  # (the launchers read nothing)
        assert lib.wahgpu_create(ctypes.byref(self.h), 0, u64(arena)) == OK
        lib.fake_reset()

    def close(self):
        self.lib.wahgpu_destroy(self.h)

    def call(self, name, *args):
        """An entry point; integers are 64-bit, None is the buffer."""
        conv = [self.buf if a is None else u64(a) if isinstance(a, int) else a for a in args]
        return getattr(self.lib, "wahgpu_" + name)(self.h, *conv)

    def script(self, name, fault=0, result=0, extra=(0, 0), ends=True):
        self.lib.fake_script(name.encode(), int(ends), u64(fault), u64(result), u64(extra[0]),
                             u64(extra[1]))

    def log(self):
        return self.lib.fake_log().decode().splitlines()

    def error(self):
        return self.lib.wahgpu_last_error(self.h).decode()


@pytest.fixture
def ctx(lib):
    c = Ctx(lib)
    yield c
    c.close()


@pytest.mark.parametrize("segmented", [False, True])
@pytest.mark.parametrize("next_call", ["synchronize", "compaction", "build"])
def test_fault_of_an_asynchronous_scan_is_reported(ctx, segmented, next_call):
    """A scan that nobody waits for and that gave up: the next call that waits
    says so, once."""
    out = U64(77)
    counts = (ctypes.c_uint64 * 8)()

    def waits():
        if next_call == "synchronize":
            return ctx.call("synchronize")
        if next_call == "compaction":
            return ctx.call("stream_compaction", None, None, 100, None, ctypes.byref(out))
        return ctx.call("build", (ctypes.c_uint32 * 4)(), 4, ctypes.c_uint32(0), None, None, None,
                        100, None, 100, counts, VP())

    ctx.script("scan", fault=1)
    if segmented:
        assert ctx.call("segmented_inclusive_scan", None, None, 100, None) == OK
    else:
        assert ctx.call("exclusive_scan", None, 100, None) == OK
    assert ctx.call("exclusive_scan", None, 100, None) == OK  # a good one takes nothing back
    assert waits() == EHIP
    assert "earlier" in ctx.error() and "scan" in ctx.error()
    assert waits() == OK


@pytest.mark.parametrize("segmented", [False, True])
def test_captured_scans_have_a_state_of_their_own(ctx, segmented):
    """Replays are outside the order of the context's calls: they share no
    counters with them, and clear their own."""
    def scan():
        if segmented:
            return ctx.call("segmented_inclusive_scan", None, None, 1000, None)
        return ctx.call("exclusive_scan", None, 1000, None)
    stream = VP(ctx.lib.wahgpu_stream(ctx.h))
    assert scan() == OK
    ctx.lib.fake_capture(stream, 1)
    assert scan() == OK
    ctx.lib.fake_capture(stream, 0)
    assert scan() == OK
    assert ctx.call("stream_compaction", None, None, 1000, None, ctypes.byref(U64())) == OK
    before, held, after, other = [x for x in ctx.log() if "state=" in x]
    state = [x.split("state=")[1].split()[0] for x in (before, held, after, other)]
    assert state[0] == state[2] == state[3] != state[1]
    assert ["captured=1" in x for x in (before, held, after, other)] == [False, True, False, False]


# entry point -> (launcher, arguments): one of each kind that waits
WAITING = {
    "merge_lit_by_val_chids": ("merge", lambda o: (None,) * 3 + (100,) + (None,) * 3 + (o,)),
    "fuse_fill_literals": ("compact", lambda o: (None, None, 100, None, o)),
    "compute_column_length": ("colen", lambda o: (None, None, 100, None, None, None, o)),
    "stream_compaction": ("compact", lambda o: (None, None, 100, None, o)),
    "decode_device": ("decode", lambda o: (None, 100, 3100, None, o)),
    "encode_device": ("encode", lambda o: (None, 3100, None, 100, o)),
}


@pytest.mark.parametrize("ends", [True, False], ids=["fault", "unended"])
@pytest.mark.parametrize("name", WAITING)
def test_scan_state_is_cleared_after_a_fault(ctx, name, ends):
    """A launch that reports a fault, or whose last block never came because the
    state was not its own: an error, and a state the next launch can use."""
    kernel, args = WAITING[name]
    out = U64(77)
    ctx.script(kernel, fault=2, result=5, ends=ends)
    assert ctx.call(name, *args(ctypes.byref(out))) == EHIP
    state = next(x for x in ctx.log() if x.startswith(kernel)).split("state=")[1].split()[0]
    at = [i for i, x in enumerate(ctx.log()) if x.startswith(kernel)][-1]
    words = [int(x.split("words=")[1]) for x in ctx.log()[at:] if x.startswith(f"fill {state} ")]
    assert words and words[0] > 1000  # the counters and every status word
    ctx.script(kernel, result=42)
    assert ctx.call(name, *args(ctypes.byref(out))) == OK and out.value == 42


@pytest.mark.parametrize("slot", ["decode", "encode"])
@pytest.mark.parametrize("ends", [True, False], ids=["fault", "unended"])
def test_combine_reports_either_half(ctx, slot, ends):
    out = U64(0)
    args = (ctypes.c_int(0), None, 50, None, 0, 3100, None, 100, ctypes.byref(out))
    ctx.script(slot, fault=1, ends=ends)
    assert ctx.call("combine_device", *args) == EHIP
    ctx.script("encode", result=7)
    assert ctx.call("combine_device", *args) == OK and out.value == 7


def test_launches_of_nothing_wait_for_no_result(ctx):
    out = U64(77)
    assert ctx.call("stream_compaction", None, None, 0, None, ctypes.byref(out)) == OK
    assert out.value == 0
    assert ctx.call("decode_device", None, 0, 100, None, ctypes.byref(out)) == OK
    ctx.script("encode", result=3)
    assert ctx.call("combine_device", ctypes.c_int(1), None, 0, None, 0, 100, None, 9,
                    ctypes.byref(out)) == OK and out.value == 3


def query(ctx, keycnt=40, nrows=100_000, keys=None):
    return ctx.call("query_range_device", None, None, None, keycnt, None, ctypes.c_uint32(0),
                    ctypes.c_uint32(9), nrows, None, ctypes.byref(U64() if keys is None else keys))


def test_range_whose_offsets_descend_is_refused(ctx):
    """Its word count is negative: refused, never a launch over 2^64 words."""
    for words in (-1, -2048, -(2**32 - 1)):
        keys = U64()
        ctx.script("range", extra=(3, 2**64 + words))
        assert query(ctx, keys=keys) == EINVAL and keys.value == 3
    for _ in range(2):
        ctx.script("range", extra=(3, 2**33 - 2))
    assert query(ctx) == OK
    assert all(int(x.split("most=")[1].split()[0]) <= 2**33 for x in ctx.log() if "most=" in x)


@pytest.mark.parametrize("arena", [256, 4096, 8192, 1 << 20, (1 << 30) + 77, 1 << 36])
def test_range_on_a_fixed_arena_is_refused_before_it_decodes(lib, arena):
    """The device gets the most words that the arena allows (4 bytes each and 8
    per 2048 of them, in blocks of 256), so a longer range decodes nothing."""
    c = Ctx(lib, arena)
    cap = int(lib.wahgpu_arena_bytes(c.h))

    def needs(words):
        up = lambda x: (x + 255) // 256 * 256  # noqa: E731
        return up(2080 + (words + 2047) // 2048 * 8) + up(4 * words)
    for words in (1, 5):
        c.script("range", extra=(1, words))
    query(c)
    most = int(c.log()[-1].split("most=")[1].split()[0])
    held = 2**29  # what the status words hold; beyond it a range comes back
    assert most >= held or needs(most + 1) > cap
    assert most == 0 or needs(most) <= cap
    lib.fake_reset()
    longest = 2**33 if cap >= needs(2**33) else most
    for words, want in ((0, OK), (longest, OK),
                        (longest + 1, ENOMEM if longest < 2**33 else EINVAL)):
        keys = U64()
        for _ in range(1 + (held < words <= longest)):
            c.script("range", extra=(1, words))
        assert query(c, keys=keys) == want and keys.value == 1
    c.close()


def device_bytes(ctx):
    """Device memory in use beside the context's arena."""
    return ctx.lib.fake_device_bytes() - int(ctx.lib.wahgpu_arena_bytes(ctx.h))


def launched(ctx):
    """Table entries and `grow` of the range launches so far."""
    lines = [x for x in ctx.log() if x.startswith("range")]
    return [(int(x.split("table=")[1].split()[0]), int(x.split("grow=")[1])) for x in lines]


def test_range_table_is_bounded_by_what_ranges_need(ctx):
    """An index of many keys and rows: a query brings 8 MB whatever its range
    could need, and keeps more only for a range that decodes by it."""
    start = device_bytes(ctx)
    for extra in ((3, 100), (10**6, 5 * 10**7), (0, 0)):  # few words, few per key and slice, none
        ctx.script("range", extra=extra)
        assert query(ctx, keycnt=10**8, nrows=2**32) == OK
    assert launched(ctx) == [(2**20, 1)] * 3
    assert device_bytes(ctx) - start == 8 << 20


def test_range_comes_back_for_a_larger_table(ctx):
    nrows, keys = 2**24, 5000
    slices = 256  # one per CU up to 10240 chunks each
    words = 13 * keys * slices
    start = device_bytes(ctx)
    for _ in range(2):  # the launch that finds it too small, then the one that decodes
        ctx.script("range", extra=(keys, words))
    assert query(ctx, keycnt=2 * keys, nrows=nrows) == OK
    (first, grow), (second, again) = launched(ctx)
    assert (first, grow, again) == (2**20, 1, 0) and second >= 0.99 * keys * slices
    held = device_bytes(ctx) - start
    assert held == 8 * second < words  # 8 bytes for 13 words
    ctx.script("range", extra=(keys, words))  # the table is kept
    assert query(ctx, keycnt=2 * keys, nrows=nrows) == OK
    assert launched(ctx)[2:] == [(second, 1)]


def test_range_does_without_a_table_it_cannot_have(ctx):
    keys, words = U64(), 13 * 256 * 9000
    ctx.script("range", extra=(1, 1))
    assert query(ctx, keycnt=10**6, nrows=2**24) == OK  # the first one is there
    ctx.lib.fake_most_bytes(u64(9 << 20))
    for _ in range(2):
        ctx.script("range", extra=(9000, words))
    assert query(ctx, keycnt=10**6, nrows=2**24, keys=keys) == OK and keys.value == 9000
    assert launched(ctx)[1:] == [(2**20, 1), (0, 0)]


def test_a_context_holds_status_words_for_what_it_scans(lib):
    """1 MB for the scans of every column, 1 MB for its graphs'; more for a decode
    or a range of more than 2^29 words."""
    start = lib.fake_device_bytes()
    c = Ctx(lib)
    held = lib.fake_device_bytes() - start
    assert held <= (2 << 20) + (64 << 10)
    out = U64()

    def states():
        return {x.split("state=")[1].split()[0] for x in c.log() if "state=" in x}
    assert c.call("stream_compaction", None, None, 2**30 - 1, None, ctypes.byref(out)) == OK
    assert c.call("decode_device", None, 2**29, 2**32, None, ctypes.byref(out)) == OK
    assert c.call("encode_device", None, 2**32, None, 100, ctypes.byref(out)) == OK
    assert device_bytes(c) - start == held and len(states()) == 1
    assert c.call("decode_device", None, 2**29 + 1, 2**32, None, ctypes.byref(out)) == OK
    assert device_bytes(c) - start == held + 8
    assert any(x.startswith("fill") and int(x.split("=")[1]) > 2**18 for x in c.log())
    for words in (2**29 + 4097, 2**33 - 2):  # found, then decoded
        at = len(launched(c))
        for _ in range(2):
            c.script("range", extra=(2, words))
        assert query(c) == OK and len(launched(c)) == at + 2
        most = [int(x.split("most=")[1].split()[0]) for x in c.log() if x.startswith("range")]
        assert most[at] < words <= most[at + 1]
    assert c.call("decode_device", None, 2**32, 2**32, None, ctypes.byref(out)) == OK
    assert device_bytes(c) - start == held + 15 * 2**20  # 2^21 words in all
    c.close()
    assert lib.fake_device_bytes() == start


class Column(ctypes.Structure):
    _fields_ = [("offset", U64), ("n", U64), ("rid_base", ctypes.c_uint32),
                ("reserved", ctypes.c_uint32)]


def batch(ctx, lens):
    cols, at = (Column * len(lens))(), 0
    for c, n in zip(cols, lens):
        c.offset, c.n = at, n
        at += n
    return ctx.call("build_batch_device", None, at, cols, ctypes.c_uint32(len(lens)), None, None,
                    None, None, None)


def test_a_reservation_that_fits_a_fixed_arena_builds_in_it(lib):
    """What wahgpu_batch_reserve lays out is enough for batches of short and long
    columns; no build asks for more than the reservation did."""
    values, cols = 2**24, 65536
    c = Ctx(lib)
    assert c.call("batch_reserve", values, ctypes.c_uint32(cols)) == OK
    need = int(lib.wahgpu_arena_bytes(c.h))
    for lens in ([20000, 5], [5, 1000], [20000] * 3, [20000, 0] * 4):
        assert batch(c, lens) == OK
        assert int(lib.wahgpu_arena_bytes(c.h)) == need
    c.close()
    f = Ctx(lib, need)
    assert f.call("batch_reserve", values, ctypes.c_uint32(cols)) == OK
    for lens in ([20000, 5], [5, 1000], [20000] * 3, [20000, 0] * 4):
        assert batch(f, lens) == OK, f.error()
    assert f.log().count("graph") == 4
    f.close()


def test_short_columns_add_no_scratch_to_a_batch(lib):
    """A batch whose last columns are short, or empty, fits where it fits with
    long columns in their place."""
    sizes = []
    for last in (20000, 5, 0):
        c = Ctx(lib)
        assert batch(c, [20000] * 65536 + [last] * 200) == OK
        sizes.append(int(lib.wahgpu_arena_bytes(c.h)))
        launches = [x.split()[0] for x in c.log()]
        assert launches == (["small"] if last < 20000 else []) + ["sort", "tail"]
        c.close()
    assert sizes[1] <= sizes[0] and sizes[2] <= sizes[0]


def test_a_batch_of_short_columns_alone_is_one_launch(ctx):
    assert batch(ctx, [5, 0, 16384, 1000]) == OK
    assert ctx.log() == ["small cols=4"]


def test_timing_covers_batches_of_short_and_long_columns(ctx):
    """Each batch of one launch set is a timed call, short columns beside it or
    alone; the short ones' launch (100 ticks of the harness's clock) is ms[0]."""
    ms, calls = (ctypes.c_double * 7)(), ctypes.c_uint32(0)
    assert ctx.call("timing_begin", ctypes.c_uint32(8)) == OK
    for lens in ([20000] * 3, [5] * 200 + [40000], [20000, 0], [5, 1000]):
        assert batch(ctx, lens) == OK
    assert ctx.call("timing_end", ms, ctypes.byref(calls)) == OK
    assert calls.value == 4
    assert 300 <= ms[0] < 400 and all(0 < x < 50 for x in ms[1:])


def build_device(ctx, n):
    return ctx.call("build_device", None, n, ctypes.c_uint32(0), None, None, None, None, None)


@pytest.mark.parametrize("warm_up", ["build", "scan", "query"])
def test_any_call_warms_up_for_a_captured_build(ctx, warm_up):
    """A context's first call lays out 2 MB of arena, also one that needs none, so
    that a column of 50000 rows can be captured next; a captured short column
    needs no call before it and lays out nothing."""
    stream = VP(ctx.lib.wahgpu_stream(ctx.h))
    ctx.lib.fake_capture(stream, 1)
    assert build_device(ctx, 1000) == OK and ctx.lib.wahgpu_arena_bytes(ctx.h) == 0
    assert build_device(ctx, 50000) == EHIP  # the arena cannot grow in a capture
    ctx.lib.fake_capture(stream, 0)
    if warm_up == "build":
        assert build_device(ctx, 1000) == OK
    elif warm_up == "scan":
        assert ctx.call("exclusive_scan", None, 1000, None) == OK
    else:
        assert query(ctx) == OK
    ctx.lib.fake_capture(stream, 1)
    assert build_device(ctx, 50000) == OK
    ctx.lib.fake_capture(stream, 0)
