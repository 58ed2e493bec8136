"""Copies between host and device: every path of vx_to_host / vx_to_host_many (through the pinned megabyte, through the ring
of pieces, straight to pinned memory) and staged uploads, byte for byte."""
import ctypes as C
import mmap
import os
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def be():
    from vexel_amd.backend import HipBackend
    b = HipBackend(0)
    yield b
    b.close()


KB, MB = 1 << 10, 1 << 20


# a word; both sides of the pinned part; both sides of a piece and of the ring of sixteen pieces; several turns of the ring
@pytest.mark.parametrize("size", [1, 4, 512 * KB, 512 * KB + 1, MB, 8 * MB - 3, 16 * MB, 16 * MB + 1, 41 * MB + 12345])
def test_download(be, size):
    src = np.random.default_rng(size).integers(0, 256, size, dtype=np.uint8)
    d = be.upload(src, permanent=True)
    for _ in range(2):
        out = np.zeros(size + 2, dtype=np.uint8)      # (at an odd address, with a byte in front and behind)
        be.to_host(out[1:-1], d)
        assert np.array_equal(out[1:-1], src) and out[0] == 0 and out[-1] == 0
    be.free(d)


@pytest.mark.parametrize("sizes", [[4, 0, 100, 64], [300 * KB, 300 * KB], [4, 33 * MB, 0, 5], [2 * MB + 7] * 16])
def test_download_of_several_ranges(be, sizes):
    rng = np.random.default_rng(len(sizes))
    src = [rng.integers(0, 256, max(1, s), dtype=np.uint8)[:s] for s in sizes]
    dev = [be.upload(s, permanent=True) for s in src]
    out = [np.zeros(s, dtype=np.uint8) for s in sizes]
    skip = np.full(9, 7, dtype=np.uint8)              # a range without a source stays as it is
    dst = (C.c_void_p * (len(sizes) + 1))(*([o.ctypes.data for o in out] + [skip.ctypes.data]))
    frm = (C.c_void_p * (len(sizes) + 1))(*(dev + [None]))
    num = (C.c_size_t * (len(sizes) + 1))(*(sizes + [9]))
    be.call("vx_to_host_many", len(sizes) + 1, dst, frm, num)
    assert all(np.array_equal(o, s) for o, s in zip(out, src)) and np.all(skip == 7)
    for p in dev:
        be.free(p)


def test_download_after_device_work_and_between_smaller_ones(be):
    """The bytes are those of everything enqueued before, in a row of calls of changing size over the same ring."""
    n = 6 * MB
    rng = np.random.default_rng(3)
    a, b = (rng.integers(0, 256, n, dtype=np.uint8) for _ in range(2))
    da, db, dc = be.upload(a, permanent=True), be.upload(b, permanent=True), be.alloc_permanent(n)
    for i in range(6):
        be.copy_buffer(db if i % 2 else da, 0, dc, 0, n)
        size = n if i % 3 else 1000
        out = np.empty(size, dtype=np.uint8)
        be.to_host(out, dc)
        assert np.array_equal(out, (b if i % 2 else a)[:size])
    for p in (da, db, dc):
        be.free(p)


# one byte; both sides of a slot; all eight slots; more ranges than slots and a range that begins inside an allocation (both ways);
# a total beyond the pinned part
@pytest.mark.parametrize("sizes", [[1], [64 * KB], [64 * KB + 1], [512 * KB], [4, 128000], [4, 0, 448 * KB], [100] * 8, [100] * 9, [300 * KB, 200 * KB], [4, 512 * KB]])
def test_small_download_by_marks(be, sizes):
    """What the caller waits for by marks: the bytes of the work enqueued last, call after call into the same slots, at odd addresses."""
    rng = np.random.default_rng(sum(sizes))
    n = sum(sizes) + 64
    a, b = (rng.integers(0, 256, n, dtype=np.uint8) for _ in range(2))
    da, db, dc = be.upload(a, permanent=True), be.upload(b, permanent=True), be.alloc_permanent(n)
    at = np.concatenate([[3], 3 + np.cumsum(sizes)[:-1]]).astype(int)
    for i in range(12):
        for k in range(11 + i % 2):                   # (the last copy is of b, of a, of b, ...)
            be.copy_buffer(db if k % 2 == 0 else da, 0, dc, 0, n)
        want = b if (10 + i % 2) % 2 == 0 else a
        out = [np.zeros(s + 2, dtype=np.uint8) for s in sizes]
        be.call("vx_to_host_many", len(sizes), (C.c_void_p * len(sizes))(*[o.ctypes.data + 1 for o in out]),
                (C.c_void_p * len(sizes))(*[int(dc + x) for x in at]), (C.c_size_t * len(sizes))(*sizes))
        for o, x, s in zip(out, at, sizes):
            assert np.array_equal(o[1:-1], want[x:x + s]) and o[0] == 0 and o[-1] == 0, (i, x)
    for p in (da, db, dc):
        be.free(p)


# both sides of where the runtime's copy takes over, from addresses of every alignment, with and without work ahead
@pytest.mark.parametrize("ahead", [0, 9])
@pytest.mark.parametrize("off", [0, 4, 1, 2, 3])
@pytest.mark.parametrize("size", [1, 3, 7, 4 * KB, 4 * KB + 1, 16 * KB, 16 * KB + 3, 64 * KB + 2, 512 * KB - 64])
def test_small_download_with_and_without_work_ahead(be, size, off, ahead):
    rng = np.random.default_rng(size + off)
    a, b = (rng.integers(0, 256, size + 16, dtype=np.uint8) for _ in range(2))
    da, db, dc = be.upload(a, permanent=True), be.upload(b, permanent=True), be.upload(a, permanent=True)
    out = np.zeros(size + 2, dtype=np.uint8)
    for turn in range(3):
        be.sync()
        for k in range(ahead):                        # (the last copy is of b)
            be.copy_buffer(da if k % 2 else db, 0, dc, 0, size + 16)
        be.call("vx_to_host", out.ctypes.data + 1, int(dc) + off, size)
        assert np.array_equal(out[1:-1], (b if ahead else a)[off:off + size]) and out[0] == 0 and out[-1] == 0
    for p in (da, db, dc):
        be.free(p)


def test_small_download_of_a_stream_at_rest_from_any_address(be):
    """64 KiB with nothing ahead take as long from an odd address as from an aligned one (byte by byte in a kernel it was 2.6 times as long)."""
    d = be.alloc_permanent(1 * MB)
    out, took = np.zeros(64 * KB, dtype=np.uint8), {0: [], 1: []}
    for off in [0, 1] * 40:
        be.sync()
        t = time.perf_counter()
        be.call("vx_to_host", out.ctypes.data, int(d) + off, out.size)
        took[off].append(time.perf_counter() - t)
    assert np.median(took[1]) < 1.5 * np.median(took[0]), {k: np.median(v) * 1e6 for k, v in took.items()}
    be.free(d)


def test_staged_uploads(be):
    """Each upload's bytes are taken when the call returns, also once the staging memory has been used up several times."""
    rows, size = 1500, 1000
    d = be.alloc_permanent(rows * 1024)
    buf = np.zeros(size, dtype=np.uint8)
    for i in range(rows):
        buf[:] = (i * 7 + np.arange(size)) % 251
        be.call("vx_to_device_staged", d + i * 1024, buf.ctypes.data, size)
    got = be.download(d, (rows, 1024), np.uint8)[:, :size]
    assert np.array_equal(got, (np.arange(rows)[:, None] * 7 + np.arange(size)[None, :]) % 251)
    big = np.random.default_rng(1).integers(0, 256, 64 * KB + 1, dtype=np.uint8)
    be.call("vx_to_device_staged", d, big.ctypes.data, big.size)
    assert np.array_equal(be.download(d, (big.size,), np.uint8), big)
    be.free(d)


# sources at addresses that 16-byte, 4-byte and single-byte loads serve; both sides of a piece of 64 KB
@pytest.mark.parametrize("at", [16, 4, 1])
@pytest.mark.parametrize("size", [576 * KB - 1, 576 * KB, 576 * KB + 17])
def test_download_from_any_address(be, at, size):
    src = np.random.default_rng(size + at).integers(0, 256, size + 32, dtype=np.uint8)
    d = be.upload(src, permanent=True)
    out = np.zeros(size + 1, dtype=np.uint8)
    be.to_host(out[:-1], d + at)
    assert np.array_equal(out[:-1], src[at:at + size]) and out[-1] == 0
    be.free(d)


# more ranges than a launch holds; sizes at the edges of 4 and 16 bytes, none and more than the staging takes; any alignment; more
# than the staging memory in all
@pytest.mark.parametrize("sizes", [[4, 0, 4], [4] * 3, [1, 3, 4, 15, 16, 17, 64, 1000] * 20, [64 * KB, 64 * KB + 1, 12, 64 * KB - 3] * 4, [40 * KB] * 30])
@pytest.mark.parametrize("shift", [0, 4, 1])
def test_staged_uploads_of_several_ranges(be, sizes, shift):
    rng = np.random.default_rng(len(sizes) + shift)
    src = [rng.integers(0, 256, max(1, s), dtype=np.uint8)[:s] for s in sizes]
    at = np.cumsum([0] + [(s + 31) // 16 * 16 for s in sizes])
    total = int(at[-1]) + 32
    want = rng.integers(0, 256, total, dtype=np.uint8)
    d = be.upload(want, permanent=True)
    n = len(sizes)
    for _ in range(2):
        dst = (C.c_void_p * (n + 1))(*([d + int(a) + shift for a in at[:-1]] + [None]))
        frm = (C.c_void_p * (n + 1))(*([s.ctypes.data for s in src] + [want.ctypes.data]))
        num = (C.c_size_t * (n + 1))(*(sizes + [9]))
        be.call("vx_to_device_staged_many", n + 1, dst, frm, num)
        for s, a in zip(src, at):
            want[a + shift:a + shift + s.size] = s
            s[:] = 255 - s                                 # the bytes are taken when the call returns
        assert np.array_equal(be.download(d, (total,), np.uint8), want)
    be.free(d)


# both sides of the smallest announced size; fresh memory, memory in use, a destination left out
@pytest.mark.parametrize("size", [2 * MB - 64, 2 * MB + 5, 9 * MB])
def test_expected_download(be, size):
    src = np.random.default_rng(size).integers(0, 256, size, dtype=np.uint8)
    d = be.upload(src, permanent=True)
    for used in (False, True):
        pages = mmap.mmap(-1, size, flags=mmap.MAP_PRIVATE | mmap.MAP_ANONYMOUS)     # (ordinary memory of which no page is there)
        out = np.frombuffer(pages, dtype=np.uint8)
        if used:
            out[:] = 1
        token = C.c_int(-1)
        dst, num = (C.c_void_p * 2)(out.ctypes.data, None), (C.c_size_t * 2)(size, 7)
        be.call("vx_to_host_expect", 2, dst, num, C.byref(token))
        assert (token.value != 0) == (not used and size >= 2 * MB and len(os.sched_getaffinity(0)) > 1)
        be.to_host(out, d)
        be.lib_call("vx_to_host_forget", be._h, token.value)
        assert np.array_equal(out, src)
    be.free(d)
