"""gp_stage_upload_async and gp_fetch: bytes arrive whole at the sizes where the copies change form (a vector of 16
bytes, one workgroup or several, one piece of the ring or many, the copy engine), whatever ran before."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 4096, 16384, 16385, 100003, (256 << 10) + 1, (1 << 20) + 3, (5 << 20) + 7, (9 << 20) + 5])
def test_upload_and_fetch_round_trip(gp, n):
    rng = np.random.default_rng(n)
    st, stream, other = C.c_void_p(), gp.Stream(), gp.Stream()
    gp.check(gp.lib().gp_stage_create(C.byref(st)))
    devs = [gp.DevBuf(n + 16) for _ in range(3)]
    for r in range(8):
        want = [rng.integers(0, 256, n, np.uint8) for _ in devs]
        for d, w in zip(devs, want):
            host = w.copy()
            gp.check(gp.lib().gp_stage_upload_async(st, C.c_void_p(d.ptr), host.ctypes.data_as(C.c_void_p), C.c_size_t(n), (stream if r % 2 else other).h))
            host[:] = 0  # the caller's buffer is free again
        for d, w in zip(devs, want):
            out, pinned = gp.host_pool.empty(n)
            assert pinned
            gp.check(gp.lib().gp_fetch(C.c_void_p(pinned), C.c_void_p(d.ptr), C.c_size_t(n), (stream if r % 2 else other).h))
            assert np.array_equal(d.download()[:n], w), (n, r)
            assert np.array_equal(out, w), (n, r)
    gp.check(gp.lib().gp_stage_destroy(st))


def test_pool_memory_comes_back_and_is_bounded(gp):
    pool = gp.HostPool()
    a, pa = pool.empty(1000)
    view = a[10:20]
    del a
    b, pb = pool.empty(1000)
    assert pb != pa  # still referred to
    del view
    c, pc = pool.empty(900)
    assert pc == pa
    pool.LIMIT = 1 << 20
    d, pd = pool.empty(2 << 20)
    assert pd is None and d.nbytes == 2 << 20


def test_sizes_mixed_on_one_handle(gp):
    """the count of arrivals goes on from copy to copy, whatever number of workgroups each of them has"""
    rng = np.random.default_rng(5)
    st, stream = C.c_void_p(), gp.Stream()
    gp.check(gp.lib().gp_stage_create(C.byref(st)))
    dev = gp.DevBuf(3 << 20)
    for r in range(40):
        n = int(rng.choice([1, 5000, 40000, 70001, 300000, 1 << 20, 3 << 20]))
        want = rng.integers(0, 256, n, np.uint8)
        gp.check(gp.lib().gp_stage_upload_async(st, C.c_void_p(dev.ptr), want.ctypes.data_as(C.c_void_p), C.c_size_t(n), stream.h))
        out, pinned = gp.host_pool.empty(n)
        gp.check(gp.lib().gp_fetch(C.c_void_p(pinned), C.c_void_p(dev.ptr), C.c_size_t(n), stream.h))
        assert np.array_equal(out, want), (n, r)
    gp.check(gp.lib().gp_stage_destroy(st))


@pytest.mark.parametrize("stop", [None, -1, 0, 37, 0x7FFFFFFF])
def test_stop_index_is_reported_with_its_number(gp, stop):
    host, dev = C.c_void_p(), C.c_void_p()
    gp.check(gp.lib().gp_host_alloc_coherent(C.byref(host), C.byref(dev), C.c_size_t(8)))
    word = C.cast(host, C.POINTER(C.c_ulonglong))
    index = None if stop is None else gp.DevBuf.from_array(np.array([stop], np.int32))
    stream = gp.Stream()
    for seq in (1, 0xFFFFFFFF):
        gp.check(gp.lib().gp_report_stop_async(C.c_void_p(index.ptr) if index else None, dev, C.c_uint(seq), stream.h))
        stream.sync()
        assert word[0] & 0xFFFFFFFF == seq
        assert word[0] >> 32 == (-1 if stop is None else stop) & 0xFFFFFFFF
    gp.check(gp.lib().gp_host_free(host))
    with pytest.raises(gp.GpError):
        gp.check(gp.lib().gp_report_stop_async(None, None, C.c_uint(1), stream.h))


class ClosedGate:
    """A gate kernel at the head of a stream: what is submitted behind it waits until open() (about a second at most)."""

    def __init__(self, gp, stream):
        self.gp, self.flag, self.gave_up = gp, gp.Flag(), gp.DevBuf(4)
        self.gave_up.fill32(0)
        gp.check(gp.lib().gp_launch_gate(C.c_void_p(self.flag.dev), C.c_ulonglong(1 << 22), C.c_void_p(self.gave_up.ptr), stream.h))

    def open(self):
        self.flag.set(1)

    def was_open_early(self):
        return bool(self.gave_up.download(np_dtype=np.int32)[0])


def test_pinned_input_is_read_in_place_and_without_a_wait(gp):
    """set_input_pinned: one transfer in stream order; the call returns while the stream is held up"""
    from gpreempt_amd import executor as gx
    rows, cols = 1024, 4096  # 16 MB
    ex = gx.Executor("toy@rows=%d,cols=%d,n=1,dtype=f32" % (rows, cols))
    n = rows * cols * 4
    host, dev = C.c_void_p(), C.c_void_p()
    gp.check(gp.lib().gp_host_alloc_coherent(C.byref(host), C.byref(dev), C.c_size_t(n)))
    x = np.frombuffer((C.c_char * n).from_address(host.value), np.float32)
    x[:] = np.random.default_rng(1).standard_normal(x.size, np.float32)
    stream = gp.Stream()
    gate = ClosedGate(gp, stream)
    assert gx.lib().gpx_set_input_pinned(ex.h, b"data", host, C.c_size_t(n), stream.h) == 0
    assert not stream.idle()
    gate.open()
    stream.sync()
    assert not gate.was_open_early()
    assert np.array_equal(ex.read_storage("data").view(np.float32), x)
    assert gx.lib().gpx_set_input_pinned(ex.h, b"data", host, C.c_size_t(n - 1), stream.h) == 4  # OutOfRange, as set_input
    assert gx.lib().gpx_set_input_pinned(ex.h, b"nothing", host, C.c_size_t(n), stream.h) == 3   # NotFound
    gp.check(gp.lib().gp_host_free(host))


def test_ordinary_input_does_not_wait_for_a_stream_that_is_held_up(gp):
    """uploads of more than eight pieces, and on a second stream, behind a closed gate: each returns, the second stream's
    arrives, and the first one's when the gate opens"""
    rng = np.random.default_rng(8)
    st, held, free = C.c_void_p(), gp.Stream(), gp.Stream()
    gp.check(gp.lib().gp_stage_create(C.byref(st)))
    sizes = [20 << 20, 3, 5 << 20, 70000, 1 << 20]
    want = [rng.integers(0, 256, n, np.uint8) for n in sizes]
    devs = [[gp.DevBuf(n) for n in sizes] for _ in range(2)]
    gate = ClosedGate(gp, held)

    def upload(d, w, stream):
        host = w.copy()
        gp.check(gp.lib().gp_stage_upload_async(st, C.c_void_p(d.ptr), host.ctypes.data_as(C.c_void_p), C.c_size_t(w.size), stream.h))
        host[:] = 0
    for d, w in zip(devs[0], want):
        upload(d, w, held)
    assert not held.idle()
    for d, w in zip(devs[1], want):
        upload(d, w, free)
    free.sync()
    assert not held.idle()
    gate.open()
    held.sync()
    assert not gate.was_open_early()
    for side in devs:
        for d, w in zip(side, want):
            assert np.array_equal(d.download(), w)
    # more than the ring may hold: the pieces come round again
    big = rng.integers(0, 256, (150 << 20) + 17, np.uint8)
    d = gp.DevBuf(big.size)
    upload(d, big, free)
    free.sync()
    assert np.array_equal(d.download(), big)
    gp.check(gp.lib().gp_stage_destroy(st))
