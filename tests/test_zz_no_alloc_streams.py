"""qh_attention_noalloc where calls meet: captured graphs replayed on other
streams beside eager calls, more streams than scratch areas, host threads that
share a stream, and the per-thread stream handle.  Histories of 20,000 keys
queued without waits, so that calls overlap on the device."""
import ctypes as C
import importlib
import threading

import numpy as np
import pytest

from test_zz_no_alloc import DeviceBuffer, dev, exact, hip, hip_check, inputs, noalloc  # noqa: F401  (fixture)

engine = importlib.import_module("qwen-30brust_amd")

pytestmark = pytest.mark.gpu
T, SHAPE = 20000, (32, 4, 128)
OUT = SHAPE[0] * SHAPE[2]
PER_THREAD = 2  # hipStreamPerThread


class Streams:
    """n HIP streams, destroyed at the end."""

    def __init__(self, n):
        self.s = [C.c_void_p() for _ in range(n)]
        for s in self.s:
            hip_check(hip().hipStreamCreate(C.byref(s)))

    def __enter__(self):
        return self.s

    def __exit__(self, *_):
        for s in self.s:
            hip_check(hip().hipStreamSynchronize(s))
            hip_check(hip().hipStreamDestroy(s))


def call(dev, q, k, v, out, klen, shape, stream, at=0):
    rc = engine.lib().qh_attention_noalloc(dev.h, q.ptr, k.ptr, v.ptr, klen, *shape, out.ptr.value + 4 * at, stream)
    assert rc == 0, engine.lib().qh_last_error(dev.h).decode()


@pytest.fixture(scope="module")
def long(dev):
    """(k, v on the device, nine queries, their outputs of calls on their own)."""
    _, k, v = inputs(5, T, *SHAPE)
    qs = [inputs(100 + i, 1, *SHAPE)[0] for i in range(9)]
    want = [noalloc(dev, q, k, v, *SHAPE) for q in qs]
    bufs = [DeviceBuffer(a) for a in (k, v, *qs)]
    yield bufs[0], bufs[1], bufs[2:], want
    for b in bufs:
        b.free()


def capture(dev, q, k, v, out, klen, shape, stream, execs):
    """`execs` executable graphs of one captured call."""
    graph, got = C.c_void_p(), [C.c_void_p() for _ in range(execs)]
    hip_check(hip().hipStreamBeginCapture(stream, 2))  # relaxed
    try:
        call(dev, q, k, v, out, klen, shape, stream)
    finally:
        hip_check(hip().hipStreamEndCapture(stream, C.byref(graph)))
    for g in got:
        hip_check(hip().hipGraphInstantiate(C.byref(g), graph, None, None, C.c_size_t(0)))
    hip_check(hip().hipGraphDestroy(graph))
    return got


@pytest.mark.parametrize("keys,heads,kvheads,d,off", [
    (1, 4, 4, 128, 0), (65, 32, 4, 128, 0), (4097, 14, 2, 64, 0), (7001, 10, 2, 128, 0), (257, 18, 2, 128, 0), (700, 32, 4, 128, 1),
    (129, 6, 3, 64, 1), (300, 4, 2, 96, 0), (33, 5, 1, 32, 0), (513, 4, 2, 256, 0), (90, 3, 1, 320, 0), (70, 1, 1, 4094, 0), (7, 2, 2, 1, 0)])
def test_captured_call(dev, keys, heads, kvheads, d, off):
    """A captured call's replays against float64, as test_attention_shapes, and
    with the eager call's bits where the register-tiled kernels apply; `off`
    floats off 16-byte alignment."""
    q, k, v = inputs(keys + heads, keys, heads, kvheads, d)
    ref = exact(q, k, v, keys, heads, kvheads, d)
    bufs = [DeviceBuffer(np.concatenate([np.zeros(off, np.float32), a])) for a in (q, k, v)]
    shifted = [type("P", (), {"ptr": C.c_void_p(b.ptr.value + 4 * off)}) for b in bufs]
    out = DeviceBuffer(np.full(heads * d, np.nan, np.float32))
    with Streams(1) as (s,):
        exe, = capture(dev, *shifted, out, k.size, (heads, kvheads, d), s, 1)
        for _ in range(3):
            hip_check(hip().hipGraphLaunch(exe, s))
            hip_check(hip().hipStreamSynchronize(s))
            got = out.read()
            if d in (64, 128) and heads <= 8 * kvheads and not off:
                assert np.array_equal(got, dev.attention(q, k, v, heads, kvheads, d))
            assert np.max(np.abs(got.reshape(heads, d) - ref)) <= 1e-5 * np.max(np.abs(ref))
            hip_check(hip().hipMemcpy(out.ptr, np.zeros_like(got).ctypes.data, got.nbytes, 1))
        hip_check(hip().hipGraphExecDestroy(exe))
    for b in bufs + [out]:
        b.free()


def test_graphs_beside_calls(dev, long):
    """One captured call, replayed on two other streams while the stream that
    captured it runs eager calls."""
    k, v, qs, want = long
    outs = [DeviceBuffer(np.zeros(OUT, np.float32)) for _ in range(3)]
    with Streams(3) as s:
        one, = capture(dev, qs[0], k, v, outs[0], T * 512, SHAPE, s[0], 1)
        two, = capture(dev, qs[1], k, v, outs[1], T * 512, SHAPE, s[0], 1)
        for _ in range(4):
            for _ in range(10):
                hip_check(hip().hipGraphLaunch(one, s[1]))
                call(dev, qs[2], k, v, outs[2], T * 512, SHAPE, s[0])
                hip_check(hip().hipGraphLaunch(two, s[2]))
            for t in s:
                hip_check(hip().hipStreamSynchronize(t))
            for o, w in zip(outs, want):
                assert np.array_equal(o.read(), w)
        for g in (one, two):
            hip_check(hip().hipGraphExecDestroy(g))
    for o in outs:
        o.free()


def test_more_streams_than_areas(dev, long):
    """Nine streams at once, twice: the second nine find areas that earlier
    streams left."""
    k, v, qs, want = long
    for _ in range(2):
        outs = [DeviceBuffer(np.zeros(20 * OUT, np.float32)) for _ in qs]
        with Streams(9) as s:
            for i in range(20):
                for q, o, t in zip(qs, outs, s):
                    call(dev, q, k, v, o, T * 512, SHAPE, t, i * OUT)
        for o, w in zip(outs, want):
            assert np.array_equal(o.read().reshape(20, OUT), np.tile(w, (20, 1)))
            o.free()


@pytest.mark.parametrize("handle", ["one stream", "per-thread handle"])
def test_host_threads(dev, long, handle):
    """Two host threads, each with its own context, calling on one stream, or
    each on its own through hipStreamPerThread."""
    k, v, qs, want = long
    n = 200
    outs = [DeviceBuffer(np.zeros(n * OUT, np.float32)) for _ in range(2)]
    devs = [engine.Device(0) for _ in range(2)]
    failed = []

    def work(i, stream):
        try:
            for j in range(n):
                call(devs[i], qs[i], k, v, outs[i], T * 512, SHAPE, stream, j * OUT)
            hip_check(hip().hipStreamSynchronize(stream))
        except BaseException as e:
            failed.append(e)

    with Streams(1) as (s,):
        stream = s if handle == "one stream" else C.c_void_p(PER_THREAD)
        threads = [threading.Thread(target=work, args=(i, stream)) for i in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    assert not failed, failed
    for o, w in zip(outs, want):
        assert np.array_equal(o.read().reshape(n, OUT), np.tile(w, (n, 1)))
        o.free()
    for d in devs:
        d.close()
