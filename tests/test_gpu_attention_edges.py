"""Attention whose values hold infinities where a kernel's tile ends: the
register-tiled kernels read the last key again past the end of a chunk, with
probability 0, and 0 times infinity must not reach the sum."""
import ctypes as C

import numpy as np
import pytest

from test_zz_no_alloc import DeviceBuffer, dev, engine, exact, inputs, noalloc  # noqa: F401  (fixture)
from test_zz_no_alloc_streams import Streams, capture, hip, hip_check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,heads,kvheads,d", [(1, 4, 4, 128), (1000, 32, 4, 128), (65, 6, 2, 64), (95, 8, 1, 64),
                                               (5000, 8, 1, 128), (70, 4, 2, 96)])
def test_infinite_value_of_a_last_key(dev, T, heads, kvheads, d):
    """+inf and -inf in elements of the last keys of 32- and 64-key tiles and of
    the whole history: those outputs are infinite, all others as float64, from
    the entry points' kernels, the general one (q, k, v off 16 bytes) and a
    captured call."""
    q, k, v = inputs(T + d, T, heads, kvheads, d)
    vv = v.reshape(T, kvheads, d)
    vv[T - 1, :, 3], vv[T - 1, :, d - 1] = np.inf, -np.inf
    for at in (31, 63):
        if at < T:
            vv[at, :, 5] = np.inf
    ref = exact(q, k, v, T, heads, kvheads, d)
    fin = np.isfinite(ref)
    assert fin.any() and not fin[:, 3].any()
    got = [noalloc(dev, q, k, v, heads, kvheads, d), dev.attention(q, k, v, heads, kvheads, d)]
    bufs = [DeviceBuffer(np.concatenate([np.zeros(1, np.float32), a])) for a in (q, k, v)]
    out = DeviceBuffer(np.zeros(heads * d, np.float32))
    assert engine.lib().qh_attention_noalloc(dev.h, *[b.ptr.value + 4 for b in bufs], k.size, heads, kvheads, d,
                                             out.ptr, None) == 0
    got.append(out.read())
    plain = [DeviceBuffer(a) for a in (q, k, v)]
    with Streams(1) as (s,):
        exe, = capture(dev, *plain, out, k.size, (heads, kvheads, d), s, 1)
        hip_check(hip().hipGraphLaunch(exe, s))
        hip_check(hip().hipStreamSynchronize(s))
        got.append(out.read())
        hip_check(hip().hipGraphExecDestroy(exe))
    for g in got:
        g = g.reshape(heads, d)
        assert np.array_equal(g[~fin], ref[~fin].astype(np.float32))
        assert np.max(np.abs(g[fin] - ref[fin])) <= 1e-5 * np.max(np.abs(ref[fin]))
    for b in bufs + plain + [out]:
        b.free()
