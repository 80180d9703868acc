"""What a failed call of the C ABI leaves behind in the caller's buffers."""
import ctypes as C
import importlib

import numpy as np
import pytest

import oracle

engine = importlib.import_module("qwen-30brust_amd")
synth = importlib.import_module("qwen-30brust_amd.synth")

pytestmark = pytest.mark.gpu


def failing_model(spec):
    """A model whose logits are not finite: infinite output norm weights."""
    img = synth.build_image(spec)
    oracle.Gguf(img).data("output_norm.weight").view(np.float32)[:] = np.inf  # a view of img
    return engine.Model(img, spec.context, device=engine.Device(0))


@pytest.mark.parametrize("spec", [synth.tiny_k(), synth.Spec(512, 2, 4, 2, 128, 8, 2, 256, 256, 64,
                                                             types=synth._k_types(), seed=3)])
def test_failed_generate_and_prefill_leave_the_outputs(spec):
    """qh_generate and qh_prefill (exact token step; batched, then run again
    exactly) fail on logits that are not finite and write no token and no
    logit; the context works on."""
    m = failing_model(spec)
    assert m.prefill_batched == (spec.head_dim == 128)
    prompt = np.array([3, 5, 7], np.uint32)
    ids, logits, am = np.full(4, 77, np.uint32), np.full(spec.vocab, 2.5, np.float32), C.c_uint32(99)
    h, lib = m.dev.h, engine.lib()
    for _ in range(2):
        for call in (lambda: lib.qh_generate(h, prompt.ctypes.data, 3, 1, ids.ctypes.data, logits.ctypes.data, logits.size),
                     lambda: lib.qh_prefill(h, prompt.ctypes.data, 3, logits.ctypes.data, logits.size, C.byref(am))):
            assert call() != 0
            assert lib.qh_last_error(h) == b"nonfinite model output"
            assert m.position == 0
            assert (ids == 77).all() and (logits == 2.5).all() and am.value == 99
    assert m.prefill_reruns == (2 if spec.head_dim == 128 else 0)


def test_null_buffers_are_refused():
    """A null pointer where host data is read or written is an error of the
    call, and the context works on."""
    spec = synth.tiny_k()
    m = engine.Model(synth.build_image(spec), spec.context, device=engine.Device(0))
    h, lib, N = m.dev.h, engine.lib(), spec.hidden
    x, y = np.ones(4 * N, np.float32), np.zeros(4 * N, np.float32)
    ids, out, prompt = np.zeros(8, np.uint32), C.c_uint32(), np.array([3], np.uint32)
    w = synth.normal(1, 32 * 8).astype(np.float32)  # 8 rows of 32 F32 weights
    sampler = engine.Sampler(1, 0.5, 4, 0.9)
    p = lambda a: a.ctypes.data  # noqa: E731
    name = b"blk.0.attn_k.weight"
    want = m.dev.attention(x[:64], y[:64], x[:64], 2, 1, 32)
    for call in (lambda: lib.qh_matvec(h, name, -1, None, N, p(y), 4 * N),
                 lambda: lib.qh_matvec(h, name, -1, p(x), N, None, 4 * N),
                 lambda: lib.qh_packed_matvec(h, p(w), w.nbytes, 0, 8, 32, None, p(y)),
                 lambda: lib.qh_packed_matvec(h, p(w), w.nbytes, 0, 8, 32, p(x), None),
                 lambda: lib.qh_dequant(h, p(w), w.nbytes, 0, 8, 32, None),
                 lambda: lib.qh_route(h, None, 8, 2, p(ids), p(y)),
                 lambda: lib.qh_route(h, p(x), 8, 2, None, p(y)),
                 lambda: lib.qh_route(h, p(x), 8, 2, p(ids), None),
                 lambda: lib.qh_argmax(h, None, 8, C.byref(out)),
                 lambda: lib.qh_attention(h, None, p(x), p(x), 64, 2, 1, 32, p(y)),
                 lambda: lib.qh_attention(h, p(x), None, p(x), 64, 2, 1, 32, p(y)),
                 lambda: lib.qh_attention(h, p(x), p(x), None, 64, 2, 1, 32, p(y)),
                 lambda: lib.qh_attention(h, p(x), p(x), p(x), 64, 2, 1, 32, None),
                 lambda: lib.qh_sample_logits(h, sampler.h, None, None, 8, C.byref(out)),
                 lambda: lib.qh_layer_forward(h, 0, None, 0, None, None, None, None),
                 lambda: lib.qh_generate(h, p(prompt), 1, 1, None, None, 0)):
        assert call() != 0
        assert lib.qh_last_error(h) in (b"null input buffer", b"null output buffer")
        assert np.array_equal(m.dev.attention(x[:64], y[:64], x[:64], 2, 1, 32), want)
    m.reset()
    first = m.forward(3)
    m.reset()
    assert np.array_equal(m.forward(3), first)
