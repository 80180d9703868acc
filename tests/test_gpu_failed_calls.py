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
