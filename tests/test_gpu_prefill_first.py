"""The first batched prefill of a freshly loaded model, which builds its
buffers, gives the bits of every later one."""
import importlib
import os

import numpy as np
import pytest

engine = importlib.import_module("qwen-30brust_amd")
synth = importlib.import_module("qwen-30brust_amd.synth")

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [20, 243])
@pytest.mark.parametrize("ff", [512, 768])
def test_first_prefill_equals_the_second(ff, n):
    t = synth._k_types(attn=8, down=8, out=8, embd=8)
    spec = synth.Spec(768, 2, 8, 2, 128, 6, 4, ff, 512, 256, types=t, seed=ff)
    img = synth.build_image(spec, threads=min(16, os.cpu_count() or 1))
    prompt = np.random.default_rng(n).integers(0, spec.vocab, n).astype(np.uint32)
    m = engine.Model(img, spec.context, device=engine.Device(0))
    first = m.prefill(prompt)[1].copy()
    m.reset()
    np.testing.assert_array_equal(first, m.prefill(prompt)[1])
