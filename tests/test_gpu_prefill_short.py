"""Batched prefill of short prompts against the FP32 oracle, as
tests/test_gpu_prefill.py checks it: the kernels for at most 32 and 64 rows
per tile in every block format, their column splits, and prompts around one
128-row tile (partial sums over fewer than eight row tiles)."""
import importlib
import os

import numpy as np
import pytest

from test_gpu_prefill import dev, model2, run_and_check  # noqa: F401  (fixtures)

engine = importlib.import_module("qwen-30brust_amd")
synth = importlib.import_module("qwen-30brust_amd.synth")

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [17, 50])
@pytest.mark.parametrize("main,out", [(synth.Q4_0, synth.Q4_0), (synth.Q8_0, synth.Q8_0), (synth.Q5_K, synth.Q5_K),
                                      (synth.Q6_K, synth.Q4_K)])
def test_short_prompt_formats(dev, main, out, n):
    t = synth._k_types(attn=main, down=main, out=out, embd=main)
    spec = synth.Spec(2048, 2, 32, 4, 128, 128, 8, 768, 512, 256, types=t, more_bits_type=synth.Q6_K, seed=n)
    img = synth.build_image(spec, threads=min(16, os.cpu_count() or 1))
    prompt = np.random.default_rng(n).integers(0, spec.vocab, n).astype(np.uint32)
    run_and_check(engine.Model(img, spec.context, device=dev), spec, img, prompt, [7], f"kind {main}, {n} tokens")


@pytest.mark.parametrize("n", [2, 127, 128, 129, 390])
def test_prompts_around_row_tiles(dev, model2, n):
    spec, img = model2
    prompt = np.random.default_rng(n).integers(0, spec.vocab, n).astype(np.uint32)
    run_and_check(engine.Model(img, spec.context, device=dev), spec, img, prompt, [7, 300], f"n={n}")


@pytest.mark.parametrize("hidden,heads,kvheads,ff", [(768, 20, 4, 256), (1280, 4, 2, 512)])
def test_short_prompt_odd_widths(dev, hidden, heads, kvheads, ff):
    """Widths of 3 and 5 super-blocks (no even column split) and short expert
    rows."""
    t = synth._k_types(attn=12, down=14, out=14, embd=12)
    spec = synth.Spec(hidden, 2, heads, kvheads, 128, 16, 4, ff, 512, 256, types=t, seed=hidden)
    img = synth.build_image(spec, threads=min(16, os.cpu_count() or 1))
    prompt = np.random.default_rng(hidden).integers(0, spec.vocab, 45).astype(np.uint32)
    m = engine.Model(img, spec.context, device=dev)
    assert m.prefill_batched
    run_and_check(m, spec, img, prompt, [7], f"hidden {hidden}")
