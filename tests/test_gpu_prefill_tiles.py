"""The batched prefill's expert GEMM tiles against the FP32 oracle, as
tests/test_gpu_prefill.py checks it: 128-row tiles in every block format with
full tiles and with remainders over and up to half a tile, 64-row tiles, and
prompts on both sides of each change of the tile size, in widths of an odd
number of 256-column super-blocks."""
import importlib
import os

import numpy as np
import pytest

from test_gpu_prefill import dev, run_and_check  # noqa: F401  (fixture)

engine = importlib.import_module("qwen-30brust_amd")
synth = importlib.import_module("qwen-30brust_amd.synth")

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("main", [synth.Q4_0, synth.Q8_0, synth.Q4_K, synth.Q5_K, synth.Q6_K])
def test_full_and_remainder_tiles(dev, main):
    """243 tokens, top 4 of 6 experts: 162 tokens per expert on average, so a
    full tile and a remainder around half a tile for most.  One layer: with so
    few experts a near-tie decided the other way by the fp16 operands moves a
    token enough to reach later tokens' routing in a second layer through the
    KV cache, which check_routing's bound (each token's own near-tie) excludes."""
    t = synth._k_types(attn=main, down=main, out=main, embd=main)
    spec = synth.Spec(768, 1, 8, 2, 128, 6, 4, 512, 512, 256, types=t, seed=main)
    img = synth.build_image(spec, threads=min(16, os.cpu_count() or 1))
    prompt = np.random.default_rng(main).integers(0, spec.vocab, 243).astype(np.uint32)
    m = engine.Model(img, spec.context, device=dev)
    assert m.prefill_batched
    run_and_check(m, spec, img, prompt, [7], f"kind {main}")


@pytest.mark.parametrize("n", [40, 41, 65, 97, 98])
@pytest.mark.parametrize("main", [synth.Q4_0, synth.Q8_0, synth.Q4_K, synth.Q5_K, synth.Q6_K])
def test_tile_rows_by_mean_tokens_per_expert(dev, main, n):
    """Top 4 of 6 experts: a mean of 26 (the last with 32-row tiles), 27, 43 and
    64 (64-row tiles, at 64 with a second tile for the experts above the mean)
    and 65 (128-row tiles)."""
    t = synth._k_types(attn=main, down=main, out=main, embd=main)
    spec = synth.Spec(768, 1, 8, 2, 128, 6, 4, 512, 512, 256, types=t, seed=100 + main)
    img = synth.build_image(spec, threads=min(16, os.cpu_count() or 1))
    prompt = np.random.default_rng(main + n).integers(0, spec.vocab, n).astype(np.uint32)
    m = engine.Model(img, spec.context, device=dev)
    assert m.prefill_batched
    run_and_check(m, spec, img, prompt, [7], f"kind {main}, {n} tokens")
