"""The persistent kernel's attention where a wavefront's run of cached positions grows past one batch
of 32 (256 positions), past what one workgroup takes (512), and into several shares: against the
launch-by-launch engine, with pages of one position, of a few, and larger than any context."""
import numpy as np
import pytest

import gradhip as G
from gradhip import synth
from helpers import assert_logits_close, lively_std

pytestmark = pytest.mark.gpu

MODELS = {
    "llama": synth.Config(synth.ARCH_MODERN, 300, 768, 2, 12, 1100),
    "gpt2-medium": synth.Config(synth.ARCH_GPT2, 300, 768, 1, 12, 1100),
    "gpt2-small": synth.Config(synth.ARCH_GPT2, 300, 512, 2, 8, 1100),
}


@pytest.mark.parametrize("page", [1, 8, 64, 1 << 17])
@pytest.mark.parametrize("name", sorted(MODELS))
def test_steps_at_the_edges_of_runs_batches_and_shares(name, page):
    cfg = MODELS[name]
    gm = G.Model.from_tensors(cfg, synth.make_weights(cfg, 31, std=lively_std(cfg), norm_noise=0.1))
    tokens = synth.uniform_tokens(1100, cfg.vocab, 32)
    fast = G.Session(gm, engine=G.ENGINE_PERSISTENT, page_tokens=page, shuffle_pages=True)
    plain = G.Session(gm, engine=G.ENGINE_EAGER)
    for at in (1, 31, 223, 253, 285, 509, 767, 1050):
        for s in (fast, plain):
            s.reset()
            s.prefill(tokens[None, :at])
        for t in range(at, at + 6):
            a, b = fast.step(tokens[t : t + 1]), plain.step(tokens[t : t + 1])
            # different orders of the same fp32 sums, as between any two engines
            assert_logits_close(np.asarray(a).reshape(-1), np.asarray(b).reshape(-1), 2e-5, f"{name} page {page} step {t}")
