"""Split passes whose products are two rounds of 64 x 64 tiles over the compute units and so, in three parts, one
round of 128 x 64: every epilogue at row counts that leave both a whole and a nearly empty tile,
against the float64 forward.  In pairs, which these rows of ordinary weights are, and in three parts, which gains too far
apart for pairs are left with (which launches that makes: test_tilings.py)."""
import numpy as np
import pytest

import gradhip as G
import ref_forward
from gradhip import synth
from helpers import lively_std

pytestmark = pytest.mark.gpu

CASES = {
    # rows                        256 rows and one more; FFN1: 320 tiles (Llama), 240 (GPT-2)
    "ffn1-257": (1, 257),
    # the last tile full, FFN1 of both blocks (384 and 288 tiles) and q, k, v after 449 rows only
    "ffn1-384": (2, 192),
    # q, k, v at 396 tiles
    "qkv-641": (1, 641),
    # W_o and FFN2 at the fewest tiles and rows of several sequences in one tile
    "resid-1347": (3, 449),
    "resid-2688": (4, 672),
    "resid-2689": (1, 2689),  # one row more: three rounds, so 128 x 128
}


@pytest.mark.parametrize("arch", [synth.ARCH_GPT2, synth.ARCH_MODERN])
@pytest.mark.parametrize("name", sorted(CASES))
def test_rows_match_the_float64_forward(name, arch):
    B, n = CASES[name]
    cfg = synth.Config(arch, 130, 768, 1, 12, 2700)
    W = synth.make_weights(cfg, 91, std=lively_std(cfg), norm_noise=0.1)
    tokens = synth.uniform_tokens(B * (n + 1), cfg.vocab, 92).reshape(B, n + 1)
    nll = G.Session(G.Model.from_tensors(cfg, W), batch=B).score(tokens[:, :-1], tokens[:, 1:])
    for b in sorted({0, B - 1}):
        ref = ref_forward.forward(cfg, W, tokens[b, :-1])
        top = ref.max(axis=1)
        want = np.log(np.exp(ref - top[:, None]).sum(axis=1)) + top - ref[np.arange(n), tokens[b, 1:]]
        # what fp32 sums give, as for the other tilings
        assert np.abs(nll[b] - want).max() <= 2e-5 * max(1.0, np.abs(want).max()), (name, b)


VOCAB = 1001  # (of the cases below; logits of 1347 rows in 128 x 64 tiles too)


@pytest.mark.parametrize("arch", [synth.ARCH_GPT2, synth.ARCH_MODERN])
@pytest.mark.parametrize("name", sorted(CASES))
def test_rows_of_three_parts_match_the_float64_forward(name, arch):
    """A gain of 1e9 in front of weights of zero, in a layer's second norm and in the last one: neither has pairs."""
    B, n = CASES[name]
    cfg = synth.Config(arch, VOCAB, 768, 1, 12, 2700)
    W = synth.make_weights(cfg, 97, std=lively_std(cfg), norm_noise=0.1)
    names = [what[0] for what in synth.tensor_specs(cfg)]
    W[names.index("layer 0 norm2 gamma")][0, 5] = W[names.index("final norm gamma")][0, 5] = 1e9
    for what in ("FFN gate", "FFN up") if cfg.modern else ("FFN W1",):
        W[names.index(f"layer 0 {what}")][5, :] = 0.0
    W[0][:, 5] = 0.0
    tokens = synth.uniform_tokens(B * (n + 1), cfg.vocab, 98).reshape(B, n + 1)
    nll = G.Session(G.Model.from_tensors(cfg, W), batch=B).score(tokens[:, :-1], tokens[:, 1:])
    for b in sorted({0, B - 1}):
        ref = ref_forward.forward(cfg, W, tokens[b, :-1])
        top = ref.max(axis=1)
        want = np.log(np.exp(ref - top[:, None]).sum(axis=1)) + top - ref[np.arange(n), tokens[b, 1:]]
        assert np.abs(nll[b] - want).max() <= 2e-5 * max(1.0, np.abs(want).max()), (name, b)
