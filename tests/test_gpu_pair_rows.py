"""Passes over many rows whose operands are two fp16 parts each (models of 512 columns and more): every tiling and
epilogue at row counts that leave ragged tiles, operands at the ends of their range, and models whose weights have
no such form, against the float64 forward.  The bounds are what fp32 sums give, as for the three-part form."""
import numpy as np
import pytest

import gradhip as G
import ref_forward
from gradhip import synth
from helpers import lively_std

pytestmark = pytest.mark.gpu


def _loss(ref, targets):
    top = ref.max(axis=1)
    return np.log(np.exp(ref - top[:, None]).sum(axis=1)) + top - ref[np.arange(len(targets)), targets]


def _check(cfg, W, B, n, seed, sequences=None):
    tokens = synth.uniform_tokens(B * (n + 1), cfg.vocab, seed).reshape(B, n + 1)
    gm = G.Model.from_tensors(cfg, W)
    nll = G.Session(gm, batch=B).score(tokens[:, :-1], tokens[:, 1:])
    last = G.Session(gm, batch=B).prefill(tokens[:, :-1])
    for b in sequences or sorted({0, B - 1}):
        with np.errstate(over="ignore"):
            ref = ref_forward.forward(cfg, W, tokens[b, :-1])
        want = _loss(ref, tokens[b, 1:])
        assert np.abs(nll[b] - want).max() <= 2e-5 * max(1.0, np.abs(want).max()), b
        assert np.abs(last[b] - ref[-1]).max() <= 1e-5 * np.abs(ref[-1]).max(), b


CASES = {
    # rows reach: name: (width, vocab, sequences, tokens)
    "32 x 32 tiles, one row past a tile": (512, 130, 1, 161),
    "64 x 64 of two sets of K": (512, 1001, 3, 171),
    "64 x 64 of one set, q, k, v; 64 x 96 of four, keys and values from the middle of the matrix": (512, 130, 3, 449),
    "128 x 64, both FFN1; a nearly empty tile": (512, 130, 3, 667),
    "128 x 128 at 512 columns": (512, 515, 11, 487),
    "64 x 96 of four sets, SwiGLU": (768, 130, 2, 150),
    "64 x 64 of one set, FFN1; four sets of 64 x 96, q, k, v": (768, 515, 1, 449),
    "64 x 64 of two sets, W_o": (768, 1001, 3, 334),
    "64 x 96 of four sets, W_o, FFN2 and logits": (768, 515, 4, 501),
    "64 x 96 of two sets, FFN2; 128 x 128 and quarters, GELU, keys and values": (768, 515, 6, 500),
    "128 x 128, all": (768, 515, 19, 474),
    "nine parts of K: one set": (576, 130, 1, 161),
    "nine parts of K: one set, FFN2 in four": (576, 301, 3, 667),
    "64 x 96 of two sets, q, k, v and GELU": (640, 130, 2, 260),
    "64 x 96 of two sets, SwiGLU": (768, 130, 2, 260),
    "128 x 64, q, k, v": (512, 130, 9, 377),
    "128 x 64, W_o": (576, 130, 17, 390),
    "128 x 128 and quarters, q, k, v": (768, 130, 5, 400),
    "128 x 128 and quarters, SwiGLU": (768, 130, 2, 520),
    "128 x 128 and quarters, W_o; a nearly empty row of tiles": (512, 130, 20, 410),
    "128 x 128 and quarters, q, k, v; quarters past the last row and the last output": (576, 130, 6, 405),
}


@pytest.mark.parametrize("arch", [synth.ARCH_GPT2, synth.ARCH_MODERN])
@pytest.mark.parametrize("name", sorted(CASES))
def test_rows_match_the_float64_forward(name, arch):
    d, vocab, B, n = CASES[name]
    cfg = synth.Config(arch, vocab, d, 1, d // 64, 700)
    _check(cfg, synth.make_weights(cfg, 101, std=lively_std(cfg), norm_noise=0.1), B, n, 102)


@pytest.mark.parametrize("arch", [synth.ARCH_GPT2, synth.ARCH_MODERN])
def test_rows_of_one_large_element_reach_the_bound_of_the_norm(arch):
    """norm(x) of a row with one element that outweighs the rest is sqrt(d) there: the largest an operand can be."""
    cfg = synth.Config(arch, 67, 512, 2, 8, 600)
    W = synth.make_weights(cfg, 103, std=lively_std(cfg), norm_noise=0.1)
    W[0][np.arange(67), np.arange(67) * 7] += 1e4
    _check(cfg, W, 1, 530, 104)


def test_operands_far_below_their_bound():
    """Gains of 1/50 to 50 in one norm: what most operands hold lies 2^-10 and more below the bound."""
    cfg = synth.Config(synth.ARCH_GPT2, 67, 512, 2, 8, 600)
    W = synth.make_weights(cfg, 105, std=lively_std(cfg), norm_noise=0.1)
    names = [what[0] for what in synth.tensor_specs(cfg)]
    for layer in range(2):
        W[names.index(f"layer {layer} norm2 gamma")][0, :] = np.geomspace(0.02, 3.0, 512)
        W[names.index(f"layer {layer} norm2 gamma")][0, 5] = 50.0
    _check(cfg, W, 1, 530, 106)


@pytest.mark.parametrize("gain", [1e6, 1e30])
def test_a_gain_too_far_above_the_others_for_two_parts(gain):
    """One gain so large that bounds say nothing about the rest (the weights behind it are zero): three parts."""
    cfg = synth.Config(synth.ARCH_MODERN, 67, 512, 1, 8, 600)
    W = synth.make_weights(cfg, 107, std=lively_std(cfg), norm_noise=0.1)
    names = [what[0] for what in synth.tensor_specs(cfg)]
    W[names.index("layer 0 norm2 gamma")][0, 5] = gain
    W[names.index("layer 0 FFN gate")][5, :] = 0.0
    W[names.index("layer 0 FFN up")][5, :] = 0.0
    _check(cfg, W, 1, 530, 108)


def test_weights_at_both_ends_of_the_range():
    """A row of weights below fp32's normal numbers, one of zeros, one of 1e12 (what comes of it is not used, but bounds
    have to count with it), and a weight 2^20 times the rest of its row."""
    cfg = synth.Config(synth.ARCH_GPT2, 67, 512, 1, 8, 600)
    W = synth.make_weights(cfg, 109, std=lively_std(cfg), norm_noise=0.1)
    names = [what[0] for what in synth.tensor_specs(cfg)]
    up, down = names.index("layer 0 FFN W1"), names.index("layer 0 FFN W2")
    W[up][:, 3] = 1e-40
    W[up][:, 4] = 0.0
    W[up][:, 6] = 1e12
    W[down][6, :] = 0.0
    W[up][9, 7] *= 2.0 ** 20
    W[down][7, :] *= 2.0 ** -20
    _check(cfg, W, 1, 530, 110)


def test_infinite_and_nan_weights_keep_their_meaning():
    cfg = synth.Config(synth.ARCH_GPT2, 301, 512, 1, 8, 200)
    W = synth.make_weights(cfg, 111, std=lively_std(cfg), norm_noise=0.1)
    W[0][300, 5] = -np.inf
    W[-1][0, 5] = 30.0  # beta of the final norm: that logit is -inf at every position
    tokens = synth.uniform_tokens(172, 300, 112)
    want = _loss(ref_forward.forward(cfg, W, tokens[:-1]), tokens[1:])
    nll = G.Session(G.Model.from_tensors(cfg, W)).score(tokens[:-1], tokens[1:])[0]
    assert np.abs(nll - want).max() <= 2e-5 * max(1.0, np.abs(want).max())
    W[0][300, 5] = np.nan
    assert np.isnan(G.Session(G.Model.from_tensors(cfg, W)).score(tokens[:-1], tokens[1:])).all()


def test_a_prompt_in_front_of_draws_from_the_whole_row():
    """Greedy picks, and draws that come to the same, are the same behind generate's prompt and behind prefill's."""
    cfg = synth.Config(synth.ARCH_MODERN, 130, 512, 2, 8, 640)
    gm = G.Model.from_tensors(cfg, synth.make_weights(cfg, 113, std=lively_std(cfg), norm_noise=0.1))
    prompt = synth.uniform_tokens(600, cfg.vocab, 114)
    for opt in (G.sampling(1e-3, 0, 1.0, 1.0), G.sampling(1.0, 0, 1.0, 1.0, True)):  # temperature 1e-3: the arg-max
        picks, s = [], G.Session(gm)
        s.prefill(prompt)
        s.decode_stream(12, opt, lambda ids, index: picks.append(ids[0]), seed=5)
        tokens = G.Session(gm).generate(prompt, 12, opt, seed=5)
        assert np.array_equal(np.asarray(tokens)[0, 600:], picks)


@pytest.mark.parametrize("arch", [synth.ARCH_GPT2, synth.ARCH_MODERN])
def test_queries_so_small_that_their_unit_leaves_fp32(arch):
    """A token whose norm(x) is zero leaves a query of the bias alone, 1e-35; behind keys of 1e-4 the unit of its scores was
    2^-150 and its masked scores not numbers.  (GPT-2: position and token cancel.)"""
    cfg = synth.Config(arch, 67, 512, 2, 8, 600)
    W = synth.make_weights(cfg, 115, std=lively_std(cfg), norm_noise=0.1)
    names = [what[0] for what in synth.tensor_specs(cfg)]
    W[0][:4] = 0.0
    if arch == synth.ARCH_GPT2:
        W[1][:] = 0.0
        W[names.index("layer 0 norm1 beta")][:] = 0.0
    for layer in range(2):
        W[names.index(f"layer {layer} b_q")][:] = 1e-35
        W[names.index(f"layer {layer} W_k")] *= np.float32(1e-6)
        W[names.index(f"layer {layer} b_k")] *= np.float32(1e-6)
    _check(cfg, W, 1, 530, 116)


@pytest.mark.parametrize("bias", [1e6, 1e20, 1e30])
def test_a_query_too_far_above_the_others_for_two_parts(bias):
    """An element of every query so large that one power of two cannot serve the rest of its row (its keys are zero)."""
    cfg = synth.Config(synth.ARCH_GPT2, 67, 512, 2, 8, 600)
    W = synth.make_weights(cfg, 117, std=lively_std(cfg), norm_noise=0.1)
    names = [what[0] for what in synth.tensor_specs(cfg)]
    W[names.index("layer 1 b_q")][0, 70] = bias
    W[names.index("layer 1 W_k")][:, 70] = 0.0
    W[names.index("layer 1 b_k")][0, 70] = 0.0
    _check(cfg, W, 1, 530, 118)


@pytest.mark.parametrize("opt", [(0.8, 0, 1.0, 1.2), (1.0, 0, 0.95, 1.1), (0.8, 40, 0.9, 1.1), (0.9, 2000, 1.0, 1.0), (1.0, 0, 1.0, 1.0, True)])
@pytest.mark.parametrize("batch, n", [(1, 600), (5, 130)])
def test_a_prompt_leaves_the_same_bits_whatever_the_call_and_the_sampler(opt, batch, n):
    """generate, and prefill with the same reply streamed or decoded behind it: the same cache and tokens."""
    cfg = synth.Config(synth.ARCH_MODERN, 5000, 512, 2, 8, 640)
    gm = G.Model.from_tensors(cfg, synth.make_weights(cfg, 119, std=lively_std(cfg), norm_noise=0.1))
    prompt = synth.uniform_tokens(batch * n, cfg.vocab, 120).reshape(batch, n)

    def cache(s):
        return [s.read_kv(b, layer, kv, pos).tobytes() for b in (0, batch - 1) for layer in (0, 1) for kv in (0, 1)
                for pos in (0, 77, n - 1)]

    s = G.Session(gm, batch=batch)
    s.prefill(prompt)
    kept = cache(s)
    picks = np.asarray(s.decode(16, G.sampling(*opt), seed=9))
    streamed, s = [], G.Session(gm, batch=batch)
    s.prefill(prompt)
    s.decode_stream(16, G.sampling(*opt), lambda ids, index: streamed.append(np.array(ids)), seed=9)
    assert np.array_equal(np.stack(streamed, axis=1), picks)
    s = G.Session(gm, batch=batch)
    tokens = np.asarray(s.generate(prompt, 16, G.sampling(*opt), seed=9))
    assert cache(s) == kept
    assert np.array_equal(tokens[:, n:], picks)


#: (arch, width, tokens): what a pass leaves of the second layer's values is no further from float64 than with three parts
CLOSENESS = [(synth.ARCH_GPT2, 512, 160), (synth.ARCH_GPT2, 512, 512), (synth.ARCH_GPT2, 512, 641), (synth.ARCH_GPT2, 512, 1000),
             (synth.ARCH_MODERN, 512, 400), (synth.ARCH_MODERN, 512, 640), (synth.ARCH_MODERN, 512, 641), (synth.ARCH_GPT2, 576, 400),
             (synth.ARCH_GPT2, 640, 384), (synth.ARCH_GPT2, 640, 385), (synth.ARCH_GPT2, 768, 320), (synth.ARCH_GPT2, 768, 321),
             (synth.ARCH_GPT2, 768, 1000), (synth.ARCH_MODERN, 768, 160), (synth.ARCH_MODERN, 768, 256), (synth.ARCH_MODERN, 768, 300),
             (synth.ARCH_MODERN, 896, 160), (synth.ARCH_GPT2, 1024, 160)]


@pytest.mark.parametrize("arch, d, n", CLOSENESS)
def test_errors_are_no_larger_than_those_of_three_parts(arch, d, n):
    """The same layers with one gain, in front of weights of zero, that leaves them no pairs."""
    cfg = synth.Config(arch, 1009, d, 2, d // 64, 1001)
    names = [what[0] for what in synth.tensor_specs(cfg)]
    errors = [[], []]
    for seed in (121, 123):
        W = synth.make_weights(cfg, seed, std=0.02, norm_noise=0.1)
        for name in ("FFN W1",) if arch == synth.ARCH_GPT2 else ("FFN gate", "FFN up"):
            W[names.index(f"layer 0 {name}")][5, :] = 0.0
        tokens = synth.uniform_tokens(n + 1, cfg.vocab, seed + 1)
        _, kv = ref_forward.forward(cfg, W, tokens[:-1], return_kv=True)
        at = range(0, n, 8)  # (values: keys carry the rounding of their angles too)
        want = np.stack([kv[1][1][pos] for pos in at])
        for form, gain in enumerate((1.0, 1e9)):
            W[names.index("layer 0 norm2 gamma")][0, 5] = gain
            s = G.Session(G.Model.from_tensors(cfg, W))
            s.score(tokens[:-1], tokens[1:])
            got = np.stack([s.read_kv(0, 1, 1, pos) for pos in at])
            errors[form].append(np.linalg.norm(got - want) / np.linalg.norm(want))
    pairs, parts = np.mean(errors, axis=1)
    assert pairs <= 1.01 * parts, (pairs, parts)  # (40000 values and more: the figures' own spread is 0.5 %)
