"""Passes over many rows (prompts and scoring) on the split bf16 products: every tiling the rows
can take, at row counts that leave ragged tiles, against the float64 forward.  The bound is
what fp32 sums give, an order below the engine's common 1e-4."""
import ctypes
import time

import numpy as np
import pytest

import gradhip as G
import ref_forward
from gradhip import synth
from helpers import lively_std

pytestmark = pytest.mark.gpu

CASES = {
    # name: (config, batch, tokens per sequence)
    "one-block-per-set": (synth.Config(synth.ARCH_MODERN, 37, 64, 2, 1, 200), 1, 161),       # K = 64, 32 x 32 tiles
    "32-gpt2": (synth.Config(synth.ARCH_GPT2, 301, 128, 2, 2, 200), 1, 193),
    "64-k4-modern": (synth.Config(synth.ARCH_MODERN, 1000, 256, 2, 4, 192), 4, 159),         # hidden width 704: 11 blocks per set
    "64-gpt2": (synth.Config(synth.ARCH_GPT2, 1001, 256, 1, 4, 200), 12, 150),               # one set over all of K
    "128-modern": (synth.Config(synth.ARCH_MODERN, 530, 192, 1, 3, 1100), 24, 1057),         # 24 k rows
    "shared-keys": (synth.Config(synth.ARCH_MODERN, 130, 128, 1, 2, 1400), 1, 1301),        # key runs of 128, merged
    "128-gpt2": (synth.Config(synth.ARCH_GPT2, 515, 128, 1, 2, 2100), 17, 2049),             # two slices of rows
}


def test_a_continued_pass_sees_the_cache_of_the_passes_before():
    """600 tokens behind 333 cached ones: key tiles that begin before the pass, pages of 16."""
    cfg = synth.Config(synth.ARCH_MODERN, 130, 128, 2, 2, 1000)
    W = synth.make_weights(cfg, 73, std=lively_std(cfg), norm_noise=0.1)
    gm = G.Model.from_tensors(cfg, W)
    tokens = synth.uniform_tokens(2 * 933, cfg.vocab, 74).reshape(2, 933)
    s = G.Session(gm, batch=2, page_tokens=16, shuffle_pages=True)
    s.prefill(tokens[:, :333])
    last = s.prefill(tokens[:, 333:])
    for b in range(2):
        ref = ref_forward.forward(cfg, W, tokens[b])
        assert np.abs(last[b] - ref[-1]).max() <= 1e-5 * np.abs(ref[-1]).max(), b


@pytest.mark.parametrize("n", [127, 128, 129])
def test_either_attention_behind_a_cache(n):
    """Up to 128 new tokens take the fp32 attention, more the split one: both sides behind 333."""
    cfg = synth.Config(synth.ARCH_GPT2, 130, 128, 2, 2, 500)
    W = synth.make_weights(cfg, 75, std=lively_std(cfg), norm_noise=0.1)
    tokens = synth.uniform_tokens(2 * 334 + 2 * n, cfg.vocab, 76).reshape(2, 334 + n)
    s = G.Session(G.Model.from_tensors(cfg, W), batch=2)
    s.prefill(tokens[:, :333])
    nll = s.score(tokens[:, 333:-1], tokens[:, 334:])
    for b in range(2):
        want = _loss(ref_forward.forward(cfg, W, tokens[b, :-1])[333:], tokens[b, 334:])
        assert np.abs(nll[b] - want).max() <= 2e-5 * max(1.0, np.abs(want).max()), b


@pytest.mark.parametrize("name", sorted(CASES))
def test_rows_match_the_float64_forward(name):
    cfg, B, n = CASES[name]
    W = synth.make_weights(cfg, 71, std=lively_std(cfg), norm_noise=0.1)
    gm = G.Model.from_tensors(cfg, W)
    tokens = synth.uniform_tokens(B * (n + 1), cfg.vocab, 72).reshape(B, n + 1)
    nll = G.Session(gm, batch=B).score(tokens[:, :-1], tokens[:, 1:])
    last = G.Session(gm, batch=B).prefill(tokens[:, :-1])
    for b in sorted({0, B - 1}):
        ref = ref_forward.forward(cfg, W, tokens[b, :-1])
        top = ref.max(axis=1)
        want = np.log(np.exp(ref - top[:, None]).sum(axis=1)) + top - ref[np.arange(n), tokens[b, 1:]]
        assert np.abs(nll[b] - want).max() <= 2e-5 * max(1.0, np.abs(want).max()), (name, b)
        assert np.abs(last[b] - ref[-1]).max() <= 1e-5 * np.abs(ref[-1]).max(), (name, b)


@pytest.mark.parametrize("n", [60, 171])
def test_a_logit_that_is_not_a_number_reaches_the_loss(n):
    """One NaN in a row of the embedding that no input uses: every loss is NaN, as it is token by token."""
    cfg = synth.Config(synth.ARCH_MODERN, 301, 128, 1, 2, 200)
    W = synth.make_weights(cfg, 81, std=lively_std(cfg), norm_noise=0.1)
    W[0][300, 5] = np.nan
    tokens = synth.uniform_tokens(2 * (n + 1), 300, 82).reshape(2, n + 1)
    gm = G.Model.from_tensors(cfg, W)
    for flags in (0, G.FLAG_STEPWISE_PROMPT):
        nll = G.Session(gm, batch=2, flags=flags).score(tokens[:, :-1], tokens[:, 1:])
        assert np.isnan(nll).all(), (flags, nll)


def _free_bytes():
    # by soname: the HIP runtime the process already has
    hip = ctypes.CDLL("libamdhip64.so.7")
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipDeviceSynchronize() == 0
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_a_short_scoring_pass_does_not_copy_the_layers():
    """Below 160 rows the layers run on the fp32 weights: only the logits matrix is split."""
    cfg = synth.Config(synth.ARCH_GPT2, 301, 1024, 4, 16, 200)
    rng = np.random.default_rng(87)
    W = [rng.standard_normal((r, c), dtype=np.float32) * np.float32(0.02) for _, r, c, _ in synth.tensor_specs(cfg)]
    layers = 4 * 4 * 12 * 1024 * 1024  # bytes of their split form, two fp16 parts per weight
    gm = G.Model.from_tensors(cfg, W)
    tokens = synth.uniform_tokens(172, cfg.vocab, 88)
    s = G.Session(gm)
    s.score(tokens[:20], tokens[1:21])
    before = _free_bytes()
    gm2 = G.Model.from_tensors(cfg, W)
    model = before - _free_bytes()
    s2 = G.Session(gm2)
    s2.score(tokens[:20], tokens[1:21])
    assert before - model - _free_bytes() < layers // 4
    s2.score(tokens[:151], tokens[1:152])
    assert before - model - _free_bytes() < layers // 4
    s2.reset()
    s2.score(tokens[:171], tokens[1:172])
    assert before - model - _free_bytes() >= layers  # from 160 rows on they are, in that form alone
    assert before - model - _free_bytes() < layers * 3 // 2


def _loss(ref, targets):
    top = ref.max(axis=1)
    return np.log(np.exp(ref - top[:, None]).sum(axis=1)) + top - ref[np.arange(len(targets)), targets]


@pytest.mark.parametrize("n", [60, 171])
def test_an_infinitely_unlikely_token_adds_nothing_to_the_loss(n):
    """A logit of -inf: an infinite weight against an activation that is positive at every position."""
    cfg = synth.Config(synth.ARCH_GPT2, 301, 128, 1, 2, 200)
    W = synth.make_weights(cfg, 83, std=lively_std(cfg), norm_noise=0.1)
    W[0][300, 5] = -np.inf
    W[-1][0, 5] = 30.0  # beta of the final norm
    tokens = synth.uniform_tokens(2 * (n + 1), 300, 84).reshape(2, n + 1)
    ref = ref_forward.forward(cfg, W, tokens[1, :-1])
    assert (ref[:, 300] == -np.inf).all()
    want = _loss(ref, tokens[1, 1:])
    nll = G.Session(G.Model.from_tensors(cfg, W), batch=2).score(tokens[:, :-1], tokens[:, 1:])
    assert np.abs(nll[1] - want).max() <= 2e-5 * max(1.0, np.abs(want).max())


def test_weights_beyond_the_range_of_the_split():
    """A weight that rounds to an infinite bf16: the gate of a hidden unit whose output is not used."""
    cfg = synth.Config(synth.ARCH_MODERN, 301, 128, 1, 2, 640)
    W = synth.make_weights(cfg, 85, std=lively_std(cfg), norm_noise=0.1)
    names = [what[0] for what in synth.tensor_specs(cfg)]
    W[names.index("layer 0 FFN gate")][5, 0] = 3.4e38
    W[names.index("layer 0 norm2 gamma")][0, 5] = 1e-3
    W[names.index("layer 0 FFN down")][0, :] = 0.0
    tokens = synth.uniform_tokens(601, cfg.vocab, 86)
    with np.errstate(over="ignore"):
        ref = ref_forward.forward(cfg, W, tokens[:-1])
    gm = G.Model.from_tensors(cfg, W)
    last = G.Session(gm).prefill(tokens[:-1])[0]
    assert np.abs(last - ref[-1]).max() <= 1e-5 * np.abs(ref[-1]).max()
    nll = G.Session(gm).score(tokens[:-1], tokens[1:])[0]
    want = _loss(ref, tokens[1:])
    assert np.abs(nll - want).max() <= 2e-5 * max(1.0, np.abs(want).max())


@pytest.mark.parametrize("spare", [7 << 18, 3 << 20, 11 << 20])
def test_passes_that_find_little_memory_left(spare, monkeypatch):
    """8 x 1000 rows with no allocation above 1.75 MiB (nothing is split, slices of 504 rows), 3 MiB (the
    logits matrix is) and 11 MiB (the layers are; slices of 2000 rows, the last with the fp32 attention).
    (No rotation: at position 1000 its fp32 angles are 2e-5 of eight layers' logits.)"""
    cfg = synth.Config(synth.ARCH_GPT2, 3000, 128, 8, 2, 1001)
    W = synth.make_weights(cfg, 89, std=lively_std(cfg), norm_noise=0.1)
    tokens = synth.uniform_tokens(8 * 1001, cfg.vocab, 90).reshape(8, 1001)
    ref = ref_forward.forward(cfg, W, tokens[7, :-1])
    monkeypatch.setenv("GRADHIP_TEST_SPARE_BYTES", str(spare))
    gm = G.Model.from_tensors(cfg, W)
    last = G.Session(gm, batch=8).prefill(tokens[:, :-1])
    assert np.abs(last[7] - ref[-1]).max() <= 1e-5 * np.abs(ref[-1]).max()
    nll = G.Session(gm, batch=8).score(tokens[:, :-1], tokens[:, 1:])
    want = _loss(ref, tokens[7, 1:])
    assert np.abs(nll[7] - want).max() <= 2e-5 * max(1.0, np.abs(want).max())
    monkeypatch.delenv("GRADHIP_TEST_SPARE_BYTES")
    assert np.abs(G.Session(gm, batch=8).score(tokens[:, :-1], tokens[:, 1:]) - nll).max() <= 2e-5 * np.abs(want).max()


def test_attention_scratch_stays_bounded():
    """64 sequences of 4500 tokens, whose split keys and values would be 670 MB: they go in groups of
    (sequence, head) pairs, some of which begin in the middle of a sequence's heads.  MiB: 231 of
    activations (a slice of 32768 rows x 7296 bytes and 512 rows of the fp32 tiles' buffers), 256 of
    keys and values, at most 1300 partial results (43, in steps of 8)."""
    cfg = synth.Config(synth.ARCH_GPT2, 130, 192, 1, 3, 4500)
    W = synth.make_weights(cfg, 91, std=lively_std(cfg), norm_noise=0.1)
    tokens = synth.uniform_tokens(64 * 4500, cfg.vocab, 92).reshape(64, 4500)
    gm = G.Model.from_tensors(cfg, W)
    G.Session(gm, batch=1).prefill(tokens[:1, :600])  # the weights' split form
    s = G.Session(gm, batch=64)
    before = _free_bytes()
    last = s.prefill(tokens)
    assert before - _free_bytes() <= (231 + 256 + 48) << 20
    for b in (0, 25, 63):
        ref = ref_forward.forward(cfg, W, tokens[b])
        assert np.abs(last[b] - ref[-1]).max() <= 1e-5 * np.abs(ref[-1]).max(), b


@pytest.mark.parametrize("arch", [synth.ARCH_GPT2, synth.ARCH_MODERN])
@pytest.mark.parametrize("d", [1088, 4160])
def test_wide_models_take_the_pass_too(arch, d):
    """Rows of more than 1024 columns, and of more than the 4096 that a wavefront's registers hold."""
    cfg = synth.Config(arch, 67, d, 1, d // 64, 180)
    rng = np.random.default_rng(93)
    W = [rng.standard_normal((r, c), dtype=np.float32) * np.float32(lively_std(cfg) if what in ("matrix", "bias") else 0.1)
         + np.float32(what == "gamma") for _, r, c, what in synth.tensor_specs(cfg)]
    tokens = synth.uniform_tokens(3 * 172, cfg.vocab, 94).reshape(3, 172)
    gm = G.Model.from_tensors(cfg, W)
    nll = G.Session(gm, batch=3).score(tokens[:, :-1], tokens[:, 1:])
    s, stepwise = G.Session(gm, batch=3), G.Session(gm, batch=3, flags=G.FLAG_STEPWISE_PROMPT)
    last = s.prefill(tokens[:, :-1])
    ref = ref_forward.forward(cfg, W, tokens[2, :-1])
    want = _loss(ref, tokens[2, 1:])
    assert np.abs(nll[2] - want).max() <= 2e-5 * max(1.0, np.abs(want).max())
    assert np.abs(last[2] - ref[-1]).max() <= 1e-5 * np.abs(ref[-1]).max()

    def seconds(session):
        session.reset()
        begin = time.perf_counter()
        session.prefill(tokens[:, :-1])
        return time.perf_counter() - begin

    stepwise.prefill(tokens[:, :-1])
    # 171 steps read every weight 171 times; the pass measured 84 to 105 times as fast
    assert min(seconds(s) for _ in range(3)) < 0.25 * min(seconds(stepwise) for _ in range(3))


def test_weights_without_pairs_hold_the_three_parts_alone():
    """A layer whose second norm's gains lie too far apart for two fp16 parts: what was begun of them is given back."""
    cfg = synth.Config(synth.ARCH_GPT2, 301, 1024, 4, 16, 200)
    rng = np.random.default_rng(95)
    W = [rng.standard_normal((r, c), dtype=np.float32) * np.float32(0.02) for _, r, c, _ in synth.tensor_specs(cfg)]
    names = [what[0] for what in synth.tensor_specs(cfg)]
    W[names.index("layer 3 norm2 gamma")][0, 5] = 1e9
    layers = 6 * 4 * 12 * 1024 * 1024  # bytes of the three parts
    tokens = synth.uniform_tokens(172, cfg.vocab, 96)
    gm = G.Model.from_tensors(cfg, W)
    s = G.Session(gm)
    s.score(tokens[:20], tokens[1:21])
    before = _free_bytes()
    s.reset()
    s.score(tokens[:171], tokens[1:172])
    assert layers <= before - _free_bytes() < layers * 5 // 4
