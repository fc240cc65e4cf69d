"""Draws without a top-k cut, where the row's split over threads and the top-p cut can go
wrong: vocabularies at the edges of what a thread holds in registers (16 and 32 elements
of 1024 or 512 threads), cuts at the very first and the very last value, flat rows whose cut
lies in a crowded bin, and rows so peaked that it lies far below the maximum."""
import numpy as np
import pytest

import gradhip as G
import oracle_lib as O
from gradhip import synth
from helpers import check_sampled_stream, lively_std

pytestmark = pytest.mark.gpu

CASES = {
    **{f"v{v}": synth.Config(synth.ARCH_MODERN, v, 64, 1, 2, 40) for v in (3, 65, 16384, 16385, 32769, 65536, 65537)},
    **{f"persistent-v{v}": synth.Config(synth.ARCH_GPT2, v, 512, 1, 8, 40) for v in (8192, 8193, 16385)},
}
SAMPLERS = [(1.0, 0.0), (1.0, 0.3), (50.0, 0.95), (0.9, 0.99999), (0.02, 0.9), (1.0, 1.0)]


@pytest.mark.parametrize("name", sorted(CASES))
def test_plain_and_top_p_streams(name):
    cfg = CASES[name]
    W = synth.make_weights(cfg, 92, std=lively_std(cfg), norm_noise=0.1)
    om, gm = O.Model.from_tensors(cfg, W), G.Model.from_tensors(cfg, W)
    prompt = synth.uniform_tokens(4, cfg.vocab, 23)
    n = 10
    s = G.Session(gm)
    for i, (T, p) in enumerate(SAMPLERS):
        u = synth.uniforms(n, 4200 + i)
        ref, rsl = O.generate_sample(om, prompt, u, T, n, 1.1, 0, p, want_logits=True)
        s.reset()
        got = s.generate(prompt, n, G.sampling(T, 0, p, 1.1), uniforms=u)
        check_sampled_stream(got[0], ref, rsl, len(prompt), u, (T, 0, p, 1.1), f"{name} T={T} top_p={p}")


def _draws_between_two_sums(V, threads):
    """Draws on a flat row of V that fall between the two ways the sampler forms the sum up to the
    end of a thread's run: element by element from where the run starts, and from the totals of
    the runs.  Every step is an fp32 addition that is restated here."""
    f = np.float32
    run, p = ((V + threads - 1) // threads) | 1, f(1) / f(V)
    length = [min(V, (t + 1) * run) - min(V, t * run) for t in range(threads)]
    total = np.zeros(run + 1, f)
    for i in range(run):
        total[i + 1] = total[i] + p
    starts, base = [], f(0)
    for w in range(0, threads, 64):
        acc = f(0)
        for t in range(w, w + 64):
            starts.append(base + acc)
            acc = acc + total[length[t]]
        base = base + acc
    starts.append(base)
    draws = []
    for t in range(threads):
        walked = starts[t]
        for _ in range(length[t]):
            walked = walked + p
        if length[t] and walked < starts[t + 1]:
            draws.append(starts[t + 1])
    return np.array(draws, f)


@pytest.mark.parametrize("vocab,persistent", [(5000, False), (16000, False), (32000, False), (40001, False),
                                              (7001, True), (16000, True)])
def test_a_draw_between_two_roundings_of_a_running_sum(vocab, persistent):
    """The walk's answer is the element at the draw, whichever of the two sums reaches it: both
    are within the roundings of 1024 + 64 additions, far less than an element of a flat row."""
    cfg = synth.Config(synth.ARCH_GPT2, vocab, 512, 1, 8, 64) if persistent \
        else synth.Config(synth.ARCH_MODERN, vocab, 64, 1, 1, 8)
    W = synth.make_weights(cfg, 5)
    W[0][:] = 0.0  # every logit is 0
    u = _draws_between_two_sums(vocab, 512 if persistent else 1024)
    u = u[np.linspace(0, len(u) - 1, 40).astype(int)]
    want = np.ceil(u.astype(np.float64) * vocab) - 1
    opt = G.sampling(1.0, 0, 1.0, 1.0)
    if persistent:
        s = G.Session(G.Model.from_tensors(cfg, W))
        got = s.generate([1, 2, 3], len(u), opt, uniforms=u)[0, 3:]
    else:
        s = G.Session(G.Model.from_tensors(cfg, W), batch=len(u))
        s.step(np.zeros(len(u), np.int32))
        got = s.pick(opt, uniforms=u)
    assert np.abs(got - want).max() <= 1, (got, want)
