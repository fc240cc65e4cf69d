"""Draws without a top-k cut, where the row's split over threads and the top-p cut can go
wrong: vocabularies at the edges of what a thread holds in registers (16 and 32 elements
of 1024 or 512 threads), cuts at the very first and the very last value, flat rows whose cut
lies in a crowded bin, and rows so peaked that it lies far below the maximum."""
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
