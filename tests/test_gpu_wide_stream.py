"""Logits of batched steps over more vocabulary tiles than one round of workgroups takes (16 outputs per tile, four
tiles per workgroup and 256 workgroups: 16384 outputs), where workgroups walk on through the matrix: against one
sequence at a time, with a last tile and a last workgroup of every kind, and the greedy picks made from them."""
import numpy as np
import pytest

import gradhip as G
from gradhip import synth
from helpers import assert_logits_close, lively_std

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [2, 16, 17, 32])
@pytest.mark.parametrize("arch,d,vocab", [
    (synth.ARCH_MODERN, 768, 16384), (synth.ARCH_MODERN, 768, 16385), (synth.ARCH_MODERN, 768, 24593),
    (synth.ARCH_MODERN, 768, 50257), (synth.ARCH_GPT2, 768, 33000), (synth.ARCH_GPT2, 1024, 20481),
    (synth.ARCH_GPT2, 512, 33001)])
def test_batched_logits_and_greedy_picks(arch, d, vocab, batch):
    cfg = synth.Config(arch, vocab, d, 1, d // 64, 64)
    gm = G.Model.from_tensors(cfg, synth.make_weights(cfg, 51, std=lively_std(cfg), norm_noise=0.1))
    tokens = synth.uniform_tokens(batch * 2, vocab, 52).reshape(batch, 2)
    s = G.Session(gm, batch=batch)
    s.step(tokens[:, 0])
    got = np.array(s.step(tokens[:, 1]))
    one = G.Session(gm, batch=1, engine=G.ENGINE_EAGER)
    for b in sorted({0, 1, batch // 2, batch - 1}):
        one.reset()
        one.step(tokens[b, :1])
        want = np.asarray(one.step(tokens[b, 1:])).reshape(-1)
        assert_logits_close(got[b], want, 2e-5, f"wide {vocab} of {batch}, sequence {b}")
    # the launch's own candidates for the picks of a call: the first largest logit of every row
    picks = s.decode(3, G.sampling(1.0, 0, 1.0, 1.0, True))
    again = G.Session(gm, batch=batch)
    again.step(tokens[:, 0])
    row = again.step(tokens[:, 1])
    for t in range(3):
        assert np.array_equal(picks[:, t], np.asarray(row).argmax(axis=1)), t
        row = again.step(np.ascontiguousarray(picks[:, t]))
