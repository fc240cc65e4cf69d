"""Passes over up to a few hundred rows (batched steps, prompts below the split products): the same
rows give the same bits whatever the tiles, the blocks of queries and the company they are in, and
agree with the float64 forward."""
import numpy as np
import pytest

import gradhip as G
import ref_forward
from gradhip import synth
from helpers import assert_logits_close, lively_std

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [256, 320, 512, 768, 1024])
def test_layernorm_of_batched_steps(d):
    """The widths whose rows stay in registers, and one that takes the general norm."""
    cfg = synth.Config(synth.ARCH_GPT2, 201, d, 2, d // 64, 16)
    W = synth.make_weights(cfg, 91, std=lively_std(cfg), norm_noise=0.3)
    s = G.Session(G.Model.from_tensors(cfg, W), batch=3)
    tokens = synth.uniform_tokens(15, cfg.vocab, 92).reshape(3, 5)
    got = [s.step(tokens[:, t]) for t in range(5)]
    for b in range(3):
        ref = ref_forward.forward(cfg, W, tokens[b])
        for t in range(5):
            assert_logits_close(got[t][b], ref[t], what=f"layernorm {d} step {t}")


@pytest.mark.parametrize("arch, d", [(synth.ARCH_GPT2, 512), (synth.ARCH_MODERN, 768)])
def test_tiles_do_not_change_a_pass(arch, d):
    """Row counts from 65 to 511 take different tiles; a sequence's logits are the same in all of them."""
    cfg = synth.Config(arch, 201, d, 2, d // 64, 80)
    W = synth.make_weights(cfg, 93, std=lively_std(cfg), norm_noise=0.1)
    gm = G.Model.from_tensors(cfg, W)
    tokens = synth.uniform_tokens(73, cfg.vocab, 94)
    ref = ref_forward.forward(cfg, W, tokens)[-1]
    last = None
    for batch in (1, 2, 3, 4, 5, 6, 7):
        got = G.Session(gm, batch=batch).prefill(np.tile(tokens, (batch, 1)))
        assert_logits_close(got[0], ref, what=f"tiles batch {batch}")
        if batch > 1:  # (one sequence's logits are formed by another kernel)
            last = got[0] if last is None else last
            for b in range(batch):
                assert got[b].tobytes() == last.tobytes(), (batch, b)


@pytest.mark.parametrize("arch, d", [(synth.ARCH_GPT2, 512), (synth.ARCH_MODERN, 768), (synth.ARCH_GPT2, 1024)])
def test_tiles_do_not_change_the_cache(arch, d):
    """Rows around whole tiles of 48 and 32: what a prompt leaves of its first positions is the same after any number
    of rows behind them, tiles of 3 x 2 and 2 x 3 among them (matrices whose outputs are no multiple of 48 too)."""
    cfg = synth.Config(arch, 201, d, 2, d // 64, 520)
    W = synth.make_weights(cfg, 99, std=lively_std(cfg), norm_noise=0.1)
    gm = G.Model.from_tensors(cfg, W)
    tokens = synth.uniform_tokens(511, cfg.vocab, 100)
    kept = None
    for n in (96, 160, 192, 193, 255, 257, 336, 384, 385, 432, 433, 511):
        s = G.Session(gm)
        got = s.prefill(tokens[:n])
        if n in (193, 384, 511):
            assert_logits_close(got, ref_forward.forward(cfg, W, tokens[:n])[-1], what=f"cache {d} {n}")
        rows = [s.read_kv(0, 1, kv, pos).tobytes() for kv in (0, 1) for pos in (0, 31, 47, 95)]
        kept = kept or rows
        assert rows == kept, n


def test_tiles_do_not_change_a_batched_step():
    """33 to 64 sequences: up to 48 the FFN's first matrix goes tile by tile, beyond in pairs of tiles."""
    cfg = synth.Config(synth.ARCH_MODERN, 201, 768, 1, 12, 16)
    W = synth.make_weights(cfg, 97, std=lively_std(cfg), norm_noise=0.1)
    gm = G.Model.from_tensors(cfg, W)
    tokens = synth.uniform_tokens(3, cfg.vocab, 98)
    ref = ref_forward.forward(cfg, W, tokens)[-1]
    last = None
    for batch in (33, 48, 49, 64):
        s = G.Session(gm, batch=batch)
        for t in tokens:
            got = s.step(np.full(batch, t, np.int32))
        assert_logits_close(got[0], ref, what=f"step tiles batch {batch}")
        last = got[0].copy() if last is None else last
        for b in range(batch):
            assert got[b].tobytes() == last.tobytes(), (batch, b)


@pytest.mark.parametrize("batch, n, before", [(1, 8, 0), (1, 16, 0), (1, 17, 3), (1, 64, 0), (1, 65, 0), (2, 129, 0), (1, 33, 70),
                                              (3, 50, 127), (40, 9, 60)])
def test_query_blocks_do_not_change_a_pass(batch, n, before):
    """Blocks of 16 queries (pages of 64 positions and more) against blocks of 64 (smaller pages)."""
    cfg = synth.Config(synth.ARCH_MODERN, 130, 128, 2, 2, 300)
    W = synth.make_weights(cfg, 95, std=lively_std(cfg), norm_noise=0.1)
    gm = G.Model.from_tensors(cfg, W)
    tokens = synth.uniform_tokens(batch * (n + before), cfg.vocab, 96).reshape(batch, -1)
    got = []
    for page in (32, 64, 128):
        s = G.Session(gm, batch=batch, page_tokens=page, shuffle_pages=True)
        if before:
            s.prefill(tokens[:, :before])
        got.append(s.prefill(tokens[:, before:]))
    assert got[1].tobytes() == got[0].tobytes() and got[2].tobytes() == got[0].tobytes()
    ref = ref_forward.forward(cfg, W, tokens[batch - 1])[-1]
    assert_logits_close(got[1][batch - 1], ref, what=f"queries {batch} x {n}")


@pytest.mark.parametrize("arch, d", [(synth.ARCH_GPT2, 576), (synth.ARCH_MODERN, 896), (synth.ARCH_GPT2, 1152)])
def test_widths_dealt_unevenly_to_the_xcds(arch, d):
    """Runs of outputs that are no multiple of eight: the same first positions behind any number of rows, whatever tiles those take."""
    cfg = synth.Config(arch, 201, d, 2, d // 64, 520)
    W = synth.make_weights(cfg, 135, std=lively_std(cfg), norm_noise=0.1)
    gm = G.Model.from_tensors(cfg, W)
    tokens = synth.uniform_tokens(511, cfg.vocab, 136)
    kept = None
    for n in (66, 200, 300, 333, 397, 420, 511):
        s = G.Session(gm)
        got = s.prefill(tokens[:n])
        if n in (66, 397):
            assert_logits_close(got, ref_forward.forward(cfg, W, tokens[:n])[-1], what=f"uneven {d} {n}")
        rows = [s.read_kv(0, 1, kv, pos).tobytes() for kv in (0, 1) for pos in (0, 31, 47, 65)]
        kept = kept or rows
        assert rows == kept, n
