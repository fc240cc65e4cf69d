"""Steps of 2 to 16 sequences with all layers in one launch: the same bits as a launch per operation
(the graph engine), whatever the batch, the context and the place of the cache pages; and the same
results when a step has to be given up, when the chip is someone else's, and where the tags start over."""
import threading
import time

import numpy as np
import pytest

import gradhip as G
import oracle_lib as O
from gradhip import synth
from helpers import assert_logits_close, lively_std

pytestmark = pytest.mark.gpu

SHAPES = {
    "gpt2-d512": synth.Config(synth.ARCH_GPT2, 150, 512, 2, 8, 1100),
    "gpt2-d768": synth.Config(synth.ARCH_GPT2, 150, 768, 2, 12, 1100),
    "llama-d768": synth.Config(synth.ARCH_MODERN, 150, 768, 2, 12, 1100),
}
RESIDENT = {"gpt2-d512": 4, "gpt2-d768": 4, "llama-d768": 3}  # launches per step


@pytest.fixture(scope="module")
def models():
    out = {}
    for name, cfg in SHAPES.items():
        W = synth.make_weights(cfg, 101, std=lively_std(cfg), norm_noise=0.1)
        out[name] = (cfg, W, G.Model.from_tensors(cfg, W))
    return out


def _both(gm, batch, **kw):
    return G.Session(gm, batch=batch, **kw), G.Session(gm, batch=batch, engine=G.ENGINE_GRAPH, **kw)


@pytest.mark.parametrize("batch", [2, 3, 4, 5, 8, 9, 13, 16])
@pytest.mark.parametrize("name", sorted(SHAPES))
def test_bits_of_a_launch_per_operation(models, name, batch):
    """From an empty cache, and behind prompts that end before a page, a run of positions and a
    workgroup's share of the context do."""
    cfg, _, gm = models[name]
    one, many = _both(gm, batch, shuffle_pages=True)
    for prompt, steps in ((0, 3), (31, 3), (62, 4), (126, 4), (254, 4), (511, 3), (1020, 6)):
        tokens = synth.uniform_tokens(batch * (prompt + steps), cfg.vocab, 102 + prompt).reshape(batch, -1)
        for s in (one, many):
            s.reset()
            if prompt:
                s.prefill(tokens[:, :prompt])
        for t in range(prompt, prompt + steps):
            a, b = one.step(tokens[:, t]), many.step(tokens[:, t])
            assert a.tobytes() == b.tobytes(), (prompt, t)
        for seq in (0, batch - 1):
            for layer in range(cfg.layers):
                for kv in (0, 1):
                    for pos in (prompt, prompt + steps - 1):
                        assert one.read_kv(seq, layer, kv, pos).tobytes() == many.read_kv(seq, layer, kv, pos).tobytes()
    assert one.decode(1, G.sampling(1.0, 0, 1.0, 1.0, True)).shape == (batch, 1)
    assert one.last_timing()["launches_per_step"] == RESIDENT[name]


def test_more_runs_of_positions_than_halves_of_workgroups():
    """8 x 12 heads in 6 runs each behind 2560 positions: the attention goes in two rounds, and the step
    before it in one."""
    cfg = synth.Config(synth.ARCH_MODERN, 90, 768, 1, 12, 2600)
    W = synth.make_weights(cfg, 103, std=lively_std(cfg), norm_noise=0.1)
    one, many = _both(G.Model.from_tensors(cfg, W), 8, shuffle_pages=True)
    tokens = synth.uniform_tokens(8 * 2563, cfg.vocab, 104).reshape(8, -1)
    for s in (one, many):
        s.prefill(tokens[:, :2558])
    for t in range(2558, 2563):
        assert one.step(tokens[:, t]).tobytes() == many.step(tokens[:, t]).tobytes(), t


@pytest.mark.parametrize("name, batch, behind", [("gpt2-d768", 13, 4096), ("llama-d768", 16, 4096), ("llama-d768", 8, 6144),
                                                 ("gpt2-d512", 16, 6144)])
def test_three_and_four_rounds_of_runs_in_two_layers(name, batch, behind):
    """The cells of the runs are used again in every round and by the next layer; here a step adds a run per head."""
    shape = SHAPES[name]
    cfg = synth.Config(shape.arch, 90, shape.d_model, 2, shape.heads, behind + 16)
    runs = [(p + 511) // 512 for p in (behind, behind + 1)]  # (the runs of contexts this long have 512 positions)
    assert {-(-batch * cfg.heads * r // 512) for r in runs} <= {2, 3, 4} and -(-batch * cfg.heads * runs[1] // 512) >= 3
    W = synth.make_weights(cfg, 103, std=lively_std(cfg), norm_noise=0.1)
    one, many = _both(G.Model.from_tensors(cfg, W), batch, shuffle_pages=True)
    tokens = synth.uniform_tokens(batch * (behind + 3), cfg.vocab, 112).reshape(batch, -1)
    for s in (one, many):
        s.prefill(tokens[:, :behind - 2])
    for t in range(behind - 2, behind + 3):
        assert one.step(tokens[:, t]).tobytes() == many.step(tokens[:, t]).tobytes(), t
    assert one.decode(1, G.sampling(1.0, 0, 1.0, 1.0, True)).shape == (batch, 1)
    assert one.last_timing()["launches_per_step"] == RESIDENT[name]


@pytest.mark.parametrize("batch, behind", [(4, 5112), (3, 7160)])
def test_a_run_that_outgrows_the_kernel(batch, behind):
    """Up to 4 sequences take one round: one call whose first steps are resident and whose later ones are launches."""
    cfg = synth.Config(synth.ARCH_MODERN, 90, 768, 2, 12, behind + 40)
    W = synth.make_weights(cfg, 113, std=lively_std(cfg), norm_noise=0.1)
    one, many = _both(G.Model.from_tensors(cfg, W), batch, shuffle_pages=True)
    opt = G.sampling(0.9, 0, 1.0, 1.1, False)
    tokens = synth.uniform_tokens(batch * behind, cfg.vocab, 114).reshape(batch, behind)
    for s in (one, many):
        s.prefill(tokens)
    assert batch * 12 * ((behind + 511) // 512) <= 512 < batch * 12 * ((behind + 30 + 511) // 512)
    for n, resident in ((5, True), (25, False)):
        assert one.decode(n, opt, seed=n).tobytes() == many.decode(n, opt, seed=n).tobytes()
        assert (one.last_timing()["launches_per_step"] == RESIDENT["llama-d768"]) == resident


@pytest.mark.parametrize("name", sorted(SHAPES))
def test_steps_match_the_oracle(models, name):
    cfg, W, gm = models[name]
    s = G.Session(gm, batch=3)
    tokens = synth.uniform_tokens(18, cfg.vocab, 104).reshape(3, 6)
    got = [s.step(tokens[:, t]) for t in range(6)]
    for b in range(3):
        ref = O.Session(O.Model.from_tensors(cfg, W))
        for t in range(6):
            assert_logits_close(got[t][b], ref.step(int(tokens[b, t])), what=f"resident {name} step {t}")


def test_pages_of_32_positions_and_small_ones(models):
    """32 positions per page is the least the kernel takes; below, launches."""
    cfg, _, gm = models["llama-d768"]
    tokens = synth.uniform_tokens(4 * 70, cfg.vocab, 105).reshape(4, 70)
    got = []
    for page in (16, 32, 128):
        s = G.Session(gm, batch=4, page_tokens=page, shuffle_pages=True)
        s.prefill(tokens[:, :60])
        got.append(np.stack([s.step(tokens[:, t]) for t in range(60, 70)]))
    assert got[0].tobytes() == got[1].tobytes() == got[2].tobytes()


def _calls(s, cfg):
    """Every kind of call, one after the other on one session."""
    out = []
    prompt = synth.uniform_tokens(s.batch * 5, cfg.vocab, 106).reshape(s.batch, 5)
    plain, greedy = G.sampling(0.9, 0, 1.0, 1.1, False), G.sampling(1.0, 0, 1.0, 1.0, True)
    out.append(s.generate(prompt, 7, plain, seed=3))
    out.append(s.decode(6, greedy))
    streamed = []
    s.decode_stream(6, plain, lambda ids, i: streamed.append(np.array(ids)), seed=4)
    out.append(np.stack(streamed))
    out.append(s.step(prompt[:, 0]))
    s.reset()
    out.append(s.prefill(prompt))
    s.reset()
    out.append(s.score(prompt, prompt[:, ::-1].copy()))
    out.append(s.decode(4, plain, seed=5))
    return out


@pytest.mark.parametrize("spins", ["0", "3"])
def test_a_step_that_gives_up_runs_as_launches(models, monkeypatch, spins):
    """With next to no patience (a wait may look at a cell once or a few times) the first step of
    whatever call gives up; the call's results are those of the launches."""
    cfg, _, gm = models["llama-d768"]
    want = _calls(G.Session(gm, batch=5, engine=G.ENGINE_GRAPH), cfg)
    monkeypatch.setenv("GRADHIP_TEST_RESIDENT_SPINS", spins)
    s = G.Session(gm, batch=5)
    for i, (a, b) in enumerate(zip(_calls(s, cfg), want)):
        assert np.asarray(a).tobytes() == np.asarray(b).tobytes(), (spins, i)
    if spins == "0":
        assert s.last_timing()["launches_per_step"] > 10  # it did give up
    # ... and each call as the one that meets it
    prompt = synth.uniform_tokens(25, cfg.vocab, 106).reshape(5, 5)
    plain = G.sampling(0.9, 0, 1.0, 1.1, False)
    for call in ("decode", "stream", "step"):
        res = []
        for s in (G.Session(gm, batch=5), G.Session(gm, batch=5, engine=G.ENGINE_GRAPH)):
            long = np.tile(prompt, (1, 4))
            s.prefill(long)  # one pass: nothing resident before the call
            if call == "decode":
                res.append(s.decode(6, plain, seed=8))
            elif call == "stream":
                got = []
                s.decode_stream(6, plain, lambda ids, i: got.append(np.array(ids)), seed=8)
                res.append(np.stack(got))
            else:
                res.append(s.step(prompt[:, 1]))
            res.append(s.step(prompt[:, 2]))
        assert res[0].tobytes() == res[2].tobytes() and res[1].tobytes() == res[3].tobytes(), call


@pytest.mark.parametrize("name", sorted(SHAPES))
def test_a_session_that_gave_up_tries_again(models, monkeypatch, name):
    """The step that gives up is the call's first one or a late one; so many steps later, twice as many the second
    time, the session's steps are resident again."""
    cfg, _, gm = models[name]
    greedy, plain = G.sampling(1.0, 0, 1.0, 1.0, True), G.sampling(0.9, 0, 1.0, 1.1, False)
    prompt = synth.uniform_tokens(5 * 40, cfg.vocab, 109).reshape(5, 40)
    monkeypatch.setenv("GRADHIP_TEST_RESIDENT_REST", "4")
    for first in (0, 17):
        monkeypatch.setenv("GRADHIP_TEST_RESIDENT_SPINS", f"0,{first},1")
        s, ref = _both(gm, 5)
        for x in (s, ref):
            x.prefill(prompt)  # one pass: nothing resident before the calls
        for n, opt, resident in ((24, plain, False), (4, plain, False), (3, greedy, True), (9, plain, True)):
            assert s.decode(n, opt, seed=n).tobytes() == ref.decode(n, opt, seed=n).tobytes(), (first, n)
            assert (s.last_timing()["launches_per_step"] == RESIDENT[name]) == resident, (first, n)
        assert s.step(prompt[:, 0]).tobytes() == ref.step(prompt[:, 0]).tobytes()
    monkeypatch.setenv("GRADHIP_TEST_RESIDENT_SPINS", "0,0,2")
    s, ref = _both(gm, 5)
    for x in (s, ref):
        x.prefill(prompt)
    for i, resident in enumerate([False] + 4 * [False] + [False] + 8 * [False] + 3 * [True]):
        assert s.decode(1, plain, seed=i).tobytes() == ref.decode(1, plain, seed=i).tobytes(), i
        assert (s.last_timing()["launches_per_step"] == RESIDENT[name]) == resident, i


@pytest.mark.parametrize("looks", [1, 4, 12, 40])
@pytest.mark.parametrize("name", ["gpt2-d768", "llama-d768"])
def test_giving_up_in_a_long_context(models, monkeypatch, name, looks):
    """Three runs of positions per head: with more or fewer looks it is the rows, q or another workgroup's share
    that is not waited for, in a streamed run and in single steps."""
    cfg, _, gm = models[name]
    plain = G.sampling(0.9, 0, 1.0, 1.1, False)
    prompt = synth.uniform_tokens(9 * 1050, cfg.vocab, 111).reshape(9, 1050)
    monkeypatch.setenv("GRADHIP_TEST_RESIDENT_SPINS", f"{looks},3,2")
    monkeypatch.setenv("GRADHIP_TEST_RESIDENT_REST", "2")
    out = []
    for s in _both(gm, 9, shuffle_pages=True):
        s.prefill(prompt)
        got = []
        s.decode_stream(12, plain, lambda ids, i: got.append(np.array(ids)), seed=8)
        out.append(np.stack(got).tobytes() + b"".join(s.step(prompt[:, t]).tobytes() for t in range(5)))
    assert out[0] == out[1]


def test_tags_start_over(models, monkeypatch):
    cfg, _, gm = models["llama-d768"]
    monkeypatch.setenv("GRADHIP_TEST_NEAR_WRAP", "5")
    one, many = _both(gm, 4)
    tokens = synth.uniform_tokens(4 * 12, cfg.vocab, 107).reshape(4, 12)
    for t in range(12):
        assert one.step(tokens[:, t]).tobytes() == many.step(tokens[:, t]).tobytes(), t


def test_sessions_on_several_threads(models):
    """Two batched sessions and a single-sequence one at the same time: only one may have the chip to
    itself, the others go on as launches or wait their turn."""
    cfg, _, gm = models["llama-d768"]
    opt = G.sampling(0.9, 0, 1.0, 1.1, False)
    prompts = {b: synth.uniform_tokens(b * 20, cfg.vocab, 108 + b).reshape(b, 20) for b in (1, 4, 9)}
    want = {b: G.Session(gm, batch=b).generate(p, 24, opt, seed=b) for b, p in prompts.items()}
    bad = []

    def run(b):
        s = G.Session(gm, batch=b)
        for _ in range(5):
            if s.generate(prompts[b], 24, opt, seed=b).tobytes() != want[b].tobytes():
                bad.append(b)

    threads = [threading.Thread(target=run, args=(b,)) for b in prompts]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=60)
    assert not bad and not any(t.is_alive() for t in threads)


def _beside_a_batch(gm, vocab, call):
    """Runs call(session, prompts) of a batch on a thread of its own and 20 steps of a single sequence from 5 ms later
    on; which of the two ended first, and what both returned."""
    prompts = synth.uniform_tokens(13 * 12, vocab, 130).reshape(13, 12)
    tokens = synth.uniform_tokens(20, vocab, 131)
    batch, single = G.Session(gm, batch=13), G.Session(gm, batch=1)
    want = call(batch, prompts), [single.step([t]) for t in tokens]  # alone, and everything has been used once
    batch.reset()
    single.reset()
    order, out, started = [], {}, threading.Event()

    def run():
        started.set()
        out["batch"] = call(batch, prompts)
        order.append("batch")

    thread = threading.Thread(target=run)
    thread.start()
    started.wait()
    time.sleep(0.005)
    out["single"] = [single.step([t]) for t in tokens]
    order.append("single")
    thread.join(timeout=60)
    assert not thread.is_alive()
    assert out["batch"].tobytes() == want[0].tobytes()
    assert np.stack(out["single"]).tobytes() == np.stack(want[1]).tobytes()
    return order


@pytest.mark.parametrize("kind", ["generate", "stream"])
def test_a_single_sequence_does_not_wait_for_a_whole_batched_call(models, kind):
    """A batch of 900 tokens (some 50 ms) has the chip; 20 single steps (2 ms) that begin 5 ms later end before it."""
    cfg, _, gm = models["llama-d768"]
    opt = G.sampling(0.9, 0, 1.0, 1.1, False)

    def call(s, prompts):
        if kind == "generate":
            return s.generate(prompts, 900, opt, seed=9)
        got = []
        s.prefill(prompts)
        s.decode_stream(900, opt, lambda ids, i: got.append(np.array(ids)), seed=9)
        return np.stack(got)

    assert _beside_a_batch(gm, cfg.vocab, call) == ["single", "batch"]


def test_a_callback_may_use_any_session(models):
    """Inside the callback of a streamed batch, and of a streamed single sequence, which has the chip."""
    cfg, _, gm = models["llama-d768"]
    opt = G.sampling(1.0, 0, 1.0, 1.0, True)
    prompt = {b: synth.uniform_tokens(b * 10, cfg.vocab, 120 + b).reshape(b, 10) for b in (1, 3, 6)}
    alone = {b: G.Session(gm, batch=b).generate(prompt[b], 5, opt) for b in (1, 6)}
    for outer, inner in ((3, 1), (3, 6), (1, 6)):
        other = G.Session(gm, batch=inner)
        s = G.Session(gm, batch=outer)
        s.prefill(prompt[outer])
        seen = []
        s.decode_stream(4, opt, lambda ids, i: seen.append(other.generate(prompt[inner], 5, opt)))
        assert len(seen) == 4
        for got in seen:
            assert got.tobytes() == alone[inner].tobytes(), (outer, inner)
