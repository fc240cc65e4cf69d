"""The work a program gives this framework, as cases that can be timed.

Every case is one call pattern of the public Python binding (the same entry points the C ABI
and the C++ adapter have): a prompt and a run of generated tokens, a loop of single steps with
the caller's own sampler, a chat turn that streams its reply, a prompt alone, or the scoring of
token windows.  Models are the three block shapes the framework is configured for (a GPT-2
block at width 512 and at width 768, a Llama block at width 768), with weights N(0, 0.02) from
a fixed seed; prompts and draws come from the seed of the inputs.  All arithmetic is fp32.

A case is a dict of plain values:
  kind      generate | fresh_generate | step | stream | prefill | score
  model     a key of MODELS; vocab and context: the checkpoint's vocabulary and maximum length
  batch     sequences decoded in lock step
  prompt    prompt tokens per sequence (score: tokens per window)
  new       tokens generated, or single steps made, per sequence
  temperature, top_k, top_p, penalty, greedy   the sampler's options
"""
import collections
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "grad.cpp_amd"))
import gradhip as G  # noqa: E402
from gradhip import synth  # noqa: E402

#: name: (block, d_model, layers, heads)
MODELS = {
    "gpt2-small": (synth.ARCH_GPT2, 512, 6, 8),
    "gpt2-medium": (synth.ARCH_GPT2, 768, 8, 12),
    "llama": (synth.ARCH_MODERN, 768, 8, 12),
}

GREEDY = {"temperature": 1.0, "top_k": 0, "top_p": 1.0, "penalty": 1.0, "greedy": True}
GREEDY_PENALTY = {**GREEDY, "penalty": 1.2}
#: the defaults of the text generator: no cut, repetition penalty 1.2
PLAIN = {"temperature": 0.8, "top_k": 0, "top_p": 1.0, "penalty": 1.2, "greedy": False}
TOP_K_P = {"temperature": 0.8, "top_k": 40, "top_p": 0.9, "penalty": 1.1, "greedy": False}
NUCLEUS = {"temperature": 1.0, "top_k": 0, "top_p": 0.95, "penalty": 1.1, "greedy": False}
WIDE_K = {"temperature": 0.9, "top_k": 200, "top_p": 1.0, "penalty": 1.0, "greedy": False}
SAMPLERS = (GREEDY, GREEDY_PENALTY, PLAIN, TOP_K_P, NUCLEUS, WIDE_K)


def _case(kind, model, vocab, context, batch, prompt, new, sampler=GREEDY):
    return {"kind": kind, "model": model, "vocab": vocab, "context": context, "batch": batch, "prompt": prompt,
            "new": new, **sampler}


def listed():
    def named(name, *a, **k):
        return {"name": name, **_case(*a, **k)}

    return [
        # one token through the small model, the logits back on the host: the smallest call there is
        named("step-small", "step", "gpt2-small", 5000, 96, 1, 0, 1),
        # the generation benchmark of the reference: a session per request, a three-token prompt, 64 sampled tokens
        named("request-small", "fresh_generate", "gpt2-small", 5000, 1024, 1, 3, 64, PLAIN),
        # a short completion with the text generator's greedy defaults
        named("complete-medium", "generate", "gpt2-medium", 16000, 256, 1, 32, 64, GREEDY_PENALTY),
        # the headline: one sampled stream on the Llama block
        named("sample-llama", "generate", "llama", 16000, 256, 1, 32, 96, TOP_K_P),
        # a chat turn: a few hundred tokens of context, then a streamed reply with nucleus sampling
        named("chat-llama", "stream", "llama", 16000, 1024, 1, 397, 64, NUCLEUS),
        # a caller with a sampler of its own over a handful of sequences
        named("steps-llama-4", "step", "llama", 16000, 256, 4, 61, 24),
        # a modest serving batch, ragged in no dimension that matters to the caller
        named("serve-llama-13", "generate", "llama", 32000, 512, 13, 77, 48, TOP_K_P),
        # batched decoding of many short requests
        named("serve-llama-64", "generate", "llama", 16000, 256, 64, 128, 48),
        # long prompts in a batch, then decoding over a long cache
        named("long-llama-16", "generate", "llama", 16000, 2048, 16, 1536, 48),
        # a document read in one go before anything is generated
        named("prefill-llama-1999", "prefill", "llama", 16000, 2048, 1, 1999, 0),
        # evaluation: loss of token windows, the evaluation command's own batch of eight
        named("score-llama-8x256", "score", "llama", 16000, 256, 8, 256, 0),
        # evaluation at the presets' context with the GPT-2 block
        named("score-medium-16x1024", "score", "gpt2-medium", 16000, 1024, 16, 1024, 0),
    ]


def _log_int(rng, lo, hi):
    return int(round(2.0 ** rng.uniform(np.log2(lo), np.log2(hi))))


def draw(rng):
    kind = rng.choice(("generate", "generate", "generate", "fresh_generate", "step", "stream", "prefill", "prefill",
                       "score", "score"))
    model = rng.choice(("gpt2-small", "gpt2-medium", "llama", "llama"))
    vocab = 5000 if model == "gpt2-small" else rng.choice((16000, 16000, 32000, 50257))
    context = rng.choice((256, 1024, 2048))
    batch = 1 if kind in ("fresh_generate", "stream") else _log_int(rng, 1, 64)
    sampler = rng.choice(SAMPLERS)
    new = {"prefill": 0, "score": 0, "step": _log_int(rng, 1, 24)}.get(kind) if kind in ("prefill", "score", "step") \
        else _log_int(rng, 4, 64)
    # no drawn case is larger than the largest listed one: at most 16 k tokens in one prompt pass
    longest = min(context - new, 16384 // batch)
    prompt = _log_int(rng, 1, longest) if kind in ("generate", "fresh_generate", "step", "stream") \
        else _log_int(rng, min(24, longest), longest)
    return _case(kind, model, vocab, context, batch, prompt, new, sampler)


def _config(case):
    arch, d, layers, heads = MODELS[case["model"]]
    return synth.Config(arch, case["vocab"], d, layers, heads, case["context"])


# A program loads a checkpoint once and opens sessions on it; so do the cases of one process.
_MODELS = collections.OrderedDict()


def _model(case):
    key = (case["model"], case["vocab"], case["context"])
    if key not in _MODELS:
        while len(_MODELS) >= 6:
            _MODELS.popitem(last=False)
        cfg = _config(case)
        gen = torch.Generator(device="cuda").manual_seed(1009)
        tensors = []
        for _, rows, cols, what in synth.tensor_specs(cfg):
            if what in ("matrix", "bias"):
                t = (torch.randn(rows, cols, generator=gen, device="cuda") * 0.02).cpu().numpy()
            else:
                t = np.full((rows, cols), 1.0 if what == "gamma" else 0.0, np.float32)
            tensors.append(t)
        _MODELS[key] = G.Model.from_tensors(cfg, tensors)
    _MODELS.move_to_end(key)
    return _MODELS[key]


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    model = _model(case)
    state = {"case": case, "model": model, "seed": int(seed),
             "opt": G.sampling(case["temperature"], case["top_k"], case["top_p"], case["penalty"], case["greedy"])}

    def ids(n):
        return rng.integers(0, case["vocab"], (case["batch"], n), dtype=np.int32)

    state["prompt"] = ids(case["prompt"])
    if case["kind"] == "step":
        state["next"] = np.ascontiguousarray(ids(case["new"]).T)
    if case["kind"] == "score":
        state["targets"] = ids(case["prompt"])
    if case["kind"] != "fresh_generate":
        state["session"] = G.Session(model, batch=case["batch"])
    return state


def run(state):
    case, opt, seed = state["case"], state["opt"], state["seed"]
    kind = case["kind"]
    if kind == "generate":
        return state["session"].generate(state["prompt"], case["new"], opt, seed=seed)
    if kind == "fresh_generate":
        session = G.Session(state["model"], batch=case["batch"])
        tokens = session.generate(state["prompt"], case["new"], opt, seed=seed)
        session.close()
        return tokens
    session = state["session"]
    session.reset()
    if kind == "score":
        return session.score(state["prompt"], state["targets"])
    if kind == "prefill":
        return session.prefill(state["prompt"])
    if kind == "step":
        if case["prompt"]:
            session.prefill(state["prompt"])
        return [session.step(ids) for ids in state["next"]]
    reply = []
    session.prefill(state["prompt"])
    session.decode_stream(case["new"], opt, lambda ids, index: reply.append(ids[0]), seed=seed)
    return np.asarray(reply, np.int32)


def work(case):
    """Every matrix once per dependent pass over the model (a prompt, or one token of every
    sequence), the cache rows read and written, the outputs; the products behind the outputs.
    Of a prompt whose last position alone is asked for, the last layer needs only its keys and
    values everywhere else."""
    cfg = _config(case)
    d, f, v, layers, b = cfg.d_model, cfg.d_ff, cfg.vocab, cfg.layers, case["batch"]
    layer = 4 * d * d + (3 if cfg.modern else 2) * d * f
    weights = layers * layer + v * d
    n, new = case["prompt"], case["new"]
    passes, flops, cache, out = 0, 0.0, 0, 0
    if n:
        passes += 1
        rows_full = n if case["kind"] == "score" else 1  # rows that need all of the last layer and the logits
        pairs = n * (n + 1) / 2
        flops += 2.0 * b * (n * (layers - 1) * layer + n * 2 * d * d + rows_full * (layer - 2 * d * d + v * d))
        flops += 4.0 * b * d * ((layers - 1) * pairs + (pairs if case["kind"] == "score" else n))
        cache += b * layers * 2 * n * d
        out += b * n if case["kind"] == "score" else b * v if case["kind"] == "prefill" else 0
    for i in range(new):
        passes += 1
        flops += 2.0 * b * weights + 4.0 * b * layers * d * (n + i + 1)
        cache += b * layers * 2 * (n + i + 2) * d
        out += b * v if case["kind"] == "step" else b
    return {"bytes": 4.0 * (passes * weights + cache + out), "flops": flops}


def tolerance(case):
    # Logits and losses: fp32 sums of up to a few thousand terms through eight layers.  Token ids are
    # the same unless two candidates tie within that error; a sequence differs from such a tie on.
    return {"rel": 1e-5, "max": 2e-4, "differ": 0.01}
