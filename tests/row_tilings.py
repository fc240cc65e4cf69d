"""Which forms and tilings a pass over many rows takes, by the library's own rules (tilings.h, compiled for the host)."""
import os
import subprocess

from gradhip import synth

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MIN_SCORED, MIN_PROMPT = 160, 512  # rows from which a scored pass and a prompt take split products


def compile_rules(path):
    exe = os.path.join(str(path), "tilings_test")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", os.path.join(ROOT, "tests", "cpp", "tilings_test.cpp"),
                           "-o", exe])
    return exe


def ask(exe, lines):
    return subprocess.run([exe], input="\n".join(lines) + "\n", capture_output=True, text=True, check=True,
                          timeout=60).stdout.splitlines()


def launches(exe, cases):
    """Of every (arch, width, vocabulary, sequences, tokens, whether the weights have pairs), scored and as a prompt: the set of
    (form, epilogue, tiling) it runs; keys: keys and values alone, of the last layer of a prompt."""
    lines, wanted = [], []
    for arch, d, vocab, B, n, fit in cases:
        cfg = synth.Config(arch, vocab, d, 1, d // 64, n + 1)
        M, F = B * n, cfg.d_ff
        ffn1, act = (2 * F, "swiglu") if cfg.modern else (F, "gelu")
        lines += [f"layers {d} {ffn1} {M}", f"logits {d} {vocab} {M}"]
        wanted.append([("qkv", 3 * d, d), ("keys", 2 * d, d), ("resid", d, d), (act, ffn1, d), ("resid", d, F), ("logits", vocab, d)])
        for what, N, K in wanted[-1]:
            lines += [f"parts {M} {N} {K}", f"pairs {M} {N} {K} {what if what in ('gelu', 'swiglu', 'logits') else 'rows'}"]
    out = iter(ask(exe, lines))
    found = []
    for (arch, d, vocab, B, n, fit), products in zip(cases, wanted):
        layers, logits = next(out), next(out)
        taken = set()
        for what, N, K in products:
            tiling = {"parts": next(out), "pairs": next(out)}
            least = {"keys": MIN_PROMPT, "logits": 0}.get(what, MIN_SCORED)
            form = (logits if what == "logits" else layers) if fit else "parts"
            if B * n >= least:
                taken.add((form, what, tiling[form]))
        found.append(taken)
    return found
