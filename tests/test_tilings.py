"""What the GPU tests of passes over many rows launch, by the rules that choose forms and tilings: every combination that a
rule can give has a case, so that a change of the rules cannot leave a kernel without one."""
import pytest

import row_tilings
import test_gpu_pair_rows
import test_gpu_split_tall
from gradhip import synth

BLOCKS = (synth.ARCH_GPT2, synth.ARCH_MODERN)


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    return row_tilings.compile_rules(tmp_path_factory.mktemp("tilings"))


def _all(rules, cases):
    return set().union(*row_tilings.launches(rules, cases))


def test_every_launch_in_pairs_has_a_case(rules):
    cases = [(arch, *case, True) for case in test_gpu_pair_rows.CASES for arch in BLOCKS]
    cases += [(*case, True) for case in test_gpu_pair_rows.MORE_CASES]
    sizes = [(arch, d, vocab, B, n, True) for arch in BLOCKS for d in (512, 576, 640, 768, 1024, 1280, 1536)
             for vocab in (130, 515, 1001, 5000, 16000, 50257) for B in (1, 2, 3, 4, 5, 6, 9, 17, 32)
             for n in (20, 24, 33, 40, 60, 90, 130, 171, 250, 300, 400, 520, 1000, 2000) if 24 <= B * n <= 16384]
    can = {launch for launch in _all(rules, sizes) if launch[0] == "pairs"}
    assert len(can) >= 43, sorted(can)
    assert can <= _all(rules, cases), sorted(can - _all(rules, cases))


def test_whole_vocabularies_are_scored_in_the_tilings_that_programs_use(rules):
    cases = [(arch, *case, True) for case in test_gpu_pair_rows.CASES for arch in BLOCKS]
    cases += [(*case, True) for case in test_gpu_pair_rows.MORE_CASES]
    tested = {tiling for form, what, tiling in _all(rules, cases) if (form, what) == ("pairs", "logits")}
    for vocab in (5000, 16000, 32000, 50257):
        for n in (24, 60, 171, 256, 700, 2048, 16384):
            for d in (512, 768):
                taken, = row_tilings.launches(rules, [(synth.ARCH_MODERN, d, vocab, 1, n, True)])
                assert {t for form, what, t in taken if (form, what) == ("pairs", "logits")} <= tested, (vocab, n, d, taken)


def test_three_parts_of_128_x_64_tiles_have_cases(rules):
    cases = [(arch, 768, test_gpu_split_tall.VOCAB, B, n, False) for B, n in test_gpu_split_tall.CASES.values() for arch in BLOCKS]
    assert {("parts", what, "128x64") for what in ("qkv", "resid", "gelu", "swiglu", "logits")} <= _all(rules, cases)
    more, = row_tilings.launches(rules, [(synth.ARCH_GPT2, 768, 130, 1, 2689, False)])  # one row more than a round takes
    assert ("parts", "resid", "128") in more


def test_forms_change_where_the_gpu_tests_say(rules):
    for d, n, in_pairs, change in test_gpu_pair_rows.FORMS.values():
        if change is None:
            taken, = row_tilings.launches(rules, [(synth.ARCH_GPT2, d, 301, 1, n, True)])
            assert {form for form, what, _ in taken if what != "logits"} == {"pairs" if in_pairs else "parts"}, (d, n)


def _rounds(M, N, rows, outputs):
    """Of the XCD that is dealt the most workgroups, by the kernel's map of ids (gemm16_kernel), on its 32 compute units."""
    row_groups, runs = -(-M // (16 * rows)), -(-N // (16 * outputs))
    dealt = [0] * 8
    for at in range(-(-runs // 8) * 8 * row_groups):
        xcd, slot = at & 7, at >> 3
        dealt[xcd] += xcd + 8 * (slot // row_groups) < runs
    return -(-max(dealt) // 32)


def test_few_rows_take_the_tiles_that_the_fullest_xcd_ends_first_with(rules):
    """Widths whose runs of outputs are no multiple of eight among them: 511 x 576 in 3 x 2 tiles were two rounds taken for one."""
    sizes = [(M, N, six) for M in (65, 96, 150, 200, 256, 333, 397, 420, 511) for N in (512, 576, 640, 832, 896, 1152, 1408, 2304, 5504)
             for six in (0, 1)]
    out = row_tilings.ask(rules, [f"few {M} {N} {six}" for M, N, six in sizes])
    for (M, N, six), got in zip(sizes, out):
        each = {"2x2": 40, "1x2": 24 if N > 1024 else 25, "2x1": 25 if N > 1024 else 24, "1x1": 17}
        if six:
            each.update({"3x2": 59, "2x3": 62})
        cost = {name: _rounds(M, N, *map(int, name.split("x"))) * us for name, us in each.items()}
        assert got == min(cost, key=cost.get), (M, N, six, cost)  # (the first of equals)
