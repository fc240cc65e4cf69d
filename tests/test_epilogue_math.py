"""GELU, SiLU and exponentials of the pair products' epilogues, compiled for the host: with a 2^x and a reciprocal as far off
as the hardware's, the errors of the first two against double are no larger than those of tanhf, expf and a division, those
of the exponentials no larger than what 2^x leaves of its own, and they have next to no error in common."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_errors_are_no_larger_than_the_functions_own(tmp_path):
    exe = str(tmp_path / "epilogue_math_test")
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-Wall", "-Wextra",
                           os.path.join(ROOT, "tests", "cpp", "epilogue_math_test.cpp"), "-o", exe])
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60, check=True).stdout.strip().split("\n")
    lines = [line.split() for line in out]
    ratios = {tuple(line[:2]): float(line[2]) for line in lines if line[0] in ("gelu", "silu")}
    assert len(ratios) == 12
    assert max(ratios.values()) <= 1.0, ratios
    # (the argument's fraction is rounded too: at most 2^-26, a sixth of a typical error of 2^x, so 1.4 % more)
    assert [float(line[1]) <= 1.02 for line in lines if line[0] == "exp"] == [True]
    assert [abs(float(line[2])) <= 10.0 for line in lines if line[0] == "common"] == [True]  # a sixth of an fp32 unit
    ends = [line for line in lines if line[:2] == ["ends", "gelu"]]
    for line, want in zip(ends, (0.0, 0.0, 0.0, 200.0, 1e12, float("nan"))):
        for got in (float(line[2]), float(line[4])):
            assert got == want or abs(got - want) <= 1e-25 or (want != want and got != got), line
    ends = [float(line[2]) for line in lines if line[:2] == ["ends", "exp"]]
    assert ends[0] == 0.0 and ends[1] == 0.0 and ends[2] <= 1e-40 and ends[3] == 1.0 and ends[4] != ends[4]
