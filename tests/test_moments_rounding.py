"""Second moments about a provisional centre: the difference <uv> - <u><v> rounds
once (csrc/rounding.hpp, compiled for the host), against exact fractions."""
import os
import random
import subprocess
from fractions import Fraction

from ocelot_amd import build

CSRC = os.path.join(build.HERE, "csrc")


def _cases(rng, count):
    """(S, n, a, b, S / n - a b rounded), the exact value away from a tie between
    two doubles by more than what second-order rests can move."""
    out = []
    while len(out) < count:
        n = rng.randint(3, 10 ** rng.randint(1, 8))
        a, b = (rng.gauss(0, 0.15) for _ in range(2))
        if rng.random() < 0.5:
            b = a
        S = n * (a * b + rng.uniform(0.3, 2.0))
        exact = Fraction(S) / n - Fraction(a) * Fraction(b)
        near = float(exact)
        gap = Fraction(abs(float.fromhex("0x1p-52") * near))
        if abs(exact - Fraction(near)) < Fraction(45, 100) * gap / 2:
            out.append((S, n, a, b, near))
    return out


def test_difference_rounds_once(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text('#include "rounding.hpp"\n#include <cstdio>\nint main() {\n  int bad = 0;\n' + "".join(
        f"  bad += ocsc::centred_difference({S.hex()}, {n}., {a.hex()}, {b.hex()}) != {v.hex()};\n"
        for S, n, a, b, v in _cases(random.Random(3), 400)) + '  printf("%d", bad);\n}\n')
    subprocess.run(["g++", "-std=c++17", "-O1", "-ffp-contract=off", "-I", CSRC, "-o", str(exe), str(src)], check=True)
    assert subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout == "0"
