"""The scaling of a sixfold-growing state (csrc/hwt_scale.h), run on the CPU through its
own loop: whatever the pieces, the steps add up, and the exponent left over stays below
one bit after a scaling and below 64 steps' growth and one bit before it."""
import math
import shutil
import subprocess

import numpy as np
import pytest

from conftest import ROOT

PROGRAM = r"""
#include "hwt_scale.h"
#include <cstdio>
#include <cstdlib>
// argv: pieces of one state's steps.  Out: steps made, bits scaled away, the most steps
// between scalings, the largest and smallest number of bits over 2^-32 left after one.
int main(int, char **)
{
    hwt::SixfoldScale s;
    long long steps = 0, since = 0, most = 0, bits = 0, piece;
    double over = 0, hi = 0, lo = 0;  // log2 of the state: grows by log2 6 a step
    const double log2_6 = 2.5849625007211561815;
    while (std::scanf("%lld", &piece) == 1)
        hwt::scaled_steps(
            s, (int)piece,
            [&](int c) {
                if (c < 1) std::abort();
                steps += c;
                since += c;
                if (since > most) most = since;
            },
            [&](double f) {
                int e = 0;
                if (__builtin_frexp(f, &e) != 0.5) std::abort();  // a power of two
                bits += 1 - e;
                since = 0;
                over = steps * log2_6 - bits;
                if (over > hi) hi = over;
                if (over < lo) lo = over;
            });
    std::printf("%lld %lld %lld %.17g %.17g %.17g\n", steps, bits, most, hi, lo, steps * log2_6 - bits);
}
"""


@pytest.fixture(scope="module")
def emulate(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if not cxx:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("scale")
    (d / "scale.cpp").write_text(PROGRAM)
    inc = ROOT / "diku.optionspricing_amd" / "csrc"
    subprocess.run([cxx, "-O2", "-std=c++17", f"-I{inc}", "-o", d / "scale", d / "scale.cpp"], check=True)

    def run(pieces):
        text = " ".join(str(int(p)) for p in pieces)
        return [float(v) for v in subprocess.run([d / "scale"], input=text, check=True, capture_output=True,
                                                 text=True).stdout.split()]
    return run


PIECES = {
    "one": [1_000_000], "ones": [1] * 5000, "63 then 64": [63, 64] * 2000, "65s": [65] * 3000, "64s": [64] * 3000,
    "zeros": [0, 1, 0, 200] * 500, "starts and swaps": np.random.default_rng(1).integers(0, 200, 4000),
    "windows": np.random.default_rng(2).integers(1, 3000, 4000), "a few": [1, 2, 3],
    "two thousand million": [2_000_000_000],
}


@pytest.mark.parametrize("name", PIECES)
def test_scaling_follows_the_growth(emulate, name):
    steps, bits, most, hi, lo, end = emulate(PIECES[name])
    assert steps == sum(int(p) for p in PIECES[name])
    assert most <= 64
    slack = 1e-5 + steps * 2.0**-33  # the sum's own rounding here, and log2 6 in units of 2^-32
    assert -slack <= lo and hi < 1 + slack
    assert -slack <= end < 64 * math.log2(6) + 1 + slack


LEFT = r"""
#include "hwt_scale.h"
#include <cstdio>
// argv: from, to.  Out: log2 of a state that grew from step `from` to step `to` of a count
// scaled all along, less what sixfold_left gives.
int main()
{
    int from, to;
    while (std::scanf("%d %d", &from, &to) == 2) {
        hwt::SixfoldScale s;
        double bits = 0;
        auto steps = [](int) {};
        auto scale = [&](double f) {
            int e = 0;
            __builtin_frexp(f, &e);
            bits += e - 1;
        };
        hwt::scaled_steps(s, from, steps, scale);
        bits = 0;
        hwt::scaled_steps(s, to - from, steps, scale);
        std::printf("%.17g\n", (to - from) * 2.5849625007211561815 + bits - hwt::sixfold_left(from, to));
    }
}
"""


def test_what_the_scaling_left(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if not cxx:
        pytest.skip("no host compiler")
    (tmp_path / "left.cpp").write_text(LEFT)
    inc = ROOT / "diku.optionspricing_amd" / "csrc"
    subprocess.run([cxx, "-O2", "-std=c++17", f"-I{inc}", "-o", tmp_path / "left", tmp_path / "left.cpp"], check=True)
    r = np.random.default_rng(3)
    pairs = [(0, 0), (0, 63), (0, 64), (63, 64), (63, 127), (1, 64), (64, 64), (0, 1_000_000)]
    pairs += [tuple(sorted(r.integers(0, 300_000, 2))) for _ in range(500)]
    text = " ".join(f"{a} {b}" for a, b in pairs)
    out = subprocess.run([tmp_path / "left"], input=text, check=True, capture_output=True, text=True).stdout
    assert all(-2 <= float(v) <= 2 for v in out.split())
