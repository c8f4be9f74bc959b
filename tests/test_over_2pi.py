"""gather::over_2pi, x/2π without a division, against the division: compiled for the
CPU from the header's own text."""
import os
import re
import subprocess
from fractions import Fraction

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "claire_amd", "csrc",
                      "gather_device.hpp")

MAIN = r"""
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <initializer_list>
#define __device__
#define __forceinline__ inline
%s
static uint64_t state = 1;
static uint64_t next() { state ^= state << 13; state ^= state >> 7; state ^= state << 17; return state; }
static long bad = 0;
static void check(double x) {
    const double want = x / kTwoPi, got = over_2pi(x);
    if (!(got == want || (std::isnan(got) && std::isnan(want)))) ++bad;
}
int main() {
    // every FP32 mantissa in one binade: products and corrections of other binades,
    // signs and FP32 subnormals are those times a power of two
    for (uint32_t m = 0; m < (1u << 23); ++m) check(1.0 + m * 0x1p-23);
    // arguments of RK4's last stage, x - s6*f with both in FP32
    for (int i = 0; i < 4000000; ++i) {
        const float x = static_cast<float>((next() >> 11) * 0x1p-53 * kTwoPi);
        const float f = static_cast<float>(((next() >> 11) * 0x1p-53 - 0.5) * 40.0);
        check(x - (1.0 / 24.0) * static_cast<double>(f));
    }
    // any double that neither over- nor underflows on the way
    for (int i = 0; i < 4000000; ++i)
        check(std::ldexp(1.0 + (next() >> 12) * 0x1p-52, static_cast<int>(next() %% 1600) - 800) * (next() & 1 ? 1 : -1));
    for (double x : {0.0, -0.0, static_cast<double>(INFINITY), -static_cast<double>(INFINITY), static_cast<double>(NAN),
                     0x1p-149, -0x1p-149, 0x1.fffffep127})
        check(x);
    std::printf("%%ld\n", bad);
    return 0;
}
"""


def test_equals_the_division(tmp_path):
    with open(HEADER) as f:
        text = re.search(r"constexpr double kTwoPi = .*?\n}\n", f.read(), flags=re.S).group(0)
    assert "over_2pi" in text
    (tmp_path / "t.cpp").write_text(MAIN % text)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-o", tmp_path / "t", tmp_path / "t.cpp"], check=True)
    r = subprocess.run([tmp_path / "t"], capture_output=True, text=True, timeout=100, check=True)
    assert r.stdout.strip() == "0"


def test_the_quotient_is_faithful():
    """What the proof in the header needs: the reciprocal rounded to nearest, and the
    first quotient less than one unit in the last place off (half from its rounding,
    the rest from the reciprocal's error)."""
    b = 2.0 * 3.14159265358979323846
    inv = 1.0 / b
    error = abs(Fraction(inv) * Fraction(b) - 1)
    assert Fraction(1, 2) + error * 2 ** 53 < 1
