"""mb_math.h's division by a known divisor (div_by) against the division
itself, bit for bit: integers over lattice units of every magnitude, divisors
with all-ones, all-zero and random mantissas among them."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]

PROGRAM = r"""
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <random>
#define __host__
#define __device__
#define __forceinline__ inline
#include "mb_math.h"
int main() {
    std::mt19937_64 r(7);
    for (long i = 0; i < 3000000; ++i) {
        uint64_t bits = ((uint64_t)(1023 - 160 + r() % 320) << 52) | (r() & ((1ull << 52) - 1));
        if (i % 5 == 0) bits |= ((1ull << 52) - 1) & ~(uint64_t)(r() % 4);
        if (i % 7 == 0) bits &= ~((1ull << 52) - 1) | (r() % 8);
        double b;
        std::memcpy(&b, &bits, 8);
        int64_t g = (int64_t)(r() >> (33 + r() % 31));
        if (r() & 1) g = -g;
        const double q = mb::div_by((double)g, b, 1.0 / b), want = (double)g / b;
        if (std::memcmp(&q, &want, 8) != 0 && !(g == 0 && q == 0.0)) {
            std::printf("%lld / %a: %a, not %a\n", (long long)g, b, q, want);
            return 1;
        }
    }
    return 0;
}
"""


def test_div_by_is_exact(tmp_path):
    # the header's scalar code alone, compiled for the host
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text("")
    src = tmp_path / "div.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "div"
    subprocess.run(["g++", "-O1", "-std=c++17", "-ffp-contract=off", f"-I{tmp_path}", f"-I{ROOT / 'mojoboost_amd' / 'csrc'}",
                    str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
