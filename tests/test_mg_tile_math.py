"""The arithmetic helpers of the one-launch V-cycle legs (csrc/pm_mg_tile.h), compiled for the
CPU from the header's own text: div6 against the IEEE division for every mantissa, at the limits
of its exponent range and past them; div_c against the integer division over its whole range."""

from __future__ import annotations

import re
import shutil
import subprocess

import pytest

from conftest import PKG_DIR

_MAIN = r"""
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <initializer_list>
#define __device__
#define __forceinline__ inline
static inline uint32_t __umul24(uint32_t a, uint32_t b) { return (a & 0xffffffu) * (b & 0xffffffu); }
@FUNCTIONS@
static uint32_t bits(float x) { uint32_t u; std::memcpy(&u, &x, 4); return u; }
static float from(uint32_t u) { float x; std::memcpy(&x, &u, 4); return x; }
static long bad = 0;
// four values at once, as the kernels batch them
static void check(const float (&x)[4]) {
  float q[4] = {x[0], x[1], x[2], x[3]};
  div6<4>(q);
  for (int m = 0; m < 4; ++m) {
    volatile float six = 6.0f;
    const float want = x[m] / six;
    if (bits(q[m]) != bits(want) && !(want != want && q[m] != q[m])) {
      if (bad++ < 5) std::printf("div6(%a) = %a, not %a\n", x[m], q[m], want);
    }
  }
}
template <int D> static void check_div_c() {
  for (int t = 0; t < (1 << 14); ++t)
    if (div_c<D>(t) != t / D && bad++ < 5) std::printf("div_c<%d>(%d)\n", D, t);
  if constexpr (D < 63) check_div_c<D + 1>();
}
int main() {
  // every mantissa, at exponents in the middle and at both ends of the range that takes no division
  for (int e : {127, 127 - 100, 127 + 99})
    for (uint32_t m = 0; m < (1u << 23); m += 2) {
      const uint32_t u = (static_cast<uint32_t>(e) << 23) | m;
      check({from(u), from(u | 1u), -from(u), -from(u | 1u)});
    }
  // every exponent, subnormals, zeros, infinities and NaN; each beside values of the plain range
  for (uint32_t e = 0; e < 256; ++e)
    for (uint32_t m : {0u, 1u, 2u, 3u, 5u, 0x2aaaaau, 0x400000u, 0x555555u, 0x7ffffeu, 0x7fffffu}) {
      const float x = from((e << 23) | m);
      check({x, -x, x, -x});
      check({1.0f, x, 0.0f, -3.0f});
      check({-0.0f, 7.0f, 0x1p100f, -x});
    }
  check_div_c<5>();
  std::printf("%ld wrong\n", bad);
  return bad != 0;
}
"""


def _function(text: str, name: str) -> str:
    """The template function `name` of the header, up to its closing brace in column 0."""
    m = re.search(r"^template <[^>]*>\n__device__ __forceinline__ \w+ " + name + r"\(.*?^}\n", text,
                  re.S | re.M)
    assert m, name
    return m.group(0)


def test_tile_arithmetic_equals_division(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if not cxx:
        pytest.skip("no host C++ compiler")
    text = (PKG_DIR / "csrc" / "pm_mg_tile.h").read_text()
    src = tmp_path / "tile_math.cpp"
    src.write_text(_MAIN.replace("@FUNCTIONS@", _function(text, "div6") + _function(text, "div_c")))
    exe = tmp_path / "tile_math"
    # the device library's own rule: no contraction
    subprocess.run([cxx, "-std=c++17", "-O2", "-ffp-contract=off", "-w", "-o", str(exe), str(src),
                    "-lm"], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    assert run.returncode == 0, run.stdout
