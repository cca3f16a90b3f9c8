"""The evaluator's division (div_rn of astmath.h) on the CPU: its steps as they
stand in the header, from reciprocal estimates anywhere within the bound the
header gives for the GPU's (relative error 4.7e-8), against IEEE division.
Divisors and numerators over the range the evaluator meets, with mantissas near
all ones and all zeros, numerators of 1, and the hardest quotients there are:
those next to the middle between two doubles.  For divisors within 1023 of an
all-ones mantissa, where the quotient's rounding does depend on the estimate,
it is the one that an MI355X gives: the reciprocal's rounding for all ones
itself, 0x1.000000af8p-1 (for a divisor in [1, 2)) for the others."""
import os
import re
import subprocess

import pytest

from asteroid_amd import build

PROGRAM = r"""
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
static double estimate;
static double __builtin_amdgcn_rcp(double) { return estimate; }
#define __device__
%s
static uint64_t state = 88172645463325252ull;
static uint64_t rnd() {
  state ^= state << 13;
  state ^= state >> 7;
  state ^= state << 17;
  return state * 2685821657736338717ull;
}
static double make(uint64_t mantissa, int exponent) {
  const uint64_t b = ((uint64_t)(1023 + exponent) << 52) | (mantissa & (((uint64_t)1 << 52) - 1));
  double x;
  memcpy(&x, &b, 8);
  return x;
}
static uint64_t mantissa() {
  const uint64_t r = rnd();
  switch (r & 7) {
    case 0: return ~(rnd() & 15);          // near all ones
    case 1: return rnd() & 15;             // near a power of two
    case 2: return ~(uint64_t)0 << (r >> 3) %% 52;
    default: return rnd();
  }
}
static long long pairs = 0, wrong = 0;
static void check(double n, double d) {
  static const double ends[] = {-4.7e-8, -4.6e-8, -1e-8, 0, 1e-8, 4.6e-8, 4.7e-8};
  const uint64_t r = rnd();
  const double err = (r & 1) ? ends[(r >> 1) %% 7] : ((double)(r >> 11) / 9007199254740992.0 * 2 - 1) * 4.7e-8;
  estimate = (double)((long double)1 / d * (1 + (long double)err));
  uint64_t bits;
  memcpy(&bits, &d, 8);
  const uint64_t below = ~bits & (((uint64_t)1 << 52) - 1);  // of all ones
  if (below < 1024) {
    const double e = std::ldexp(below ? 0x1.000000af8p-1 : 0x1.0000000000001p-1, -std::ilogb(d));
    estimate = d < 0 ? -e : e;
  }
  const double got = div_rn(n, d), want = n / d;
  pairs++;
  if (memcmp(&got, &want, 8)) {
    if (wrong++ < 10) printf("%%a / %%a estimate %%a: %%a, not %%a\n", n, d, estimate, got, want);
  }
}
int main() {
  for (int i = 0; i < 6000000; ++i) {
    const double d = make(mantissa(), (int)(rnd() %% 120) - 80), n = make(mantissa(), (int)(rnd() %% 120) - 80);
    check((rnd() & 1) ? n : -n, (rnd() & 1) ? d : -d);
    check(1.0, d);
    check(0.0, d);
  }
  // (n / d) 2^53 or 2^54 = M + s / d with M odd: s / d past the middle of two
  // doubles.  M is s times the inverse of -d modulo the power of two.
  for (int i = 0; i < 6000000; ++i) {
    const uint64_t D = (mantissa() & (((uint64_t)1 << 52) - 1)) | ((uint64_t)1 << 52) | 1;
    uint64_t inv = D;
    for (int k = 0; k < 5; ++k) inv *= 2 - D * inv;
    for (int p = 53; p <= 54; ++p) {
      const int64_t s = 2 * (int64_t)(rnd() %% 3) + 1, sign = (rnd() & 1) ? 1 : -1;
      const uint64_t mask = ((uint64_t)1 << p) - 1;
      uint64_t M = ((uint64_t)(-sign * s) * inv) & mask;
      if (M < (uint64_t)1 << 53) M += (uint64_t)1 << 53;
      if (M >> 54) continue;
      const unsigned __int128 top = (unsigned __int128)M * D + (__int128)(sign * s);
      if ((uint64_t)top & mask) continue;
      const unsigned __int128 N = top >> p;
      if (N >> 53) continue;
      const int e = (int)(rnd() %% 60) - 60;
      check(std::ldexp((double)(uint64_t)N, e), std::ldexp((double)D, e - (int)(rnd() %% 20)));
    }
  }
  printf("%%lld pairs, %%lld wrong\n", pairs, wrong);
  return wrong != 0;
}
"""


def _fma():
    try:
        with open("/proc/cpuinfo") as f:
            return " fma " in f.read()
    except OSError:
        return False


@pytest.mark.skipif(not _fma(), reason="no FMA unit")
def test_division_is_ieee_division(tmp_path):
    with open(os.path.join(build.CSRC, "astmath.h")) as f:
        code = re.search(r"^__device__ inline double div_rn.*?^}", f.read(), re.M | re.S).group(0)
    src, exe = tmp_path / "division.cpp", tmp_path / "division"
    src.write_text(PROGRAM % code)
    subprocess.run(["g++", "-O2", "-std=c++17", "-mfma", "-ffp-contract=off", str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0 and int(r.stdout.split()[-4]) > 2e7, r.stdout[-3000:]
