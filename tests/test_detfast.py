"""The short double sequences of detfast.h give the float results of the full
ones (detmath.h, philox.h) bit for bit: compiled for the host with the same
fused operations (its reciprocal seeds are of the same accuracy) and compared
over the arguments' whole range, with the range ends and the zeros."""

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <math.h>
#include <stdio.h>
#include "detfast.h"
static uint64_t s = 88172645463325252ull;
static uint32_t rnd() { s ^= s << 13; s ^= s >> 7; s ^= s << 17; return (uint32_t)(s >> 16); }
static bool same(float a, float b) { return gsbn_fbits(a) == gsbn_fbits(b) || (a != a && b != b); }
static float full24(uint32_t k1, uint32_t k2) {
  const double u1 = (double)(k1 + 1u) / 16777216.0, u2 = (double)k2 / 16777216.0;
  return (float)(gsbn_sqrt(-2.0 * gsbn_log(u1)) * gsbn_cos2pi(u2));
}
int main() {
  long bad = 0;
  double far = 0;
  for (long i = 0; i < 1000000; ++i) {
    uint32_t b = rnd();
    if (i < 64) b = 0x00800000u - 32 + (uint32_t)i;          /* smallest normal float */
    else if (i < 128) b = 0x3f800000u - 32 + (uint32_t)(i - 64); /* 1 */
    else if (i < 132) b = (i & 1 ? 0x7f800000u : 0u) | (i & 2 ? 0x80000000u : 0u); /* 0, inf */
    const float x = gsbn_bitsf(b);
    bad += !same(gsbn_logf_guarded(x), (float)gsbn_log((double)x));
    bad += !same(gsbn_expf_guarded(x), (float)gsbn_exp((double)x));
    const float e = (float)rnd() * (194.0f / 4294967296.0f) - 105.0f;
    bad += !same(gsbn_expf_guarded(e), (float)gsbn_exp((double)e));
    bad += !same((float)gsbn_exp_cold(e), (float)gsbn_exp((double)e));
    uint32_t k1 = rnd() >> 8, k2 = rnd() >> 8;
    if (i < 64) k1 = 0xffffffu - (uint32_t)i;                 /* u1 = 1 and below */
    if (i >= 64 && i < 128) k2 = 0x400000u - 32 + (uint32_t)(i - 64); /* cos = 0 */
    if (i >= 128 && i < 192) k2 = 0x800000u - 32 + (uint32_t)(i - 128);
    if (i >= 192 && i < 224) k2 = (uint32_t)(i - 192);
    bad += !same(gsbn_normal24_guarded(k1, k2), full24(k1, k2));
    bad += !same(gsbn_normal24_cold(k1, k2), full24(k1, k2));
    if (e >= -87.0f && e <= 88.0f) far = fmax(far, fabs(gsbn_exp_short(e) / gsbn_exp(e) - 1));
    if (b > 0x00800000u && b < 0x7f800000u && x != 1.0f)
      far = fmax(far, fabs(gsbn_log_short(x) / gsbn_log(x) - 1));
  }
  printf("%ld %g\n", bad, far);
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
def test_short_forms_round_to_the_full_results(tmp_path):
    src = tmp_path / "t.cpp"
    src.write_text(SOURCE)
    exe = str(tmp_path / "t")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-I",
                    os.path.join(ROOT, "gsbn_amd", "csrc"), "-o", exe, str(src)], check=True)
    bad, far = subprocess.run([exe], check=True, stdout=subprocess.PIPE, text=True).stdout.split()
    assert int(bad) == 0
    # the guard is 2048 units of 2^-53 to 2^-52; the distance has to stay ten times below
    assert float(far) < 2048 * 2.0 ** -53 / 10
