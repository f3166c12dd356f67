"""The bounds that detfast.h states, with seeds as far off as it allows (2^-24
relative, both ways, where the host's own are nearer): every short form within
2e-14 of the full one, and no float result that differs."""

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
int main() {
  long bad = 0;
  double flog = 0, fnorm = 0, fexp = 0, frcp = 0, frsq = 0;
  for (long i = 0; i < 2000000; ++i) {
    uint32_t b = 0x00800000u + rnd() % (0x7f800000u - 0x00800000u);
    if (i < 4096) b = 0x3f800000u - 2048 + (uint32_t)i; /* about 1 */
    const float x = gsbn_bitsf(b);
    bad += !same(gsbn_logf_guarded(x), (float)gsbn_log((double)x));
    if (x != 1.0f) flog = fmax(flog, fabs(gsbn_log_short(x) / gsbn_log(x) - 1));
    const float e = (float)rnd() * (175.0f / 4294967296.0f) - 87.0f;
    bad += !same(gsbn_expf_guarded(e), (float)gsbn_exp((double)e));
    fexp = fmax(fexp, fabs(gsbn_exp_short(e) / gsbn_exp(e) - 1));
    uint32_t k1 = rnd() >> 8, k2 = rnd() >> 8;
    if (i < 4096) k1 = 0xfffffeu - (uint32_t)i; /* u1 just below 1 */
    else if (i < 8192) k2 = 0x400000u - 2048 + (uint32_t)(i - 4096); /* cos about 0 */
    const double u1 = (double)(k1 + 1u) / 16777216.0, u2 = (double)k2 / 16777216.0;
    const double z = gsbn_sqrt(-2.0 * gsbn_log(u1)) * gsbn_cos2pi(u2);
    bad += !same(gsbn_normal24_guarded(k1, k2), (float)z);
    if (k1 != 0xffffffu && z != 0) fnorm = fmax(fnorm, fabs(gsbn_normal24_short(k1, k2) / z - 1));
    /* one Newton step on the seeds, as the short forms take it */
    const double d = 1.0 + (double)(b & 0x7fffff) / 8388608.0;
    double y = gsbn_rcp_seed(d);
    y = fma(y, fma(-d, y, 1.0), y);
    frcp = fmax(frcp, fabs(y * d - 1));
    const double q = gsbn_rsq_seed(d), g = d * q;
    frsq = fmax(frsq, fabs(fma(0.5 * g, fma(-g, q, 1.0), g) / sqrt(d) - 1));
  }
  printf("%ld %g %g %g %g %g\n", bad, flog, fnorm, fexp, frcp, frsq);
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
@pytest.mark.parametrize("error", ["5.9604644775390625e-08", "-5.9604644775390625e-08"])
def test_bounds_with_seeds_of_24_bits(tmp_path, error):
    src = tmp_path / "t.cpp"
    src.write_text(SOURCE)
    exe = str(tmp_path / "t")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-DGSBN_SEED_ERROR=" + error,
                    "-I", os.path.join(ROOT, "gsbn_amd", "csrc"), "-o", exe, str(src)], check=True)
    out = subprocess.run([exe], check=True, stdout=subprocess.PIPE, text=True).stdout.split()
    bad, (flog, fnorm, fexp, frcp, frsq) = int(out[0]), map(float, out[1:])
    assert bad == 0
    ulp = 2.0 ** -52
    assert frcp < 2.0 ** -48 + 2 * ulp and frsq < 1.5 * 2.0 ** -48 + 3 * ulp
    assert max(flog, fnorm, fexp) < 2e-14
    # the guard, 2048 units of 2^-53 of the smallest mantissa, is ten times that
    assert 2048 * 2.0 ** -53 > 10 * 2e-14
