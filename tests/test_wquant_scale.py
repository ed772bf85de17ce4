"""The group formats' scale arithmetic of the weight quantizer (csrc/mq_wquant.hip), on the CPU: the
division-free quotient (div_limit of csrc/mq_rotate.h) rounded to fp16 equals the IEEE quotient rounded to
fp16 for every non-negative float, +inf and NaN included, for L = 15 (uint4 range) and 7 (int4 absmax)."""
import os
import shutil
import subprocess

import pytest

C_SRC = r"""
#include <math.h>
#include <immintrin.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

static float f_of(uint32_t b) { float x; memcpy(&x, &b, 4); return x; }
static float div_limit(float am, float L) {
    const float c = 1.0f / L, q0 = am * c, e = fmaf(-q0, L, am), q1 = fmaf(e, c, q0);
    return isinf(am) ? am : q1;
}
/* to fp16, round to nearest even; every NaN as one */
static int half_of(float x) { return isnan(x) ? -1 : (int)_cvtss_sh(x, _MM_FROUND_TO_NEAREST_INT); }

int main(void) {
    const float Ls[2] = {15.0f, 7.0f};
    for (int li = 0; li < 2; ++li) {
        unsigned long long bad = 0;
#pragma omp parallel for reduction(+ : bad) schedule(static, 1 << 20)
        for (long long b = 0; b <= 0x7fc00000LL; ++b) {
            const float am = f_of((uint32_t)b);
            if (half_of(am / Ls[li]) != half_of(div_limit(am, Ls[li]))) ++bad;
        }
        printf("fp16 scale L=%g mismatches %llu\n", Ls[li], bad);
        if (bad) return 1;
    }
    return 0;
}
"""


@pytest.mark.skipif(shutil.which("gcc") is None, reason="needs gcc")
def test_fp16_scales_exhaustive(tmp_path):
    src, exe = tmp_path / "scale.c", tmp_path / "scale"
    src.write_text(C_SRC)
    subprocess.run(["gcc", "-O2", "-mfma", "-mf16c", "-ffp-contract=off", "-fopenmp", str(src), "-o", str(exe), "-lm"],
                   check=True)
    env = dict(os.environ)
    env.setdefault("OMP_NUM_THREADS", str(os.cpu_count() or 1))
    res = subprocess.run([str(exe)], capture_output=True, text=True, env=env, timeout=900)
    assert res.returncode == 0, res.stdout + res.stderr
    assert res.stdout.count("mismatches 0") == 2
