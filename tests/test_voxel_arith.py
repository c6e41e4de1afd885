"""The exact divisions of the voxel kernels (cookiedough_amd/csrc/k_voxel.hip),
swept on the host with the reciprocal rounded to nearest and one ulp off either
way, as v_rcp_f32 may give it:

- ls_row: floor(((255 - h) << 16) / (fish * (step + 1))) for every height, step
  and fish of 4 to 257 (256 times a cosine of the ray's angle);
- udiv24 with a span's length: floor(65536 / length), and with ts_height's
  numerator and divisor: the tunnelscape's height as the reference forms it in
  FP32 (code/tunnelscape.cpp:75-84)."""
import shutil
import subprocess

import pytest

SRC = r"""
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>
static float ulp(float x, int d) { uint32_t u; memcpy(&u, &x, 4); u += (uint32_t)d; memcpy(&x, &u, 4); return x; }
#ifndef HALF
#define HALF 0.5f
#endif
static uint32_t udiv24(uint32_t num, uint32_t den, float rcp)
{
    const float qf = fmaf((float)num, rcp, -HALF);
    const uint32_t q = (uint32_t)(int32_t)qf;
    return q + (num - ((q & 0xffffffu) * (den & 0xffffffu)) >= den ? 1u : 0u);
}
int main(void)
{
    long bad[3] = {0, 0, 0}, n[3] = {0, 0, 0};
    for (int fish = 4; fish <= 257; ++fish)
        for (int s = 1; s <= 512; ++s) {
            const float den = (float)fish * (float)s, r = 1.0f / den;
            for (int d = -1; d <= 1; ++d) {
                const float rcp = ulp(r, d);
                for (int h = 0; h < 256; ++h) {
                    const float num = fmaf((float)h, -65536.f, 16711680.f);
                    const float q = truncf(fmaf(num, rcp, -HALF));
                    const uint32_t got = (uint32_t)(int32_t)q + (fmaf(-q, den, num) >= den ? 1u : 0u);
                    bad[0] += got != ((uint32_t)(255 - h) << 16) / (uint32_t)(fish * s);
                    ++n[0];
                }
            }
        }
    for (uint32_t len = 1; len < (1u << 18); ++len)
        for (int d = -1; d <= 1; ++d, ++n[1])
            bad[1] += udiv24(65536u, len, ulp(1.0f / (float)len, d)) != 65536u / len;
    for (uint32_t h = 0; h <= 159; ++h)
        for (uint32_t s = 1; s <= 512; ++s) {
            const float wide = (float)((159u - h) << 8) / 0.28125f;
            const uint32_t want = (uint32_t)(int32_t)wide / s;
            for (int d = -1; d <= 1; ++d, ++n[2])
                bad[2] += udiv24((159u - h) << 13, 9u * s, ulp(1.0f / (float)(9u * s), d)) != want;
        }
    for (int k = 0; k < 3; ++k) printf("%ld %ld ", bad[k], n[k]);
    return 0;
}
"""


def _run(tmp_path, *flags):
    cc = shutil.which("gcc") or shutil.which("cc")
    if cc is None:
        pytest.skip("no C compiler")
    src, exe = tmp_path / "voxel.c", tmp_path / "voxel"
    src.write_text(SRC)
    subprocess.run([cc, "-O2", "-ffp-contract=off", *flags, "-o", str(exe), str(src), "-lm"], check=True)
    v = [int(x) for x in subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()]
    return v[0::2], v[1::2]


def test_divisions(tmp_path):
    bad, n = _run(tmp_path)
    assert n == [254 * 512 * 3 * 256, ((1 << 18) - 1) * 3, 160 * 512 * 3]
    assert bad == [0, 0, 0]


def test_without_the_half(tmp_path):
    """an estimate that is not lowered by a half overshoots"""
    bad, _ = _run(tmp_path, "-DHALF=0.0f")
    assert bad[0] > 0, bad
