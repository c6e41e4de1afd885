"""The in-place blur's chunks of steps (cookiedough_amd/csrc/ckd_b07_scan.h, the
loops of b07_scan_line): over every line length, edge and chunk size, whole
lines and lines that stop before their last pixel, the chunks take each step
once, the middle run's need no test of the edges, and the step that saves a
stopped line's state is not among them."""
import shutil
import subprocess

import pytest

from conftest import ROOT

SRC = r"""
#include <cstdio>
#include "ckd_b07_scan.h"
#ifdef OLD
#define LAST(len, n) (len - 17)
#else
#define LAST(len, n) ckd::b07_scan_last(len, n)
#endif
int main()
{
    long bad = 0, middle = 0;
    const int sizes[] = {4, 6, 8, 10, 12, 16};
    for (int k : sizes)
        for (int m = k; m <= 40; m += m < 18 ? 1 : 11)
            for (int e = m - 1; e <= m; ++e)
                for (int len = e + m + 1; len < e + m + 120; ++len)
                    for (int split = 0; split < 2; ++split) {
                        const int nSteps = split ? len - 1 : len + e, last = LAST(len, nSteps);
                        int p = 0, next = 0;
                        auto chunk = [&](bool edge) {
                            bad += p != next;
                            next = p + k;
                            if (edge) return;
                            ++middle;
                            // back > 0, every lane's pixel before the last one, output
                            // with the full divisor, no step past the end
                            bad += !(p - e - m > 0 && p + 15 < len - 1 && p + k - 1 - e < len - e && p + k <= nSteps);
                            bad += split && p + k - 1 >= nSteps - 1;
                        };
                        for (; p <= e + m && p < nSteps; p += k) chunk(true);
                        for (; p <= last; p += k) chunk(false);
                        for (; p < nSteps; p += k) chunk(true);
                        bad += next < nSteps;
                    }
    std::printf("%ld %ld\n", bad, middle);
}
"""


def _run(tmp_path, *flags):
    cc = shutil.which("g++")
    if cc is None:
        pytest.skip("no C++ compiler")
    src, exe = tmp_path / "chunks.cpp", tmp_path / "chunks"
    src.write_text(SRC)
    subprocess.run([cc, "-std=c++17", "-O2", f"-I{ROOT / 'cookiedough_amd' / 'csrc'}", *flags, "-o", str(exe), str(src)],
                   check=True)
    return [int(v) for v in subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()]


def test_chunks(tmp_path):
    bad, middle = _run(tmp_path)
    assert bad == 0 and middle > 10000


def test_whole_lines_limit_misses_a_stopped_line(tmp_path):
    """the limit of whole lines, taken for both"""
    assert _run(tmp_path, "-DOLD")[0] > 0
