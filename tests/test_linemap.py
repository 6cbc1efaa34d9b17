"""The line offsets of the kernels (jt_linemap.hpp), compiled for the host:
every offset against the language's own division, over the group sizes and
line counts that plans accept (totals up to 2^40 points)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <initializer_list>
#include <random>
#include "jt_linemap.hpp"
static long long bad = 0, n = 0, split = 0;
// lines lines in groups of d, at (l % d)*3 + (l / d)*s1
static void check(int64_t lines, int64_t d, std::initializer_list<int64_t> ls) {
    const int64_t s1 = 5 * d + 1;
    int64_t first = 0;
    jt::exact_maps(jt::LineMap(lines, d, 3, s1, 7), [&](int64_t off, const jt::LineMap& m) {
        for (int64_t l : ls) {
            if (l < first || l >= first + m.nlines) continue;
            n++;
            const int64_t got = off + m.base(l - first), want = l % d * 3 + l / d * s1;
            if ((got != want || m.es != 7) && bad++ < 5)
                std::printf("line %lld of %lld in groups of %lld: %lld, not %lld\n", (long long)l, (long long)lines,
                            (long long)d, (long long)got, (long long)want);
        }
        first += m.nlines;
        split += m.nlines != lines;
    });
    if (first != lines && bad++ < 5) std::printf("%lld lines, not %lld\n", (long long)first, (long long)lines);
}
int main() {
    std::mt19937_64 rng(20110602);
    auto edges = [&](int64_t d, int64_t k) {
        for (int64_t m : {d * k, d * k - d / 2})  // a partly filled last group too
            for (int64_t g : {int64_t(0), int64_t(1), k / 2, k - 1})
                check(m, d, {g * d, g * d + 1, g * d + d / 2, g * d + d - 1, (int64_t)(rng() % (uint64_t)m)});
    };
    for (int64_t d = 1; d <= 2048; d++)
        for (int64_t k : {1, 2, 3, 7, 1000, 65537}) edges(d, k);
    // a few lines of slices, where the multiplied quotient alone is too coarse
    for (int64_t d : {INT64_C(3087000000), INT64_C(3099363912), INT64_C(4294967291), INT64_C(6442450944),
                      (INT64_C(1) << 38) - 1, INT64_C(1) << 38})
        for (int64_t k : {2, 3, 4}) edges(d, k);
    if (!split) {
        std::printf("no map was split\n");
        return 1;
    }
    for (int i = 0; i < 4000; i++) {
        const int64_t d = 2 + (int64_t)(rng() >> (24 + rng() % 38));
        edges(d, 1 + (int64_t)(rng() % (uint64_t)((INT64_C(1) << 41) / d + 1)));
    }
    std::printf("%lld checked, %lld wrong\n", n, bad);
    return bad != 0;
}
"""


def test_line_offsets(tmp_path):
    cxx = shutil.which("g++") or shutil.which("clang++") or shutil.which("amdclang++")
    if not cxx:
        pytest.skip("no host C++ compiler")
    src, exe = tmp_path / "linemap.cpp", tmp_path / "linemap"
    src.write_text(PROGRAM)
    subprocess.run([cxx, "-O2", "-std=c++17", "-I", os.path.join(ROOT, "jtransforms_amd", "csrc"), str(src), "-o",
                    str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
