"""The 32-bit word form of the scan line walk (csrc/scan_bits.hpp,
walk_row_bits32) against the 64-bit form, which test_scan_bits.py checks
against the point-by-point walk: every line of up to 10 points and random
lines of up to 32, on the host."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(__file__), "..", "tess2_amd", "csrc")
HARNESS = r"""
#define __host__
#define __device__
#define __forceinline__ inline
#include <cstdio>
#include <initializer_list>
#include "scan_bits.hpp"
static long bad = 0;
static void check(unsigned r, int n, int xl, int xr)
{
    int a = xl, b = xr, mn = n - 1, mx = 0, c = xl, d = xr, mn2 = n - 1, mx2 = 0;
    t2::walk_row_bits(r, n, a, b, mn, mx);
    t2::walk_row_bits32(r, n, c, d, mn2, mx2);
    if (a != c || b != d || mn != mn2 || mx != mx2) ++bad;
}
int main()
{
    for (int n = 1; n <= 10; ++n)
        for (unsigned r = 0; r < (1u << n); ++r)
            for (int xl = 0; xl < n; ++xl)
                for (int xr = 0; xr < n; ++xr) check(r, n, xl, xr);
    unsigned long long s = 88172645463325252ull;
    for (int it = 0; it < 1000000; ++it) {
        s ^= s << 13; s ^= s >> 7; s ^= s << 17;
        const int n = 11 + (int)(s % 22);
        const unsigned all = n == 32 ? ~0u : (1u << n) - 1u;
        unsigned r = (unsigned)(s >> 11) & all;
        if (it & 1) r |= (unsigned)(s >> 3) & all;
        if (it % 3 == 0) r = all & ~(r & (r >> 1));
        check(r, n, (int)((s >> 40) % n), (int)((s >> 50) % n));
    }
    for (int xl = 0; xl < 32; ++xl)
        for (int xr = 0; xr < 32; ++xr)
            for (unsigned r : {0u, ~0u, 1u, 1u << 31, 3u << 30, ~1u}) check(r, 32, xl, xr);
    printf("mismatches %ld\n", bad);
    return bad != 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_word_walk_matches_long_walk(tmp_path):
    src, exe = tmp_path / "w.cpp", tmp_path / "w"
    src.write_text(HARNESS)
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)])
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr
