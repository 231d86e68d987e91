"""The bucket hash's distance bound (tess2_amd/csrc/buckets.hpp) on the host:
no position of a bucket is nearer to an interval than bucket_gap says, wherever
the box lies and however many buckets an axis has.  A bound above the true
distance would let the exact assignment's search skip the bucket of the nearest
site.  The true distance is taken in long double; positions are random, with
those next to bucket edges on either side, intervals of up to a few buckets
around them.  The search compares squares widened by 2e-6 (FP32: 1e-4)."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "tess2_amd", "csrc")

HARNESS = r"""
#define __host__
#define __device__
#define __forceinline__ inline
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <algorithm>
#include "buckets.hpp"
using namespace t2;

int main()
{
    std::mt19937_64 g(12345);
    auto u = [&] { return std::uniform_real_distribution<double>(0.0, 1.0)(g); };
    long bad = 0, cases = 0, tight = 0;
    const double offsets[] = {0.0, 1.0, -3.5, 1000.0, 20000.0, -60000.0};
    const int dims[] = {1, 7, 59, 640, 9000, 300000, 16000000};
    for (double off : offsets)
        for (int dim : dims)
            for (double extent : {1.0, 250.0}) {
                const float lo = (float)off, hi = (float)(off + extent);
                if (!(hi > lo)) continue;
                HashP h{};
                // as staging makes it: cell from the box, dims from the cell
                const double cell = ((double)hi - lo) / (dim - 0.5);
                h.lo[0] = lo;
                h.inv = (float)(1.0 / cell);
                h.cell = (float)cell;
                h.dims[0] = (int)((hi - lo) / cell) + 1;
                h.slack = bucket_slack(h.dims[0]);
                for (int k = 0; k < 40000; ++k) {
                    // a particle, half of them within a few ulp of an edge
                    float p = (float)(lo + u() * ((double)hi - lo));
                    if (k & 1) {
                        const int i = (int)(u() * h.dims[0]);
                        p = (float)(lo + (double)i * cell);
                        for (int n = (int)(u() * 4); n > 0; --n)
                            p = std::nextafterf(p, u() < 0.5 ? -1e30f : 1e30f);
                    }
                    p = std::min(std::max(p, lo), hi);
                    const int b = bucket_index(p, lo, h.inv, h.dims[0]);
                    // an interval near it, touching it, around it or far away
                    const double s = (k & 2) ? 4.0 * cell : 3.0 * extent;
                    float x0 = (float)(p + (u() - 0.5) * s);
                    float x1 = (k & 4) ? x0 : (float)(x0 + u() * 2.0 * cell);
                    if (k % 16 == 5) x0 = x1 = p;
                    if (x1 < x0) std::swap(x0, x1);
                    const long double d =
                        std::max(0.0L, std::max((long double)x0 - p, (long double)p - x1));
                    const float gap = bucket_gap(x0 - lo, x1 - lo, b, h);
                    ++cases;
                    if ((long double)gap * gap > d * d * (1.0L + 1e-6L)) {
                        if (++bad < 10)
                            std::printf("off %g dims %d: p %.9g [%.9g, %.9g] bucket %d gap %.9g "
                                        "distance %.9Lg\n", off, h.dims[0], p, x0, x1, b, gap, d);
                    }
                    if (gap > 0.0f) ++tight;
                }
            }
    std::printf("%ld cases, %ld with a gap, %ld bad\n", cases, tight, bad);
    return bad || tight < cases / 4;
}
"""

SHELLS = r"""
int main()
{
    std::mt19937_64 g(777);
    auto u = [&] { return std::uniform_real_distribution<double>(0.0, 1.0)(g); };
    long bad = 0, bounded = 0, far = 0;
    for (int k = 0; k < 400; ++k) {
        // boxes of unlike sides, far from zero too
        const double off = k % 3 == 0 ? 0.0 : (k % 3 == 1 ? 5000.0 : -300.0);
        double ext[3], cell = 1.0;
        for (int a = 0; a < 3; ++a) ext[a] = std::pow(10.0, 2.0 * u());
        cell = std::cbrt(ext[0] * ext[1] * ext[2] / (10.0 + 3000.0 * u()));
        HashP h{};
        h.cell = (float)cell;
        h.inv = (float)(1.0 / cell);
        float top[3];
        int most = 0;
        for (int a = 0; a < 3; ++a) {
            h.lo[a] = (float)off;
            top[a] = (float)(off + ext[a]);
            h.dims[a] = (int)((top[a] - h.lo[a]) / cell) + 1;
            most = std::max(most, h.dims[a]);
        }
        h.slack = bucket_slack(most);
        for (int q = 0; q < 60; ++q) {
            // a box inside, across the sides or far outside
            float lo[3], hi[3];
            int c0[3], c1[3];
            const double s = q % 3 == 0 ? 0.0 : (q % 3 == 1 ? 0.5 : 40.0);
            for (int a = 0; a < 3; ++a) {
                lo[a] = (float)(off + (u() * (1.0 + 2.0 * s) - s) * ext[a]);
                hi[a] = q % 2 ? lo[a] : (float)(lo[a] + 3.0 * u() * cell);
                c0[a] = bucket_index(lo[a], h.lo[a], h.inv, h.dims[a]);
                c1[a] = bucket_index(hi[a], h.lo[a], h.inv, h.dims[a]);
            }
            float rl[3], rh[3];
            for (int a = 0; a < 3; ++a) {
                rl[a] = lo[a] - h.lo[a];
                rh[a] = hi[a] - h.lo[a];
            }
            for (int r = 0; r < 12; ++r) {
                const float b2 = beyond_shell2(r, c0, c1, rl, rh, h);
                if (b2 > 0.0f) ++bounded;
                if (b2 > (float)((r + 20) * cell) * (float)((r + 20) * cell)) ++far;
                for (int n = 0; n < 60; ++n) {
                    long double d2 = 0.0L;
                    bool out = false;
                    for (int a = 0; a < 3; ++a) {
                        float p = (float)(h.lo[a] + u() * ((double)top[a] - h.lo[a]));
                        if (n % 4 == 0) {   // next to the edges just past the shell
                            const int i = n % 8 ? c0[a] - r : c1[a] + r + 1;
                            p = std::nextafterf((float)(h.lo[a] + (double)i * cell),
                                                n % 8 ? -1e30f : 1e30f);
                        }
                        p = std::min(std::max(p, h.lo[a]), top[a]);
                        const int b = bucket_index(p, h.lo[a], h.inv, h.dims[a]);
                        out |= b < c0[a] - r || b > c1[a] + r;
                        const long double d = std::max(
                            0.0L, std::max((long double)lo[a] - p, (long double)p - hi[a]));
                        d2 += d * d;
                    }
                    if (out && (long double)b2 > d2 * (1.0L + 2e-6L)) ++bad;
                }
            }
        }
    }
    std::printf("%ld bounds, %ld of boxes far outside, %ld bad\n", bounded, far, bad);
    return bad || bounded < 1000 || far < 1000;
}
"""


def _run(tmp_path, name, code):
    src = tmp_path / (name + ".cpp")
    src.write_text(code)
    exe = tmp_path / name
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-I", CSRC, str(src),
                           "-o", str(exe)])
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ missing")
def test_bound_beyond_a_shell(tmp_path):
    """No position outside the shell is nearer than beyond_shell2 says, and
    boxes far outside the hash are not left to the shell's number alone."""
    _run(tmp_path, "shell", HARNESS[:HARNESS.index("int main")] + SHELLS)


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ missing")
def test_gap_is_a_lower_bound(tmp_path):
    _run(tmp_path, "gap", HARNESS)
