// owner_tiles.hpp -- the tile of grid points that a wave of the exact
// assignment searches for at once (host code, includable without the HIP headers).
#pragma once

#include <algorithm>

namespace t2 {

// 2^bits[a] points on axis a; 64 / points lanes per point
struct OwnerTile {
    int bits[3];
    int points;   // 64, 8 or 1
};

// particles that a wave meets, at one a bucket: the tile's box, and the
// buckets about it that the nearest sites of its points can lie in, at most all
inline double tile_meets(const OwnerTile &t, const double step[3], const int buckets[3])
{
    double m = 1.0, all = 1.0;
    for (int a = 0; a < 3; ++a) {
        m *= ((1 << t.bits[a]) - 1) * step[a] + 2.5;
        all *= buckets[a];
    }
    return std::min(m, all);
}

// dims: grid points; step: their distance in buckets; buckets: of the hash.
//
// A wave on 64 points loads every particle once for all of them, but where the
// grid is coarser than the particles it meets all particles of its box one
// after the other: 14,500 for 200,000 particles on 9^3.  On 8 points or one, its
// lanes share the particles of each run of buckets and the boxes are smaller,
// at more waves.  The time in us is taken as the chain of one wave plus the
// issue of all waves, each with a part per particle met; the constants are a
// fit of 1000 to 200,000 uniform particles on 2^3 to 129^3 with 64, 8 and 1
// points a wave (200,000 on 9^3 1808, 96 and 17 us, on 33^3 108, 35 and 70, on
// 65^3 69, 111 and 441; a lane per point took 57, 93 and 111).  The edges double
// on the axis where that keeps the box shortest (200,000 on 300 x 300 x 9: 4 x
// 4 x 4 points 205 us, a lane per point 145, 8 x 8 x 1 points 87).
// Particles in a small part of the grid are few to meet (1,000 in a hundredth of
// its edge on 257^3: 8.2 ms with 64 points, 30 with 8, 88 with one).
inline OwnerTile owner_tile(const int dims[3], const double step[3], const int buckets[3])
{
    static const struct { int points; double chain, met, wave, issue; } fit[3] = {
        {64, 20.0, 0.14, 1.5e-3, 5e-5}, {8, 17.0, 0.07, 0.5e-3, 5e-5}, {1, 15.0, 0.0, 1.8e-3, 0.0}};
    OwnerTile best{}, t{};
    double least = 0.0;
    for (int k = 2; k >= 0; --k) {
        t.points = fit[k].points;
        while ((1 << (t.bits[0] + t.bits[1] + t.bits[2])) < t.points) {
            int at = -1;
            double shortest = 0.0;
            for (int pass = 0; pass < 2 && at < 0; ++pass)   // no longer than the grid first
                for (int a = 0; a < 3; ++a) {
                    const double edge = (double)(2 << t.bits[a]) * step[a];
                    if ((pass || (1 << t.bits[a]) < dims[a]) && (at < 0 || edge < shortest)) {
                        at = a;
                        shortest = edge;
                    }
                }
            ++t.bits[at];
        }
        double waves = 1.0;
        for (int a = 0; a < 3; ++a) waves *= ((dims[a] - 1) >> t.bits[a]) + 1;
        const double m = tile_meets(t, step, buckets);
        const double us = fit[k].chain + fit[k].met * m + waves * (fit[k].wave + fit[k].issue * m);
        // at most 400 particles in a row, as many as were measured (a clustered
        // block holds many times the mean in some tiles), unless there are no
        // more; tiles are counted in an int
        const bool few = m * fit[k].points / 64.0 <= 400.0 ||
                         m >= (double)buckets[0] * buckets[1] * buckets[2];
        if (k == 2 || (us < least && few) || waves * fit[k].points >= 2e9) {
            least = us;
            best = t;
        }
    }
    return best;
}

}  // namespace t2
