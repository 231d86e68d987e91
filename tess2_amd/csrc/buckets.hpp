// buckets.hpp -- the bucket hash's geometry: the bucket of a position, and how
// near the positions of a bucket can be (includable without the HIP headers).
#pragma once

#include <cmath>

namespace t2 {

// uniform bucket hash of the particles: bucket (i,j,k) holds the particles
// with floor((x - lo) * inv) == (i,j,k), clamped to the grid of dims buckets
struct HashP {
    float lo[3];
    float inv;      // 1 / cell
    float cell;
    int dims[3];
    float slack;    // cells a position can lie outside its bucket (bucket_slack)
};

__host__ __device__ __forceinline__ int bucket_index(float q, float lo, float inv, int dim)
{
    const int i = (int)floorf((q - lo) * inv);
    return i < 0 ? 0 : (i >= dim ? dim - 1 : i);
}

// The float arithmetic of bucket_index and bucket_gap is off by a few ulp of
// the bucket number: a position lies up to that much outside its bucket.
__host__ __device__ __forceinline__ float bucket_slack(int most_buckets)
{
    return 0.001f + 4.8e-7f * (float)most_buckets;
}

// Distance on one axis from [a, b] (relative to the hash's origin) to the
// positions of bucket i: no position of the bucket is nearer by more than a
// few ulp of the distance.  Relative to the origin, since a difference of
// absolute edges is off by an ulp of the coordinate, more than the slack where the
// box lies far from zero (6e-5 at 1000; the slack of 200,000 particles in a
// unit box is 1.7e-5).
__host__ __device__ __forceinline__ float bucket_gap(float a, float b, int i, const HashP &h)
{
    const float left = (float)i * h.cell, right = left + h.cell;
    return fmaxf(0.0f, fmaxf(left - b, a - right) - h.slack * h.cell);
}

// Squared distance from the box [lo, hi] (relative to the origin, in buckets c0
// to c1) to the buckets beyond shell r, infinite when there are none: on some
// axis such a bucket is past the shell, on the others it is at least as far as
// the hash.  The shell alone (r buckets) says little about a box outside the
// hash: a point 300 buckets off meets 300 shells before the first bound passes
// its nearest site (60,000 particles in a pencil of 1 : 100 : 100 on 33^3: 319
// -> 7.3 ms; 276 with two particles a bucket).  Inside the hash the shell's bound
// costs less and ends as soon (64,000 on 129^3 132 us, with this bound 135).
__host__ __device__ __forceinline__ float beyond_shell2(int r, const int *c0, const int *c1,
                                                        const float *lo, const float *hi,
                                                        const HashP &h)
{
    float past[3], off[3];
    for (int a = 0; a < 3; ++a) {
        float g = INFINITY;
        if (c0[a] - r > 0) g = bucket_gap(lo[a], hi[a], c0[a] - r - 1, h);
        if (c1[a] + r < h.dims[a] - 1) g = fminf(g, bucket_gap(lo[a], hi[a], c1[a] + r + 1, h));
        past[a] = g * g;
        const float d = fmaxf(lo[a] - (float)h.dims[a] * h.cell, -hi[a]) - h.slack * h.cell;
        off[a] = d > 0.0f ? d * d : 0.0f;
    }
    return fminf(past[0] + off[1] + off[2],
                 fminf(off[0] + past[1] + off[2], off[0] + off[1] + past[2]));
}

}  // namespace t2
