// exact.hip -- the exact-Voronoi assignment: every grid point goes to its
// nearest site (ties to the lowest particle id), located through a uniform
// bucket hash of the particles built on the device for each run.
//
// Precision modes:
//   MIXED: squared distances in float32; the FP32 decision stands only when
//          the runner-up is outside a relative window of 32 ulp around the
//          winner (each FP32 squared distance is within ~5 ulp of exact), so
//          the FP32 choice equals the exact and the FP64 choice; otherwise
//          the point is searched again in double (counted as a fallback).
//          Deposit decisions of cells near the data-bounds threshold, or with
//          ill-conditioned circumcenters, are re-made in double the same way.
//   FP64:  every distance, circumcenter and bound test in double.
#include "kernels.hpp"
#include "geom.hpp"
#include "deposit.hpp"
#include "owner_tiles.hpp"

#include <algorithm>

namespace t2 {

enum { EX_DEPOSIT = 0, EX_INCOMPLETE = 2, EX_OUTSIDE = 3, EX_DEGENERATE = 4 };

// ---------------------------------------------------------------------------
// bucket hash: count, exclusive scan, scatter (particles sorted by bucket,
// stored as float4 {x, y, z, id bits})
// ---------------------------------------------------------------------------
__device__ __forceinline__ int bucket_of(float4 p, const HashP &h)
{
    const int x = bucket_index(p.x, h.lo[0], h.inv, h.dims[0]);
    const int y = bucket_index(p.y, h.lo[1], h.inv, h.dims[1]);
    const int z = bucket_index(p.z, h.lo[2], h.inv, h.dims[2]);
    return (z * h.dims[1] + y) * h.dims[0] + x;
}

// bucket of every particle and its rank there (in no set order: the searches
// decide ties by id)
__device__ __forceinline__ void hash_count(int wg, const float4 *__restrict__ pts, int np,
                                           const HashP &h, unsigned *__restrict__ cnt,
                                           int2 *__restrict__ bk)
{
    const int p = wg * 256 + threadIdx.x;
    if (p >= np) return;
    const int b = bucket_of(pts[p], h);
    bk[p] = make_int2(b, (int)atomicAdd(&cnt[b], 1u));
}

// the fourth word is the particle's id: its index, or with several blocks
// its home key (rank << 23 | cell), which also breaks distance ties
__device__ __forceinline__ void hash_scatter(int wg, const float4 *__restrict__ pts, int np,
                                             const int2 *__restrict__ bk,
                                             const unsigned *__restrict__ start,
                                             float4 *__restrict__ sorted,
                                             const int *__restrict__ key)
{
    const int p = wg * 256 + threadIdx.x;
    if (p >= np) return;
    const int2 b = bk[p];
    const float4 q = pts[p];
    sorted[start[b.x] + (unsigned)b.y] =
        make_float4(q.x, q.y, q.z, __int_as_float(key ? key[p] : p));
}

// ---------------------------------------------------------------------------
// nearest site of a grid point
// ---------------------------------------------------------------------------
__device__ __forceinline__ bool better64(double d, int id, double bd, int bid)
{
    return d < bd || (d == bd && id < bid);
}

// The buckets of shell r around bucket c (Chebyshev distance r), as runs of
// the bucket-sorted particle array: buckets are numbered x fastest, so the
// buckets of a row that lies on the shell's z or y faces form one run
// [start[b0], start[b1 + 1]); an inner row contributes its two end buckets.
// Each (dz, dy) row gives at most two runs, visited in order by the caller.
struct ShellRow {
    unsigned a0, a1, b0, b1;   // runs [a0, a1) and [b0, b1)
};

__device__ __forceinline__ ShellRow shell_row(int r, int dz, int dy, int y, int z, int cx,
                                              const HashP &h, const unsigned *__restrict__ start)
{
    const int row = (z * h.dims[1] + y) * h.dims[0];
    const bool face = (dz == -r || dz == r || dy == -r || dy == r);
    ShellRow s{0u, 0u, 0u, 0u};
    if (face) {
        const int xa = max(cx - r, 0), xb = min(cx + r, h.dims[0] - 1);
        s.a0 = start[row + xa];
        s.a1 = start[row + xb + 1];
    } else {
        if (cx - r >= 0) {
            s.a0 = start[row + cx - r];
            s.a1 = start[row + cx - r + 1];
        }
        if (cx + r < h.dims[0]) {
            s.b0 = start[row + cx + r];
            s.b1 = start[row + cx + r + 1];
        }
    }
    return s;
}

__device__ __forceinline__ void home_bucket(float gx, float gy, float gz, const HashP &h, int c[3])
{
    const float q[3] = {gx, gy, gz};
#pragma unroll
    for (int i = 0; i < 3; ++i) c[i] = bucket_index(q[i], h.lo[i], h.inv, h.dims[i]);
}

// search in double; returns the owner id
__device__ int nearest_f64(float gx, float gy, float gz, const HashP &h,
                           const unsigned *__restrict__ start, const float4 *__restrict__ hp)
{
    int c[3];
    home_bucket(gx, gy, gz, h, c);
    const float rel[3] = {gx - h.lo[0], gy - h.lo[1], gz - h.lo[2]};
    double best = 1e300;
    int bid = 0x7fffffff;
    const int rmax = h.dims[0] + h.dims[1] + h.dims[2];
    for (int r = 0; r <= rmax; ++r) {
        for (int dz = -r; dz <= r; ++dz) {
            const int z = c[2] + dz;
            if (z < 0 || z >= h.dims[2]) continue;
            for (int dy = -r; dy <= r; ++dy) {
                const int y = c[1] + dy;
                if (y < 0 || y >= h.dims[1]) continue;
                const ShellRow sr = shell_row(r, dz, dy, y, z, c[0], h, start);
                for (int k = 0; k < 2; ++k) {
                    const unsigned s1 = k ? sr.b1 : sr.a1;
                    for (unsigned s = k ? sr.b0 : sr.a0; s < s1; ++s) {
                        const float4 p = hp[s];
                        const double ex = (double)gx - (double)p.x;
                        const double ey = (double)gy - (double)p.y;
                        const double ez = (double)gz - (double)p.z;
                        const double d = ex * ex + ey * ey + ez * ez;
                        const int id = __float_as_int(p.w);
                        if (better64(d, id, best, bid)) {
                            best = d;
                            bid = id;
                        }
                    }
                }
            }
        }
        if (bid == 0x7fffffff) continue;
        // every bucket beyond shell r is at least r cells away, less what the
        // float bucket arithmetic can be off
        const double lb = fmax(0.0, (double)r - (double)h.slack) * (double)h.cell;
        if (r > 0 && lb * lb > best * (1.0 + 1e-9) + 1e-300) break;
        // most end above (this bound's squares are floats: a few ulp more)
        if (r > 1 &&
            (double)beyond_shell2(r, c, c, rel, rel, h) > best * (1.0 + 2e-6) + 1e-300)
            break;
    }
    return bid;
}

// ---------------------------------------------------------------------------
// The nearest sites of the P points of a tile at once: the wave takes the
// buckets around the tile's box shell by shell.  With P = 64 every lane meets
// every particle of a bucket; with 8 points or one (grids coarser than the
// particles, owner_tile) the 64 / P lanes of a point take a run's particles in
// turn and compare what they found at the end.  With P = 64 the particles are
// wave-uniform (scalar loads, no per-lane runs), a row of buckets farther from
// the box than the largest best distance of the lanes is skipped, and nothing
// diverges.  A lane by itself sees 27 buckets where the tile sees up to 64, but
// its wave runs the longest of 64 different row sequences, and in a cluster's
// core it cannot skip the full buckets around its own: 262k particles on 192^3
// 0.48 -> 0.29 ms, 8 Plummer blocks on 128^3 6.4 -> 1.06, 262k on 63^3
// 0.108 -> 0.067.  Vector issue bounds it: 13 instructions per particle met.
// ---------------------------------------------------------------------------
struct Tile {
    float lo[3], hi[3];   // box of the tile's points (uniform)
};

__device__ __forceinline__ float uniform_f(float x)
{
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x)));
}

// largest value of the lanes
template <class T> __device__ __forceinline__ T wave_max(T x)
{
    for (int off = 32; off >= 1; off >>= 1) {
        const T y = __shfl_xor(x, off);
        x = y > x ? y : x;
    }
    return x;
}

// Calls visit(particle) for every particle that may be the nearest of a lane's
// point, all lanes together, until no unvisited one can be: reach() is the
// wave's largest squared distance still to beat (infinite before the first
// particle), widened by the caller's rounding margin.
template <int P, bool OUT, class Visit, class Reach>
__device__ __forceinline__ void tile_search(const Tile &t, const HashP &h,
                                            const unsigned *__restrict__ start,
                                            const float4 *__restrict__ hp, Visit visit,
                                            Reach reach)
{
    const int lane = (int)(threadIdx.x & 63);
    int c0[3], c1[3];
    home_bucket(t.lo[0], t.lo[1], t.lo[2], h, c0);
    home_bucket(t.hi[0], t.hi[1], t.hi[2], h, c1);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        c0[a] = __builtin_amdgcn_readfirstlane(c0[a]);
        c1[a] = __builtin_amdgcn_readfirstlane(c1[a]);
    }
    // the box relative to the hash's origin, and its distance to bucket i on
    // axis a
    float lo[3], hi[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        lo[a] = uniform_f(t.lo[a] - h.lo[a]);
        hi[a] = uniform_f(t.hi[a] - h.lo[a]);
    }
    auto gap = [&](int i, int a) { return bucket_gap(lo[a], hi[a], i, h); };
    constexpr unsigned L = 64 / P;   // lanes per point: each meets its share of a run
    auto run = [&](unsigned s0, unsigned s1) {
        unsigned s = s0 + (L > 1 ? (unsigned)lane / P : 0u);
        for (; s + 3 * L < s1; s += 4 * L) {
            const float4 p0 = hp[s], p1 = hp[s + L], p2 = hp[s + 2 * L], p3 = hp[s + 3 * L];
            visit(p0);
            visit(p1);
            visit(p2);
            visit(p3);
        }
        for (; s < s1; s += L) visit(hp[s]);
    };
    const int rmax = h.dims[0] + h.dims[1] + h.dims[2];
    double m2 = INFINITY;
    auto near = [&](float d2, int x) {   // bucket x of a row at squared distance d2
        const float gx = gap(x, 0);
        return x < 0 || x >= h.dims[0] || (double)(d2 + gx * gx) <= m2;
    };
    for (int r = 0; r <= rmax; ++r) {
        // the shell's rows, one per lane: its buckets' runs
        const int z0 = max(c0[2] - r, 0), z1 = min(c1[2] + r, h.dims[2] - 1);
        const int y0 = max(c0[1] - r, 0), y1 = min(c1[1] + r, h.dims[1] - 1);
        const int ny = y1 - y0 + 1, nrow = ny * (z1 - z0 + 1);
        const int xa = max(c0[0] - r, 0), xb = min(c1[0] + r, h.dims[0] - 1);
        for (int i0 = 0; i0 < nrow; i0 += 64) {
            const int i = i0 + lane;
            unsigned a0 = 0, a1 = 0, b0 = 0, b1 = 0;
            float d2 = 0.0f;
            if (i < nrow) {
                const int z = z0 + i / ny, y = y0 + i % ny;
                const long long row = ((long long)z * h.dims[1] + y) * h.dims[0];
                const float gy = gap(y, 1), gz = gap(z, 2);
                d2 = gy * gy + gz * gz;
                // the row's end buckets only when they are near enough
                const bool lo = near(d2, c0[0] - r), hi = near(d2, c1[0] + r);
                if (r == 0 || z < c0[2] - r + 1 || z > c1[2] + r - 1 || y < c0[1] - r + 1 ||
                    y > c1[1] + r - 1) {
                    a0 = start[row + (lo ? xa : min(xa + 1, xb))];
                    a1 = start[row + (hi ? xb + 1 : max(xb, xa))];
                } else {
                    if (lo && c0[0] - r >= 0) {
                        a0 = start[row + c0[0] - r];
                        a1 = start[row + c0[0] - r + 1];
                    }
                    if (hi && c1[0] + r < h.dims[0]) {
                        b0 = start[row + c1[0] + r];
                        b1 = start[row + c1[0] + r + 1];
                    }
                }
            }
            unsigned long long todo = __ballot((a0 < a1 || b0 < b1) && (double)d2 <= m2);
            while (todo) {
                const int l = __ffsll(todo) - 1;
                todo &= todo - 1ull;
                run((unsigned)__builtin_amdgcn_readlane((int)a0, l),
                    (unsigned)__builtin_amdgcn_readlane((int)a1, l));
                const unsigned e0 = (unsigned)__builtin_amdgcn_readlane((int)b0, l),
                               e1 = (unsigned)__builtin_amdgcn_readlane((int)b1, l);
                if (e0 < e1) run(e0, e1);
            }
        }
        // the squared gaps are floats: a few ulp more
        m2 = (double)reach() * (1.0 + 2e-6);
        if (OUT) {
            if ((double)beyond_shell2(r, c0, c1, lo, hi, h) > m2) break;
        } else {
            // every bucket beyond shell r is at least r cells from the box
            const double lb = fmax(0.0, (double)r - (double)h.slack) * (double)h.cell;
            if (r > 0 && lb * lb > m2) break;
        }
    }
}

// on: this lane has a point (the others see the same particles and are
// ignored); the 64 / P lanes of a point end with the same answer
template <int P, bool OUT>
__device__ __forceinline__ int tile_nearest_f32(float gx, float gy, float gz, bool on,
                                                const Tile &t, const HashP &h,
                                                const unsigned *__restrict__ start,
                                                const float4 *__restrict__ hp)
{
    float best = INFINITY, second = INFINITY;
    int bid = -1;
    tile_search<P, OUT>(
        t, h, start, hp,
        [&](const float4 p) {
            const float ex = gx - p.x, ey = gy - p.y, ez = gz - p.z;
            const float d = ex * ex + ey * ey + ez * ez;
            second = fminf(second, fmaxf(best, d));
            bid = d < best ? __float_as_int(p.w) : bid;
            best = fminf(best, d);
        },
        [&] {
            float b = best;
            for (int off = P; off < 64; off <<= 1) b = fminf(b, __shfl_xor(b, off));
            return wave_max(on ? b * 1.0001f + 1e-30f : 0.0f);
        });
    for (int off = P; off < 64; off <<= 1) {
        const float ob = __shfl_xor(best, off), os = __shfl_xor(second, off);
        const int oid = __shfl_xor(bid, off);
        second = fminf(fminf(second, os), fmaxf(best, ob));
        bid = ob < best ? oid : bid;   // of two equal ones neither stands
        best = fminf(best, ob);
    }
    // decided only if the runner-up is clearly farther (32 ulp window) and
    // nothing underflowed, or the point coincides with a site: exact in float
    const float tau = 32.0f * 5.9604645e-8f;
    if (bid >= 0 && best > 1e-30f && second > best * (1.0f + tau)) return bid;
    if (bid >= 0 && best == 0.0f && second > 1e-30f) return bid;
    return -1;
}

template <int P, bool OUT>
__device__ __forceinline__ int tile_nearest_f64(float gx, float gy, float gz, bool on,
                                                const Tile &t, const HashP &h,
                                                const unsigned *__restrict__ start,
                                                const float4 *__restrict__ hp)
{
    double best = 1e300;
    int bid = 0x7fffffff;
    auto meet = [&](double d, int id) {
        const bool b = better64(d, id, best, bid);
        best = b ? d : best;
        bid = b ? id : bid;
    };
    tile_search<P, OUT>(
        t, h, start, hp,
        [&](const float4 p) {
            const double ex = (double)gx - (double)p.x;
            const double ey = (double)gy - (double)p.y;
            const double ez = (double)gz - (double)p.z;
            meet(ex * ex + ey * ey + ez * ez, __float_as_int(p.w));
        },
        [&] {
            double b = best;
            for (int off = P; off < 64; off <<= 1) b = fmin(b, __shfl_xor(b, off));
            return wave_max(on ? b * (1.0 + 1e-9) + 1e-300 : 0.0);
        });
    for (int off = P; off < 64; off <<= 1)
        meet(__shfl_xor(best, off), __shfl_xor(bid, off));
    return bid;
}

// a wave per tile of P block grid points (owner_tile), 64 / P lanes per point.
// With several blocks the owner is a home key (rank << 23 | cell) and the
// counts go to the home block's cell (npts_tab / stex_tab by rank).
template <int P, bool OUT>
__global__ __launch_bounds__(256) void k_owner(GridP gp, HashP h,
                                               const unsigned *__restrict__ start,
                                               const float4 *__restrict__ hp, int *__restrict__ owner,
                                               int prec, unsigned *ctrs, OwnerTile ot, int tiles_x,
                                               int tiles_y, int ntiles, const int *__restrict__ status,
                                               int *__restrict__ npts, int ncells,
                                               int *const *__restrict__ npts_tab,
                                               const int *const *__restrict__ stex_tab,
                                               unsigned *__restrict__ defq, unsigned defq_cap)
{
    const int wave = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (wave >= ntiles) return;
    const int lane = threadIdx.x & 63, pt = lane & (P - 1);
    const int tx = wave % tiles_x, ty = (wave / tiles_x) % tiles_y, tz = wave / (tiles_x * tiles_y);
    const int g0[3] = {tx << ot.bits[0], ty << ot.bits[1], tz << ot.bits[2]};
    const int lx0 = g0[0] + (pt & ((1 << ot.bits[0]) - 1)),
              ly0 = g0[1] + ((pt >> ot.bits[0]) & ((1 << ot.bits[1]) - 1)),
              lz0 = g0[2] + (pt >> (ot.bits[0] + ot.bits[1]));
    const bool on_grid = lx0 < gp.bnum_idx[0] && ly0 < gp.bnum_idx[1] && lz0 < gp.bnum_idx[2];
    const bool mine = on_grid && lane < P;   // the point's lane that writes and counts
    // off-grid lanes of an edge tile stand in for an on-grid point of the
    // tile but write nothing and count nothing
    const int lx = on_grid ? lx0 : g0[0], ly = on_grid ? ly0 : g0[1], lz = on_grid ? lz0 : g0[2];
    const long long lidx = ((long long)lz * gp.bnum_idx[1] + ly) * gp.bnum_idx[0] + lx;
    const int gx = gp.bmin_idx[0] + lx, gy = gp.bmin_idx[1] + ly, gz = gp.bmin_idx[2] + lz;
    const float px = idx2phys1(gx, gp.step[0], gp.gmin[0]);
    const float py = idx2phys1(gy, gp.step[1], gp.gmin[1]);
    const float pz = idx2phys1(gz, gp.step[2], gp.gmin[2]);
    const bool in_block = px >= gp.bmin[0] && px <= gp.bmax[0] && py >= gp.bmin[1] &&
                          py <= gp.bmax[1] && pz >= gp.bmin[2] && pz <= gp.bmax[2];
    if (!in_block && mine) owner[lidx] = -1;
    int o = -1;
    bool failed = false;
    const bool on = in_block && on_grid;
    if (__ballot(on)) {
        Tile t;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            t.lo[a] = uniform_f(idx2phys1(gp.bmin_idx[a] + g0[a], gp.step[a], gp.gmin[a]));
            const int last = min(g0[a] + (1 << ot.bits[a]) - 1, gp.bnum_idx[a] - 1);
            t.hi[a] = uniform_f(idx2phys1(gp.bmin_idx[a] + last, gp.step[a], gp.gmin[a]));
        }
        if (prec == 0) o = tile_nearest_f32<P, OUT>(px, py, pz, on, t, h, start, hp);
        else o = tile_nearest_f64<P, OUT>(px, py, pz, on, t, h, start, hp);
        if (!on || !mine) o = -1;
        failed = on && mine && o < 0 && prec == 0;
    }
    // FP32 filter failures go to a queue that k_owner_deferred searches in
    // FP64 with full waves: searched here, one failing lane would hold its
    // 63 neighbours for a whole FP64 search.  C_DEFER counts every failure
    // (one atomic per wave); beyond the queue's end the search runs inline.
    bool defer = false;
    const unsigned long long dm = __ballot(failed);
    if (dm) {
        const int leader = __ffsll(dm) - 1;
        unsigned base = 0;
        if (lane == leader) base = atomicAdd(&ctrs[C_DEFER], (unsigned)__popcll(dm));
        base = __shfl(base, leader);
        const unsigned slot = base + (unsigned)__popcll(dm & ((1ull << lane) - 1ull));
        if (failed && slot < defq_cap) {
            defq[slot] = (unsigned)lidx;
            defer = true;
        }
    }
    if (in_block && mine) {
        if (o < 0 && !defer) o = nearest_f64(px, py, pz, h, start, hp);
        owner[lidx] = o;           // -1 for a deferred point until its FP64 search
    }
    // points per deposited cell; the lanes of a tile mostly share owners, so
    // one atomic per distinct owner in the wave
    const int hc = npts_tab ? (o & 0x7fffff) : o;
    const int *hst = npts_tab && o >= 0 ? stex_tab[o >> 23] : status;
    int *hnp = npts_tab && o >= 0 ? npts_tab[o >> 23] : npts;
    const bool cnt = mine && in_block && o >= 0 && (npts_tab || o < ncells) &&
                     hst[hc] == EX_DEPOSIT;
    unsigned long long pend = __ballot(cnt);
    while (pend) {
        const int leader = __ffsll((unsigned long long)pend) - 1;
        const int val = __builtin_amdgcn_readlane(o, leader);
        const unsigned long long same = __ballot(cnt && o == val);
        if (lane == leader) atomicAdd(&hnp[hc], __popcll(same));
        pend &= ~same;
    }
}

// the FP64 search of the points k_owner deferred, one lane per point (the
// queue holds the points of each wave together, so lanes stay close)
__global__ __launch_bounds__(256) void k_owner_deferred(GridP gp, HashP h,
                                                        const unsigned *__restrict__ start,
                                                        const float4 *__restrict__ hp,
                                                        int *__restrict__ owner,
                                                        const unsigned *ctrs,
                                                        const unsigned *__restrict__ defq,
                                                        unsigned defq_cap,
                                                        const int *__restrict__ status,
                                                        int *__restrict__ npts, int ncells,
                                                        int *const *__restrict__ npts_tab,
                                                        const int *const *__restrict__ stex_tab)
{
    unsigned n = ctrs[C_DEFER];
    if (n > defq_cap) n = defq_cap;
    const unsigned nx = (unsigned)gp.bnum_idx[0], ny = (unsigned)gp.bnum_idx[1];
    for (unsigned i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const unsigned lidx = defq[i];
        const int lx = (int)(lidx % nx), ly = (int)((lidx / nx) % ny), lz = (int)(lidx / (nx * ny));
        const float px = idx2phys1(gp.bmin_idx[0] + lx, gp.step[0], gp.gmin[0]);
        const float py = idx2phys1(gp.bmin_idx[1] + ly, gp.step[1], gp.gmin[1]);
        const float pz = idx2phys1(gp.bmin_idx[2] + lz, gp.step[2], gp.gmin[2]);
        const int o = nearest_f64(px, py, pz, h, start, hp);
        owner[lidx] = o;
        if (o < 0) continue;
        const int hc = npts_tab ? (o & 0x7fffff) : o;
        const int *hst = npts_tab ? stex_tab[o >> 23] : status;
        int *hnp = npts_tab ? npts_tab[o >> 23] : npts;
        if ((npts_tab || o < ncells) && hst[hc] == EX_DEPOSIT) atomicAdd(&hnp[hc], 1);
    }
}

void launch_owner(const GridP &gp, const HashP &h, const unsigned *start, const float4 *hp,
                  int *owner, int prec, unsigned *ctrs, const int *status, int *npts, int ncells,
                  int *const *npts_tab, const int *const *stex_tab, unsigned *defq,
                  unsigned defq_cap, hipStream_t s)
{
    double step[3];
    for (int a = 0; a < 3; ++a) step[a] = (double)gp.step[a] * (double)h.inv;
    const OwnerTile ot = owner_tile(gp.bnum_idx, step, h.dims);
    int n[3];
    for (int a = 0; a < 3; ++a) n[a] = ((gp.bnum_idx[a] - 1) >> ot.bits[a]) + 1;
    const int ntiles = n[0] * n[1] * n[2];
    if (ntiles <= 0) return;
    // a grid that leaves the particles' box by more than a bucket
    bool out = false;
    for (int a = 0; a < 3; ++a) {
        const float g0 = idx2phys1(gp.bmin_idx[a], gp.step[a], gp.gmin[a]);
        const float g1 = idx2phys1(gp.bmin_idx[a] + gp.bnum_idx[a] - 1, gp.step[a], gp.gmin[a]);
        out |= g0 < h.lo[a] - h.cell || g1 > h.lo[a] + (float)(h.dims[a] + 1) * h.cell;
    }
    auto *kernel = out ? (ot.points == 64 ? k_owner<64, true>
                                          : (ot.points == 8 ? k_owner<8, true> : k_owner<1, true>))
                       : (ot.points == 64 ? k_owner<64, false>
                                          : (ot.points == 8 ? k_owner<8, false>
                                                            : k_owner<1, false>));
    hipLaunchKernelGGL(kernel, dim3((ntiles + 3) / 4), dim3(256), 0, s, gp, h, start, hp, owner,
                       prec, ctrs, ot, n[0], n[1], ntiles, status, npts, ncells, npts_tab, stex_tab,
                       defq, prec == 0 ? defq_cap : 0u);
    if (prec == 0 && defq_cap > 0) {
        const unsigned nblk = defq_cap / 256 + 1;
        hipLaunchKernelGGL(k_owner_deferred, dim3(nblk < 2048 ? nblk : 2048), dim3(256), 0, s,
                           gp, h, start, hp, owner, ctrs, defq, defq_cap, status, npts, ncells,
                           npts_tab, stex_tab);
    }
}

// ---------------------------------------------------------------------------
// deposit status of each cell: its star is complete and every Voronoi vertex
// (circumcenter of a star tet) lies inside the data bounds +- 2 FLT_EPSILON
// (the reference's CellGridPts test, src/dense.cpp:1381-1392, on the exact
// bbox of the cell).  Both are "for all tets of the star" conditions, so they
// are decided tet by tet: one lane per tet flags its vertices
//   - incomplete: a hull face (neighbour -1) makes its three vertices hull
//     vertices (the star traversal of neighbor_edges would meet it);
//   - outside: its circumcenter leaves the bounds;
//   - defined: its circumcenter exists (flat tets of exactly cospherical
//     points have none and are skipped; a cell with none is degenerate).
// MIXED decides with the FP32 circumcenter and its error bound (cc.w) and
// recomputes in FP64 only when the bound straddles a threshold; FP64
// recomputes every circumcenter.  The flags are plain byte stores of 1.
// ---------------------------------------------------------------------------
__device__ __forceinline__ int comp4(const int4 &q, int i)
{
    return i == 0 ? q.x : (i == 1 ? q.y : (i == 2 ? q.z : q.w));
}

__device__ __forceinline__ void exact_flags(int wg, int nwg, const BlockIn &in, const GridP &gp,
                                            int prec, unsigned char *__restrict__ flags,
                                            unsigned *ctrs)
{
    const int nc = in.ncells;
    unsigned char *inc = flags, *out = flags + nc, *def = flags + 2 * (size_t)nc;
    float lo[3], hi[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const float e = (gp.dmax[i] - gp.dmin[i]) * 2.0f * FLT_EPSILON;
        lo[i] = gp.dmin[i] - e;
        hi[i] = gp.dmax[i] + e;
    }
    __shared__ unsigned s_fb;
    if (threadIdx.x == 0) s_fb = 0;
    __syncthreads();
    unsigned nfb = 0;   // FP64 re-checks of this lane
    for (int t = wg * 256 + threadIdx.x; t < in.ntets; t += nwg * 256) {
        const int4 vv = in.tets[2 * t];
        if (vv.x >= nc && vv.y >= nc && vv.z >= nc && vv.w >= nc) continue;   // ghosts only
        const int4 nb = in.tets[2 * t + 1];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (comp4(nb, i) >= 0) continue;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int u = comp4(vv, k);
                if (k != i && u < nc) inc[u] = 1;
            }
        }
        bool decided = false, is_out = false, is_def = false;
        if (prec == 0) {
            const float4 c = in.cc[t];
            const float err = c.w;   // NaN or inf: undecidable in float
            if (err >= 0.0f && err < 1e-3f) {
                bool surely_in = true, surely_out = false;
                const float q[3] = {c.x, c.y, c.z};
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    surely_in &= (q[i] - err > lo[i]) && (q[i] + err < hi[i]);
                    surely_out |= (q[i] + err < lo[i]) || (q[i] - err > hi[i]);
                }
                if (surely_in || surely_out) {
                    decided = true;
                    is_def = true;
                    is_out = surely_out;
                }
            }
            nfb += decided ? 0u : 1u;
        }
        if (!decided) {
            const float4 a = in.pts[vv.x], b = in.pts[vv.y], c = in.pts[vv.z], d = in.pts[vv.w];
            double ox, oy, oz;
            circumcenter_f64(a.x, a.y, a.z, b.x, b.y, b.z, c.x, c.y, c.z, d.x, d.y, d.z, ox, oy, oz);
            if (!(isnan(ox) || isnan(oy) || isnan(oz))) {
                is_def = true;
                is_out = ox < (double)lo[0] || oy < (double)lo[1] || oz < (double)lo[2] ||
                         ox > (double)hi[0] || oy > (double)hi[1] || oz > (double)hi[2];
            }
        }
        if (is_def) {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int u = comp4(vv, k);
                if (u < nc) {
                    def[u] = 1;
                    if (is_out) out[u] = 1;
                }
            }
        }
    }
    // one global atomic per workgroup (and few workgroups): same-address
    // atomics serialize in L2, ~10 ns each, and one per wave outlasted the
    // kernel's own work
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) nfb += __shfl_xor(nfb, m);
    if ((threadIdx.x & 63) == 0 && nfb) atomicAdd(&s_fb, nfb);
    __syncthreads();
    if (threadIdx.x == 0 && s_fb) atomicAdd(&ctrs[C_FALLBACK], s_fb);
}

__device__ __forceinline__ void exact_classify(int wg, const int *__restrict__ v2t, int nc,
                                               const unsigned char *__restrict__ flags,
                                               int *status)
{
    const int v = wg * 256 + threadIdx.x;
    if (v >= nc) return;
    int st;
    if (v2t[v] < 0 || flags[v]) st = EX_INCOMPLETE;
    else if (!flags[2 * (size_t)nc + v]) st = EX_DEGENERATE;
    else if (flags[nc + v]) st = EX_OUTSIDE;
    else st = EX_DEPOSIT;
    status[v] = st;
}

// What the owner search needs, in two launches with the scan of the bucket
// counts between: the bucket hash (the first bh workgroups) and the deposit
// status of each cell.  The two are independent, and for small blocks each
// step is a launch of 3 to 4 us (4,000 cells on 49^3, whole run: 153 us
// apart, 143 together).
__global__ __launch_bounds__(256) void k_exact_count(BlockIn in, GridP gp, int prec,
                                                     unsigned char *__restrict__ flags,
                                                     unsigned *ctrs, int np, HashP h,
                                                     unsigned *__restrict__ cnt,
                                                     int2 *__restrict__ bk, int bh)
{
    if ((int)blockIdx.x < bh) hash_count((int)blockIdx.x, in.pts, np, h, cnt, bk);
    else exact_flags((int)blockIdx.x - bh, (int)gridDim.x - bh, in, gp, prec, flags, ctrs);
}

__global__ __launch_bounds__(256) void k_exact_place(BlockIn in,
                                                     const unsigned char *__restrict__ flags,
                                                     int *status, int np,
                                                     const int2 *__restrict__ bk,
                                                     const unsigned *__restrict__ start,
                                                     float4 *__restrict__ sorted,
                                                     const int *__restrict__ key, int bh)
{
    if ((int)blockIdx.x < bh) hash_scatter((int)blockIdx.x, in.pts, np, bk, start, sorted, key);
    else exact_classify((int)blockIdx.x - bh, in.v2t, in.ncells, flags, status);
}

// start: one word more than there are buckets (the extra one turns into the
// total)
void launch_exact_setup(const BlockIn &in, const GridP &gp, int np, const HashP &h,
                        unsigned *start, unsigned *sums, int2 *bk, float4 *sorted, const int *key,
                        int *status, int prec, unsigned *ctrs, unsigned char *flags,
                        hipStream_t s)
{
    const int nbk = h.dims[0] * h.dims[1] * h.dims[2];
    const int bh = (np + 255) / 256;
    const int bt = in.ncells > 0 ? std::min(4096, (in.ntets + 255) / 256) : 0;
    const int bc = (in.ncells + 255) / 256;
    if (bh + bt > 0)
        hipLaunchKernelGGL(k_exact_count, dim3(bh + bt), dim3(256), 0, s, in, gp, prec, flags,
                           ctrs, np, h, start, bk, bh);
    launch_scan_u32(start, (unsigned)nbk + 1u, sums, s);
    if (bh + bc > 0)
        hipLaunchKernelGGL(k_exact_place, dim3(bh + bc), dim3(256), 0, s, in,
                           (const unsigned char *)flags, status, np, (const int2 *)bk,
                           (const unsigned *)start, sorted, key, bh);
}

// ---------------------------------------------------------------------------
// density, CIC of deposited cells without points (the point counts come from
// k_owner)
// ---------------------------------------------------------------------------

// With several blocks a point owned by another block's cell is that
// block's contribution, keyed like a received point (1 << 31 | rank << 24 |
// cell << 1), so that the fold orders it after this block's own cells.
__global__ void k_exact_density(GridP gp, const int *__restrict__ owner, const int *__restrict__ status,
                                const int *__restrict__ npts, int ncells, CellOut o, int prec,
                                int *const *__restrict__ npts_tab,
                                const int *const *__restrict__ stex_tab, int self)
{
    const size_t n = (size_t)gp.bnum_idx[0] * gp.bnum_idx[1] * gp.bnum_idx[2];
    for (size_t g = (size_t)blockIdx.x * blockDim.x + threadIdx.x; g < n;
         g += (size_t)gridDim.x * blockDim.x) {
        const int ow = owner[g];
        if (ow < 0) continue;
        int N;
        unsigned key;
        if (npts_tab) {
            const int r = ow >> 23, cell = ow & 0x7fffff;
            if (stex_tab[r][cell] != EX_DEPOSIT) continue;
            N = npts_tab[r][cell];
            key = r == self ? cell_key(cell, 0)
                            : (0x80000000u | ((unsigned)r << 24) | cell_key(cell, 0));
        } else {
            if (ow >= ncells || status[ow] != EX_DEPOSIT) continue;
            N = npts[ow];
            key = cell_key(ow, 0);
        }
        const float m = prec == 0 ? gp.mass / (float)N : (float)((double)gp.mass / (double)N);
        // an owned point is in the block and its grid, and this is its first
        // contribution (every density pass runs before any CIC pass): the
        // first-contribution stores of push_point without its atomic
        o.count[g] = 1u;
        o.first[g] = make_uint2(key, __float_as_uint(m));
        o.density[g] = (float)((double)m / (double)gp.div);
    }
}

__global__ void k_exact_cic(BlockIn in, GridP gp, const int *__restrict__ status_ex,
                            CellOut o, const Router *rt, int self)
{
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= in.ncells) return;
    const int s = status_ex[v];
    int out_status = s, out_n = 0;
    if (s == EX_DEPOSIT) {
        const int N = o.npts[v];
        if (N > 0) {
            out_status = 0;
            out_n = N;
        } else {
            const float4 p = in.pts[v];
            int mn[3];
            float m8[8];
            cic_weights(p.x, p.y, p.z, gp.mass, gp, mn, m8);
            for (int k = 0; k < 8; ++k)
                deposit_point(mn[0] + (k & 1), mn[1] + ((k >> 1) & 1), mn[2] + (k >> 2), m8[k],
                              cell_key(v, 0), gp, o, rt, self);
            out_status = 1;
            out_n = 8;
        }
    }
    o.status[v] = out_status;
    if (s != EX_DEPOSIT) o.npts[v] = 0;
    else o.npts[v] = out_n;
}

void launch_exact_tail(const BlockIn &in, const GridP &gp, const int *owner, const int *status_ex,
                       const CellOut &o, int prec, int *const *npts_tab,
                       const int *const *stex_tab, const Router *rt, int self, int parts,
                       hipStream_t s)
{
    const size_t n = (size_t)gp.bnum_idx[0] * gp.bnum_idx[1] * gp.bnum_idx[2];
    size_t blocks = (n + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    if (blocks == 0) blocks = 1;
    if (parts & 1)
        hipLaunchKernelGGL(k_exact_density, dim3((unsigned)blocks), dim3(256), 0, s, gp, owner,
                           status_ex, o.npts, in.ncells, o, prec, npts_tab, stex_tab, self);
    if ((parts & 2) && in.ncells > 0)
        hipLaunchKernelGGL(k_exact_cic, dim3((in.ncells + 255) / 256), dim3(256), 0, s, in, gp,
                           status_ex, o, rt, self);
}

}  // namespace t2
