// scan_lines.hpp -- the scanline search of a cell on words of verdicts, one
// word per line (y, z) of its box: the verdicts of a line, the state machine
// on the words, and one wave's scan and deposit of one cell.
#pragma once

#include "cell_status.hpp"
#include "deposit.hpp"
#include "geom.hpp"
#include "kernels.hpp"
#include "scan_bits.hpp"

namespace t2 {

// data-bounds filter of a cell's box and its NaN (src/dense.cpp:1381-1392)
__device__ __forceinline__ int box_status(float mnx, float mny, float mnz, float mxx, float mxy,
                                          float mxz, const GridP &gp)
{
    const float ex = (gp.dmax[0] - gp.dmin[0]) * 2.0f * FLT_EPSILON;
    const float ey = (gp.dmax[1] - gp.dmin[1]) * 2.0f * FLT_EPSILON;
    const float ez = (gp.dmax[2] - gp.dmin[2]) * 2.0f * FLT_EPSILON;
    if (mnx < gp.dmin[0] - ex || mny < gp.dmin[1] - ey || mnz < gp.dmin[2] - ez ||
        mxx > gp.dmax[0] + ex || mxy > gp.dmax[1] + ey || mxz > gp.dmax[2] + ez)
        return ST_OUTSIDE;
    if (isnan(mnx) || isnan(mny) || isnan(mnz) || isnan(mxx) || isnan(mxy) || isnan(mxz))
        return ST_DEGENERATE;
    return ST_SCAN;
}

// the verdicts of XC points x0.. of one line against nf planes, as bits
template <int XC>
__device__ __forceinline__ unsigned line_verdicts(const float4 *fa, const float2 *fb, int nf,
                                                  int nfmax, float p0, float step0, int x0,
                                                  float qy, float qz, float eps)
{
    float qx[XC], hi[XC], lo[XC];
#pragma unroll
    for (int i = 0; i < XC; ++i) {
        qx[i] = p0 + (float)(x0 + i) * step0;
        hi[i] = -INFINITY;
        lo[i] = INFINITY;
    }
    // to the wave's largest face count; a lane past its own repeats its last
#pragma unroll 2
    for (int k = 0; k < nfmax; ++k) {
        const int kk = k < nf ? k : nf - 1;
        const float4 a = fa[kk];
        const float2 b = fb[kk];
        const float ty = a.y * (qy - b.x), tz = a.z * (qz - b.y);
#pragma unroll
        for (int i = 0; i < XC; ++i) {
            const float d = a.x * (qx[i] - a.w) + ty + tz;
            hi[i] = fmaxf(hi[i], d);
            lo[i] = fminf(lo[i], d);
        }
    }
    unsigned m = 0;
#pragma unroll
    for (int i = 0; i < XC; ++i)
        if (!(hi[i] > eps && lo[i] < -eps)) m |= 1u << i;
    return m;
}

// The scanline state machine (src/dense.cpp:1486-1676) on one word per line,
// row[z * n1 + y].  Leaves the run found on each line it walks in run (which
// starts at zero) and, in that line's row word, the number of points before
// it: a line is walked once, and probes read the next z step's.  Returns the
// number of points.
__device__ __forceinline__ int scan_rows(unsigned *row, unsigned *run, int n0, int n1, int n2)
{
    int x_left = n0 / 2, x_right = n0 / 2, y_start = 0, first_x = 0;
    int zi = 0, yi = 0, tot = 0;
    bool border_found = false;
    // one line per turn, so that lanes on different cells stay together
    for (;;) {
        const int k = zi * n1 + yi;
        int min_xi = n0 - 1, max_xi = 0;
        walk_row_bits32(row[k], n0, x_left, x_right, min_xi, max_xi);
        row[k] = (unsigned)tot;
        int first_y = y_start;
        bool z_step_done = false;
        if (min_xi <= max_xi) {
            const int len = max_xi - min_xi + 1;
            run[k] = (len >= 32 ? ~0u : (1u << len) - 1u) << min_xi;
            tot += len;
            if (yi == y_start) first_x = (min_xi + max_xi) / 2;
            if (!border_found) {
                first_y = yi;
                border_found = true;
            }
        } else if (border_found) {
            z_step_done = true;
        }
        if (yi == n1 - 1 || z_step_done) {
            if (zi + 1 >= n2) break;
            int yj;
            for (yj = first_y; yj > 0; yj--)
                if (!((row[k - yi + n1 + yj] >> first_x) & 1u)) break;
            y_start = yj;
            ++zi;
            yi = y_start;
            border_found = false;
        } else {
            ++yi;
        }
    }
    return tot;
}

// one corner of the CIC deposit, eight consecutive lanes on one site
// (DistributeScalarCIC, src/dense.cpp:1787-1872): each lane its corner's box,
// the sums over the corners in their order
__device__ __forceinline__ float cic_corner(const float4 site, float scalar, const GridP &gp,
                                            int k, int mn[3])
{
    mn[0] = phys2idx1(site.x, gp.step[0], gp.gmin[0]);
    mn[1] = phys2idx1(site.y, gp.step[1], gp.gmin[1]);
    mn[2] = phys2idx1(site.z, gp.step[2], gp.gmin[2]);
    const float gx = idx2phys1(mn[0] + (k & 1), gp.step[0], gp.gmin[0]);
    const float gy = idx2phys1(mn[1] + ((k >> 1) & 1), gp.step[1], gp.gmin[1]);
    const float gz = idx2phys1(mn[2] + (k >> 2), gp.step[2], gp.gmin[2]);
    const float e2 = 2.0f * gp.eps;
    float px = site.x, py = site.y, pz = site.z;
    if (fabsf(px - gx) < gp.eps) px += e2;
    if (fabsf(py - gy) < gp.eps) py += e2;
    if (fabsf(pz - gz) < gp.eps) pz += e2;
    const float vol = fabsf((gx - px) * (gy - py) * (gz - pz));
    const int l0 = (int)(threadIdx.x & 56u);   // the site's first lane
    float v0 = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float vi = __shfl(vol, l0 + i);
        if (i <= k && v0 == 0.0f) v0 = vi;
    }
    const float w = v0 / vol;
    float tot = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) tot += __shfl(w, l0 + i);
    return w / tot * scalar;
}

// one wave's cell: lines, runs, and the points of a turn
struct LineShared {
    static constexpr int ROWS = 1024, POINTS = 2048;
    alignas(16) unsigned row[ROWS];   // also taken as int4 runs by scan_deposit
    unsigned run[ROWS];
    unsigned short list[POINTS];
};

// Scan and deposit of cell v by one wave, its F planes in fa / fb (LDS): the
// lines of the box over the lanes (in pieces of six points), the state
// machine, the points of the runs over the lanes.  False when the box has
// more than LineShared::ROWS lines or 32 points a line, or eps < 0; every
// lane calls it with the same arguments.
__device__ __forceinline__ bool scan_cell_lines(
    const int v, const float4 site, const int F, const float4 *fa, const float2 *fb, float mnx,
    float mny, float mnz, float mxx, float mxy, float mxz, const GridP &gp, const CellOut &o,
    const Router *rt, const int self, LineShared &sl)
{
    const int lane = (int)(threadIdx.x & 63);
    const int code = box_status(mnx, mny, mnz, mxx, mxy, mxz, gp);
    if (code != ST_SCAN) {
        if (lane == 0) {
            o.status[v] = code;
            o.npts[v] = 0;
        }
        return true;
    }
    const int c0 = phys2idx1(mnx, gp.step[0], gp.gmin[0]);
    const int c1 = phys2idx1(mny, gp.step[1], gp.gmin[1]);
    const int c2 = phys2idx1(mnz, gp.step[2], gp.gmin[2]);
    const int n0 = __builtin_amdgcn_readfirstlane(phys2idx1(mxx, gp.step[0], gp.gmin[0]) - c0 + 1);
    const int n1 = __builtin_amdgcn_readfirstlane(phys2idx1(mxy, gp.step[1], gp.gmin[1]) - c1 + 1);
    const int n2 = __builtin_amdgcn_readfirstlane(phys2idx1(mxz, gp.step[2], gp.gmin[2]) - c2 + 1);
    if (n0 < 1 || n1 < 1 || n2 < 1 || n0 > 32 || n1 > LineShared::ROWS ||
        n2 > LineShared::ROWS || n1 * n2 > LineShared::ROWS || !(gp.eps >= 0.0f))
        return false;
    const int R = n1 * n2;
    const float p0 = idx2phys1(c0, gp.step[0], gp.gmin[0]);
    const float p1 = idx2phys1(c1, gp.step[1], gp.gmin[1]);
    const float p2 = idx2phys1(c2, gp.step[2], gp.gmin[2]);
    for (int i = lane; i < R; i += 64) {
        sl.row[i] = 0u;
        sl.run[i] = 0u;
    }
    __syncthreads();
    // quotients below 6 * 1024 by the float reciprocal: the error stays far
    // below the 0.5 / n margin of i + 0.5
    const int nc = (n0 + 5) / 6;
    const float rc = 1.0f / (float)nc, r1 = 1.0f / (float)n1;
    for (int i = lane; i < R * nc; i += 64) {
        const int r = (int)(((float)i + 0.5f) * rc), x0 = (i - r * nc) * 6;
        const int z = (int)(((float)r + 0.5f) * r1), y = r - z * n1;
        const unsigned m =
            line_verdicts<6>(fa, fb, F, F, p0, gp.step[0], x0, p1 + (float)y * gp.step[1],
                             p2 + (float)z * gp.step[2], gp.eps);
        atomicOr(&sl.row[r], (m << x0) & (n0 >= 32 ? ~0u : (1u << n0) - 1u));
    }
    __syncthreads();
    int tot = 0;
    if (lane == 0) tot = scan_rows(sl.row, sl.run, n0, n1, n2);
    tot = __builtin_amdgcn_readfirstlane(tot);
    __syncthreads();
    if (lane == 0) {
        o.status[v] = tot > 0 ? ST_SCAN : ST_CIC;
        o.npts[v] = tot > 0 ? tot : 8;
    }
    if (tot == 0) {
        int mn[3];
        const float m = cic_corner(site, gp.mass, gp, lane & 7, mn);
        if (lane < 8)
            deposit_point(mn[0] + (lane & 1), mn[1] + ((lane >> 1) & 1), mn[2] + (lane >> 2), m,
                          cell_key(v, gp.project ? (lane >> 2) : 0), gp, o, rt, self);
        return true;
    }
    const float m = gp.mass / (float)tot;   // src/dense.cpp:1692
    const unsigned key = cell_key(v, 0);
    constexpr int D = 4;   // deposits a lane has in flight
    unsigned routed = 0, dropped = 0;
    for (int w0 = 0; w0 < tot; w0 += LineShared::POINTS) {
        for (int r = lane; r < R; r += 64) {
            const unsigned run = sl.run[r];
            if (!run) continue;
            const int x0 = row_low(run), len = __popc(run), at = (int)sl.row[r] - w0;
            for (int i = 0; i < len; ++i)
                if (at + i >= 0 && at + i < LineShared::POINTS)
                    sl.list[at + i] = (unsigned short)(r << 5 | (x0 + i));
        }
        __syncthreads();
        const int wn = min(tot - w0, (int)LineShared::POINTS);
        for (int p0 = 0; p0 < wn; p0 += D * 64) {
            long long at[D];
            float md[D];
            unsigned kd[D];
#pragma unroll
            for (int d = 0; d < D; ++d) {
                const int p = p0 + d * 64 + lane;
                at[d] = -1;
                md[d] = m;
                kd[d] = key;
                if (p >= wn) continue;
                const unsigned e = sl.list[p];
                const int r = (int)(e >> 5), z = (int)(((float)r + 0.5f) * r1), y = r - z * n1;
                const int gx = c0 + (int)(e & 31u), gy = c1 + y, gz = c2 + z;
                at[d] = own_lidx(gx, gy, gz, gp);
                if (at[d] < 0) {
                    if (route_point(gx, gy, gz, m, key, rt, self)) ++routed;
                    else ++dropped;
                }
            }
            wave_push<D>(at, md, kd, gp.div, o);
        }
        __syncthreads();
    }
    if (__ballot(routed | dropped)) {
        for (int off = 32; off >= 1; off >>= 1) {
            routed += __shfl_xor(routed, off);
            dropped += __shfl_xor(dropped, off);
        }
        if (lane == 0 && routed) atomicAdd(&o.ctrs[C_ROUTED], routed);
        if (lane == 0 && dropped) atomicAdd(&o.ctrs[C_OFFBLOCK], dropped);
    }
    return true;
}

}  // namespace t2
