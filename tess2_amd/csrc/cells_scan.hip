// cells_scan.hip -- the scanline search and the deposit of many cells at a
// time, from the planes the geometry kernel left (cells_geom.hip).
//
// A workgroup takes the 64 cells of one tile:
//   1. one lane per cell: data-bounds filter and grid range of its box
//      (src/dense.cpp:1381-1410);
//   2. PtInCell (src/dense.cpp:1172-1203) of every box point: one lane per
//      line (y, z) of a box, the faces' y and z terms computed once for the
//      line's points, the verdicts left as one 32-bit word per line;
//   3. one lane per cell: the scanline state machine
//      (src/dense.cpp:1475-1701) on those words, with the runs it finds left as
//      one word per line;
//   4. the points of all runs go into one list, a lane per point deposits
//      mass/N (src/dense.cpp:1692); cells without a point deposit their site by CIC,
//      one lane per corner (src/dense.cpp:1787-1872).
// A wave on one cell runs steps 3 and 4 on one lane's worth of work: at
// 2.1M cells on 256^3 (31 box points in 10 lines, 8 deposited) it took about
// 750 vector and 640 scalar instructions a cell.
//
// A verdict is the same function of the same float operations as the point by
// point one: inside iff no face has d > eps or none has d < -eps (eps >= 0),
// held as the largest and smallest d.  Larger boxes go to a list for
// k_cell_scan_big, one wave per cell: with up to 256 lines of 32 points in the
// tiles, those in a cluster's sparse surroundings held their workgroups
// while the others had finished (57k cells of 8 Plummer blocks on 128^3: 870 us).
#include "kernels.hpp"
#include "geom.hpp"
#include "deposit.hpp"
#include "scan_bits.hpp"
#include "scan_deposit.hpp"
#include "scan_lines.hpp"

#include <algorithm>

namespace t2 {

namespace {

constexpr int SC_ROWS = 1024;        // lines per batch of cells
constexpr int SC_FACES = 1088;       // faces per batch (a tile has about 1000)
constexpr int SC_ROWS_MOST = 64;     // lines per cell, and
constexpr int SC_LINE_MOST = 16;     // points per line
constexpr int SC_POINTS = 8192;      // deposits per turn (their list overlays the planes)
constexpr int DEP = 4;               // deposits a lane has in flight

struct ScanShared {
    float4 fa[SC_FACES];             // planes {n, f0.x}
    float2 fb[SC_FACES];             // {f0.y, f0.z}
    unsigned row[SC_ROWS];           // verdicts of a line
    unsigned run[SC_ROWS];           // the run found on it
    unsigned char rcell[SC_ROWS];    // its cell in the tile
    int cmi[3][CELL_TILE];           // first grid index of a cell's box
    unsigned n[CELL_TILE];           // its points per axis, a byte each
    int roff[CELL_TILE];             // its first line
    int foff[CELL_TILE];             // its first face
    unsigned char nf[CELL_TILE];     // its faces
    unsigned char cic[CELL_TILE];    // the batch's cells without a point
    int v[CELL_TILE];
    float mpp[CELL_TILE];            // mass per point
    int pbase[CELL_TILE];            // its first point among the batch's
    int c1, rows, points, ncic;
    unsigned nlist, list0;           // list entries of a turn, the first one's place
    unsigned off[2];                 // points dropped, routed to another block
};

}  // namespace

template <bool MULTI>
__global__ __launch_bounds__(256) void k_cell_scan(CellSet<MULTI> set, PlaneBuf pb)
{
    __shared__ ScanShared sh;
    unsigned short *list = reinterpret_cast<unsigned short *>(sh.fa);   // [SC_POINTS]
    static_assert(SC_POINTS * 2 <= sizeof(sh.fa), "the list overlays the planes");
    static_assert(SC_ROWS <= 2048, "a list entry holds a line's number above five bits");
    const int t = xcd_item((int)blockIdx.x, set.ntiles);
    if (t < 0) return;
    const CellTile tile = set.tile(t);
    const GridP &gp = set.grid(tile.block);
    const CellOut o = set.out(tile.block);
    const BlockIn &in = set.in(tile.block);
    const int tid = (int)threadIdx.x, lane = tid & 63, w = tid >> 6;

    if (tid < 2) sh.off[tid] = 0u;
    if (tid == 2) sh.nlist = 0u;

    // ---- 1. one lane per cell: filter and grid range -------------------------
    int rows = 0, faces = 0;   // wave 0
    if (w == 0) {
        float4 h0 = make_float4(0.0f, 0.0f, 0.0f, 0.0f), h1 = h0;
        if (lane < tile.count) {
            h0 = pb.hdr[2 * ((long long)tile.base + lane)];
            h1 = pb.hdr[2 * ((long long)tile.base + lane) + 1];
        }
        const int F = __float_as_int(h0.w), v = __float_as_int(h1.w);
        bool live = F > 0;
        if (live) {
            const int code = box_status(h0.x, h0.y, h0.z, h1.x, h1.y, h1.z, gp);
            if (code != ST_SCAN) {
                o.status[v] = code;
                o.npts[v] = 0;
                live = false;
            }
        }
        bool big = false;
        if (live) {
            const int c0 = phys2idx1(h0.x, gp.step[0], gp.gmin[0]);
            const int c1 = phys2idx1(h0.y, gp.step[1], gp.gmin[1]);
            const int c2 = phys2idx1(h0.z, gp.step[2], gp.gmin[2]);
            const int n0 = phys2idx1(h1.x, gp.step[0], gp.gmin[0]) - c0 + 1;
            const int n1 = phys2idx1(h1.y, gp.step[1], gp.gmin[1]) - c1 + 1;
            const int n2 = phys2idx1(h1.z, gp.step[2], gp.gmin[2]) - c2 + 1;
            big = n0 < 1 || n1 < 1 || n2 < 1 || n0 > SC_LINE_MOST || n1 > SC_ROWS_MOST ||
                  n2 > SC_ROWS_MOST || n1 * n2 > SC_ROWS_MOST;
            if (!big) {
                sh.cmi[0][lane] = c0;
                sh.cmi[1][lane] = c1;
                sh.cmi[2][lane] = c2;
                sh.n[lane] = (unsigned)n0 | ((unsigned)n1 << 8) | ((unsigned)n2 << 16);
                sh.v[lane] = v;
                sh.nf[lane] = (unsigned char)F;
                rows = n1 * n2;
                faces = F;
            }
        }
        const unsigned long long bm = __ballot(big);
        if (bm) {
            const int leader = __ffsll(bm) - 1;
            unsigned at = 0;
            if (lane == leader) at = atomicAdd(pb.nbig, (unsigned)__popcll(bm));
            at = __shfl(at, leader) + (unsigned)__popcll(bm & ((1ull << lane) - 1ull));
            if (big) pb.big[at] = make_int2(tile.block, tile.base + lane);
        }
    }
    int pr = rows, pf = faces;   // wave 0: inclusive prefixes over the tile's cells
    if (w == 0)
        for (int off = 1; off < 64; off <<= 1) {
            const int a = __shfl_up(pr, off), b = __shfl_up(pf, off);
            if (lane >= off) {
                pr += a;
                pf += b;
            }
        }

    const float mass = gp.mass, eps = gp.eps;
    for (int c0 = 0; c0 < tile.count;) {
        // ---- the next cells whose lines and faces fit ------------------------
        if (w == 0) {
            const int r0 = c0 ? __shfl(pr, c0 - 1) : 0, f0 = c0 ? __shfl(pf, c0 - 1) : 0;
            const bool fits = lane < c0 || (pr - r0 <= SC_ROWS && pf - f0 <= SC_FACES);
            const unsigned long long nm = __ballot(!fits);
            const int c1 = nm ? __ffsll(nm) - 1 : 64;
            const int ro = pr - rows - r0, fo = pf - faces - f0;
            const bool on = lane >= c0 && lane < c1;
            if (on) {
                sh.roff[lane] = ro;
                sh.foff[lane] = fo;
                if (rows == 0) sh.nf[lane] = 0;
            }
            const int R = __shfl(pr, c1 - 1) - r0;
            if (lane == 0) {
                sh.c1 = c1;
                sh.rows = R;
                sh.ncic = 0;
            }
            if (on)
                for (int i = 0; i < rows; ++i) sh.rcell[ro + i] = (unsigned char)lane;
        }
        __syncthreads();
        const int c1 = sh.c1, R = sh.rows;
        // planes of the batch: half a wave per cell
        for (int c = c0 + 2 * w + (lane >> 5); c < c1; c += 8) {
            const int f = lane & 31;
            if (f < (int)sh.nf[c]) {
                const long long at = ((long long)tile.base + c) * PLANE_STRIDE + f;
                sh.fa[sh.foff[c] + f] = pb.fa[at];
                sh.fb[sh.foff[c] + f] = pb.fb[at];
            }
        }
        for (int i = tid; i < R; i += 256) sh.run[i] = 0u;
        __syncthreads();

        // ---- 2. verdicts, one lane per line ----------------------------------
        for (int i0 = w * 64; i0 < R; i0 += 256) {
            const int i = i0 + lane;
            const int r = i < R ? i : R - 1;   // idle lanes repeat the last line
            const int c = sh.rcell[r];
            const unsigned n = sh.n[c];
            const int n0 = (int)(n & 255u), n1 = (int)((n >> 8) & 255u);
            const int q = r - sh.roff[c];
            // q / n1 by the float reciprocal: exact for q < 256
            const int z = (int)(((float)q + 0.5f) * (1.0f / (float)n1)), y = q - z * n1;
            const float p0 = idx2phys1(sh.cmi[0][c], gp.step[0], gp.gmin[0]);
            const float qy = idx2phys1(sh.cmi[1][c], gp.step[1], gp.gmin[1]) +
                             (float)y * gp.step[1];
            const float qz = idx2phys1(sh.cmi[2][c], gp.step[2], gp.gmin[2]) +
                             (float)z * gp.step[2];
            const int nf = sh.nf[c];
            const float4 *fa = sh.fa + sh.foff[c];
            const float2 *fb = sh.fb + sh.foff[c];
            int nfmax = nf, nmax = n0;
            for (int off = 32; off >= 1; off >>= 1) {
                nfmax = max(nfmax, __shfl_xor(nfmax, off));
                nmax = max(nmax, __shfl_xor(nmax, off));
            }
            nfmax = __builtin_amdgcn_readfirstlane(nfmax);
            nmax = __builtin_amdgcn_readfirstlane(nmax);
            // points per turn by the wave's longest line
            unsigned m;
            if (nmax <= 3)
                m = line_verdicts<3>(fa, fb, nf, nfmax, p0, gp.step[0], 0, qy, qz, eps);
            else if (nmax <= 4)
                m = line_verdicts<4>(fa, fb, nf, nfmax, p0, gp.step[0], 0, qy, qz, eps);
            else {
                m = 0;
                for (int x0 = 0; x0 < nmax; x0 += 6)
                    m |= line_verdicts<6>(fa, fb, nf, nfmax, p0, gp.step[0], x0, qy, qz, eps)
                         << x0;
            }
            m &= n0 >= 32 ? ~0u : (1u << n0) - 1u;
            if (i < R) sh.row[i] = m;
        }
        __syncthreads();

        // ---- 3. one lane per cell: the scanline state machine ------------------
        if (w == 0) {
            const bool on = lane >= c0 && lane < c1 && rows > 0;
            const unsigned n = on ? sh.n[lane] : 0x010101u;
            const int n0 = (int)(n & 255u), n1 = (int)((n >> 8) & 255u), n2 = (int)(n >> 16);
            const int off = on ? sh.roff[lane] : 0;
            const int tot = on ? scan_rows(sh.row + off, sh.run + off, n0, n1, n2) : 0;
            if (on) {
                const int v = sh.v[lane];
                if (tot > 0) sh.mpp[lane] = mass / (float)tot;   // src/dense.cpp:1692
                o.status[v] = tot > 0 ? ST_SCAN : ST_CIC;
                o.npts[v] = tot > 0 ? tot : 8;
            }
            int pt = on ? tot : 0;
            for (int i = 1; i < 64; i <<= 1) {
                const int a = __shfl_up(pt, i);
                if (lane >= i) pt += a;
            }
            if (on) sh.pbase[lane] = pt - tot;
            if (lane == 63) sh.points = pt;
            const unsigned long long cm = __ballot(on && tot == 0);
            if (on && tot == 0) sh.cic[__popcll(cm & ((1ull << lane) - 1ull))] = (unsigned char)lane;
            if (lane == 0) sh.ncic = __popcll(cm);
        }
        __syncthreads();

        // ---- 4. deposit --------------------------------------------------------
        // the points of all runs in one list over the planes (line and x of
        // each), then a lane per point: a deposit waits for the count its
        // atomic returns, so each lane sends DEP of them before it waits
        const int P = sh.points;
        for (int w0 = 0; w0 < P; w0 += SC_POINTS) {
            for (int r = tid; r < R; r += 256) {
                const unsigned run = sh.run[r];
                if (!run) continue;
                const int x0 = row_low(run), len = __popc(run);
                const int at = sh.pbase[sh.rcell[r]] + (int)sh.row[r] - w0;
                for (int i = 0; i < len; ++i)
                    if (at + i >= 0 && at + i < SC_POINTS)
                        list[at + i] = (unsigned short)(r << 5 | (x0 + i));
            }
            __syncthreads();
            const int wn = min(P - w0, SC_POINTS);
            for (int p0 = 0; p0 < wn; p0 += DEP * 256) {
                long long at[DEP];
                unsigned cnt[DEP], key[DEP], li[DEP];
                float m[DEP];
#pragma unroll
                for (int d = 0; d < DEP; ++d) {
                    const int p = p0 + d * 256 + tid;
                    at[d] = -1;
                    if (p < wn) {
                        const unsigned e = list[p];
                        const int r = (int)(e >> 5), x = (int)(e & 31u), c = sh.rcell[r];
                        const int n1 = (int)((sh.n[c] >> 8) & 255u);
                        const int q = r - sh.roff[c];
                        const int z = (int)(((float)q + 0.5f) * (1.0f / (float)n1)),
                                  y = q - z * n1;
                        key[d] = cell_key(sh.v[c], 0);
                        m[d] = sh.mpp[c];
                        const int gx = sh.cmi[0][c] + x, gy = sh.cmi[1][c] + y,
                                  gz = sh.cmi[2][c] + z;
                        at[d] = own_lidx(gx, gy, gz, gp);
                        if (at[d] < 0)
                            atomicAdd(&sh.off[route_point(gx, gy, gz, m[d], key[d], set.router(),
                                                          tile.block)], 1u);
                        else
                            cnt[d] = atomicAdd(&o.count[at[d]], 1u);
                    }
                }
                // the turn's list entries in one reservation
#pragma unroll
                for (int d = 0; d < DEP; ++d) {
                    li[d] = ~0u;
                    if (at[d] >= 0 && store_point(at[d], cnt[d], m[d], key[d], gp.div, o))
                        li[d] = atomicAdd(&sh.nlist, 1u);
                }
                __syncthreads();
                const unsigned nlist = sh.nlist;
                if (nlist) {
                    if (tid == 0) sh.list0 = atomicAdd(&o.ctrs[C_OVF], nlist);
                    __syncthreads();
#pragma unroll
                    for (int d = 0; d < DEP; ++d)
                        if (li[d] != ~0u)
                            list_point(sh.list0 + li[d], at[d], cnt[d], m[d], key[d], o);
                    if (tid == 0) sh.nlist = 0u;
                }
                __syncthreads();
            }
        }
        const int ncic = sh.ncic;
        for (int i0 = w * 64; i0 < 8 * ncic; i0 += 256) {
            const int i = i0 + lane, k = lane & 7;
            const int v = sh.v[sh.cic[min(i >> 3, ncic - 1)]];
            int mn[3];
            const float m = cic_corner(in.pts[v], mass, gp, k, mn);
            long long at[1] = {-1};
            const float m1[1] = {m};
            const unsigned key[1] = {cell_key(v, gp.project ? (k >> 2) : 0)};
            if (i < 8 * ncic) {
                const int gx = mn[0] + (k & 1), gy = mn[1] + ((k >> 1) & 1), gz = mn[2] + (k >> 2);
                at[0] = own_lidx(gx, gy, gz, gp);
                if (at[0] < 0)
                    atomicAdd(&sh.off[route_point(gx, gy, gz, m, key[0], set.router(),
                                                  tile.block)], 1u);
            }
            wave_push<1>(at, m1, key, gp.div, o);
        }
        __syncthreads();
        c0 = c1;
    }
    if (tid < 2 && sh.off[tid]) atomicAdd(&o.ctrs[tid ? C_ROUTED : C_OFFBLOCK], sh.off[tid]);
}

// the listed cells, one wave per cell: by lines, or (very large boxes) with
// line windows and face-parallel probes
template <bool MULTI>
__global__ __launch_bounds__(64) void k_cell_scan_big(CellSet<MULTI> set, PlaneBuf pb)
{
    constexpr int RMAX = 64;
    static_assert(alignof(LineShared) >= alignof(int4) &&
                      sizeof(LineShared::row) >= RMAX * sizeof(int4),
                  "the runs overlay the lines");
    __shared__ LineShared sl;
    __shared__ float4 s_fa[PLANE_STRIDE];
    __shared__ float2 s_fb[PLANE_STRIDE];
    const int lane = (int)(threadIdx.x & 63);
    const unsigned n = *pb.nbig;
    for (unsigned i = blockIdx.x; i < n; i += gridDim.x) {
        const int2 q = pb.big[i];
        const float4 h0 = pb.hdr[2 * (long long)q.y], h1 = pb.hdr[2 * (long long)q.y + 1];
        const int F = __builtin_amdgcn_readfirstlane(__float_as_int(h0.w));
        const int v = __builtin_amdgcn_readfirstlane(__float_as_int(h1.w));
        float nx[1] = {0.0f}, ny[1] = {0.0f}, nz[1] = {0.0f};
        float fx[1] = {0.0f}, fy[1] = {0.0f}, fz[1] = {0.0f};
        if (lane < F) {
            const float4 a = pb.fa[(long long)q.y * PLANE_STRIDE + lane];
            const float2 b = pb.fb[(long long)q.y * PLANE_STRIDE + lane];
            s_fa[lane] = a;
            s_fb[lane] = b;
            nx[0] = a.x;
            ny[0] = a.y;
            nz[0] = a.z;
            fx[0] = a.w;
            fy[0] = b.x;
            fz[0] = b.y;
        }
        __syncthreads();
        const CellOut o = set.out(q.x);
        const GridP &gp = set.grid(q.x);
        const float4 site = set.in(q.x).pts[v];
        if (!scan_cell_lines(v, site, F, s_fa, s_fb, h0.x, h0.y, h0.z, h1.x, h1.y, h1.z, gp, o,
                             set.router(), q.x, sl))
            scan_deposit<1, RMAX, false, true>(v, site, F, nx, ny, nz, fx, fy, fz, h0.x, h0.y,
                                               h0.z, h1.x, h1.y, h1.z, gp, o, set.router(), q.x,
                                               s_fa, s_fb, true,
                                               reinterpret_cast<int4 *>(sl.row));
        __syncthreads();
    }
}

template <bool MULTI>
static void launch_scan(const CellSet<MULTI> &set, const PlaneBuf &pb, hipStream_t s)
{
    if (set.ntiles <= 0) return;
    hipLaunchKernelGGL((k_cell_scan<MULTI>), dim3(xcd_grid(set.ntiles)), dim3(256), 0, s, set, pb);
    hipLaunchKernelGGL((k_cell_scan_big<MULTI>), dim3(std::min(4096, set.ntiles * CELL_TILE)),
                       dim3(64), 0, s, set, pb);
}

void launch_cell_scan(const CellSet<false> &set, const PlaneBuf &pb, hipStream_t s)
{
    launch_scan<false>(set, pb, s);
}

void launch_cell_scan(const CellSet<true> &set, const PlaneBuf &pb, hipStream_t s)
{
    launch_scan<true>(set, pb, s);
}

}  // namespace t2
