// stage.hip -- device side of staging: range checks, bounding box, Morton
// order of the cells and tets, renumbering.
//
// A block arrives as the caller's arrays (one copy each); everything staging
// does to them is a device pass here: cells in Morton order of their sites
// (a stable radix sort of (key, id) pairs whose ids start ascending, so that
// ties stay in id order; ghosts after all originals), tets renumbered by
// their lowest-ranked vertex, in no set order among one vertex's.
//
// What bounds it: a block is read and written a few times (the tets: range
// check 32 B, keys 16 B + 16 B of gathered ranks and an atomic, renumbering
// 32 B in and out and 16 B of gathered numbers), which takes less than its
// copy over PCIe (32 B per tet at ~40 GB/s).  Small blocks are bound by the
// ~19 launches of about 3 us (with a sort of the tets and 4096-pair tiles 33;
// whole calls: volume() of 64,000 particles 1115 against 1029 us, 32,000
// particles on 64^3 1058 against 991).
#include "kernels.hpp"

#include <algorithm>

namespace t2 {

// One pass over the caller's arrays: xyz triples -> padded float4, the
// bounding box, and the index ranges (every tet vertex in [0, np), every
// neighbour and vert_to_tet entry in [-1, nt)).  Each workgroup leaves one
// record, which the host combines: six atomics per wave on one line instead
// took 8 ns each (1.3M tets: 217 us, of which the loads are about 15).
__global__ __launch_bounds__(256) void k_stage_check(const float *__restrict__ xyz, int np,
                                                     const int4 *__restrict__ tets, int nt,
                                                     const int *__restrict__ v2t,
                                                     float4 *__restrict__ pts,
                                                     StageInfo *__restrict__ info)
{
    __shared__ float s_lo[4][3], s_hi[4][3];
    __shared__ unsigned s_bad[4], s_odd[4];
    const int stride = (int)(gridDim.x * blockDim.x);
    const int i0 = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    bool bad = false, odd = false;
    float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (long long p = i0; p < np; p += stride) {
        const float x = xyz[3 * p], y = xyz[3 * p + 1], z = xyz[3 * p + 2];
        pts[p] = make_float4(x, y, z, 0.0f);
        const int t = v2t[p];
        bad = bad || t < -1 || t >= nt;
        odd = odd || !(fabsf(x) < INFINITY) || !(fabsf(y) < INFINITY) || !(fabsf(z) < INFINITY);
        lo[0] = fminf(lo[0], x);
        lo[1] = fminf(lo[1], y);
        lo[2] = fminf(lo[2], z);
        hi[0] = fmaxf(hi[0], x);
        hi[1] = fmaxf(hi[1], y);
        hi[2] = fmaxf(hi[2], z);
    }
    for (long long t = i0; t < nt; t += stride) {
        const int4 v = tets[2 * t], n = tets[2 * t + 1];
        bad = bad || (unsigned)v.x >= (unsigned)np || (unsigned)v.y >= (unsigned)np ||
              (unsigned)v.z >= (unsigned)np || (unsigned)v.w >= (unsigned)np ||
              n.x < -1 || n.x >= nt || n.y < -1 || n.y >= nt || n.z < -1 || n.z >= nt ||
              n.w < -1 || n.w >= nt;
    }
    for (int off = 32; off >= 1; off >>= 1)
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            lo[a] = fminf(lo[a], __shfl_xor(lo[a], off));
            hi[a] = fmaxf(hi[a], __shfl_xor(hi[a], off));
        }
    const bool any_bad = __ballot(bad) != 0ull, any_odd = __ballot(odd) != 0ull;
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        s_bad[w] = any_bad;
        s_odd[w] = any_odd;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            s_lo[w][a] = lo[a];
            s_hi[w][a] = hi[a];
        }
    }
    __syncthreads();
    StageInfo &out = info[blockIdx.x];
    if (threadIdx.x < 3) {
        const int a = threadIdx.x;
        out.lo[a] = fminf(fminf(s_lo[0][a], s_lo[1][a]), fminf(s_lo[2][a], s_lo[3][a]));
        out.hi[a] = fmaxf(fmaxf(s_hi[0][a], s_hi[1][a]), fmaxf(s_hi[2][a], s_hi[3][a]));
    }
    if (threadIdx.x == 3) out.err = s_bad[0] | s_bad[1] | s_bad[2] | s_bad[3];
    if (threadIdx.x == 4) out.nonfinite = s_odd[0] | s_odd[1] | s_odd[2] | s_odd[3];
}

int launch_stage_check(const float *xyz, int np, const int4 *tets, int nt, const int *v2t,
                       float4 *pts, StageInfo *info, hipStream_t s)
{
    const int n = std::max(np, nt);
    if (n <= 0) return 0;
    const int nb = std::min((int)STAGE_RECORDS, (n + 255) / 256);
    hipLaunchKernelGGL(k_stage_check, dim3(nb), dim3(256), 0, s, xyz, np, tets, nt, v2t, pts,
                       info);
    return nb;
}

// ---------------------------------------------------------------------------
// exclusive scan of n unsigned counts, in place
// ---------------------------------------------------------------------------
constexpr unsigned SCAN_TILE = 4096;   // 1024 lanes of four
constexpr unsigned SCAN_MOST = 16;     // entries per lane of the one-workgroup scan

// inclusive prefix sums over a wave in six additions (rows of 16 by shifts,
// then the last lane of rows 0 and 2 into 1 and 3, of row 1 into 2 and 3)
__device__ __forceinline__ unsigned wave_scan(unsigned x)
{
    x += (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xf, 0xf, false);
    x += (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xf, 0xf, false);
    x += (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xf, 0xf, false);
    x += (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xf, 0xf, false);
    x += (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xa, 0xf, false);
    x += (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xc, 0xf, false);
    return x;
}

// Exclusive scan of a[0 .. n) by a workgroup of 16 waves, n <= 1024 * per and
// per <= ROWS: each wave takes per * 64 neighbouring entries as per coalesced
// rows, scans them independently of each other, and the 16 waves' totals meet
// in LDS.  (Each lane reading its own per entries in a row instead touches a
// cache line per entry: 14,000 entries in one workgroup 11.7 against 3.8 us.)
// Returns the total.
template <unsigned ROWS>
__device__ __forceinline__ unsigned scan_1024(unsigned *__restrict__ a, unsigned n, unsigned per)
{
    __shared__ unsigned s_w[16];
    const unsigned lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const unsigned i0 = w * per * 64 + lane;
    unsigned v[ROWS], x[ROWS];
#pragma unroll
    for (unsigned k = 0; k < ROWS; ++k) {
        const unsigned i = i0 + k * 64;
        v[k] = x[k] = (k < per && i < n) ? a[i] : 0u;
    }
    unsigned run = 0;
#pragma unroll
    for (unsigned k = 0; k < ROWS; ++k) {
        x[k] = wave_scan(x[k]);
        v[k] = run + x[k] - v[k];
        run += (unsigned)__builtin_amdgcn_readlane((int)x[k], 63);
    }
    if (lane == 0) s_w[w] = run;
    __syncthreads();
    unsigned base = 0, all = 0;
#pragma unroll
    for (unsigned i = 0; i < 16; ++i) {
        const unsigned t = s_w[i];
        base += i < w ? t : 0u;
        all += t;
    }
#pragma unroll
    for (unsigned k = 0; k < ROWS; ++k) {
        const unsigned i = i0 + k * 64;
        if (k < per && i < n) a[i] = base + v[k];
    }
    return all;
}

__global__ __launch_bounds__(1024) void k_scan_tiles(unsigned *__restrict__ a, unsigned n,
                                                     unsigned *__restrict__ sums)
{
    const unsigned i0 = blockIdx.x * SCAN_TILE;
    const unsigned total = scan_1024<4>(a + i0, min(n - i0, (unsigned)SCAN_TILE), 4);
    if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

// one workgroup over n <= 1024 * ROWS entries
template <unsigned ROWS>
__global__ __launch_bounds__(1024) void k_scan_one(unsigned *__restrict__ a, unsigned n)
{
    scan_1024<ROWS>(a, n, (n + 1023) / 1024);
}

static void scan_one(unsigned *a, unsigned n, hipStream_t s)
{
    if (n <= 4096)
        hipLaunchKernelGGL((k_scan_one<4>), dim3(1), dim3(1024), 0, s, a, n);
    else
        hipLaunchKernelGGL((k_scan_one<SCAN_MOST>), dim3(1), dim3(1024), 0, s, a, n);
}

__global__ __launch_bounds__(1024) void k_scan_bases(unsigned *__restrict__ a, unsigned n,
                                                     const unsigned *__restrict__ sums)
{
    const unsigned base = sums[blockIdx.x];
    const unsigned i = blockIdx.x * SCAN_TILE + threadIdx.x;
#pragma unroll
    for (unsigned k = 0; k < 4; ++k)
        if (i + k * 1024 < n) a[i + k * 1024] += base;
}

// n up to 1024 * SCAN_MOST in one workgroup, else tiles and their sums
void launch_scan_u32(unsigned *a, unsigned n, unsigned *sums, hipStream_t s)
{
    if (n == 0) return;
    if (n <= 1024u * SCAN_MOST) {
        scan_one(a, n, s);
        return;
    }
    const unsigned tiles = (n + SCAN_TILE - 1) / SCAN_TILE;
    hipLaunchKernelGGL(k_scan_tiles, dim3(tiles), dim3(1024), 0, s, a, n, sums);
    launch_scan_u32(sums, tiles, sums + tiles, s);
    hipLaunchKernelGGL(k_scan_bases, dim3(tiles), dim3(1024), 0, s, a, n,
                       (const unsigned *)sums);
}

size_t scan_sums_words(size_t n)
{
    if (n <= 1024 * SCAN_MOST) return 0;
    const size_t tiles = (n + SCAN_TILE - 1) / SCAN_TILE;
    return tiles + scan_sums_words(tiles);
}

// ---------------------------------------------------------------------------
// stable radix sort of (key, id) pairs, 8 bits a pass.  A workgroup of four
// waves owns a tile of 256 * ROUNDS consecutive pairs, each wave a quarter of
// them in rounds of 64; hist is digit-major ([digit][tile]), so its exclusive
// scan gives each tile's first slot per digit.
// ---------------------------------------------------------------------------
template <int ROUNDS>
__global__ __launch_bounds__(256) void k_sort_hist(const unsigned *__restrict__ key, unsigned n,
                                                   int shift, unsigned *__restrict__ hist,
                                                   unsigned ntiles)
{
    __shared__ unsigned s_h[256];
    s_h[threadIdx.x] = 0u;
    __syncthreads();
    const unsigned base = blockIdx.x * (256 * ROUNDS);
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
        const unsigned i = base + r * 256 + threadIdx.x;
        if (i < n) atomicAdd(&s_h[(key[i] >> shift) & 255u], 1u);
    }
    __syncthreads();
    hist[threadIdx.x * ntiles + blockIdx.x] = s_h[threadIdx.x];
}

// LAST: a pair's slot is its rank, id_out takes the ids of the first nfirst
// only
template <int ROUNDS, bool LAST>
__global__ __launch_bounds__(256) void k_sort_scatter(const unsigned *__restrict__ key,
                                                      const unsigned *__restrict__ id,
                                                      unsigned n, int shift,
                                                      const unsigned *__restrict__ hist,
                                                      unsigned ntiles,
                                                      unsigned *__restrict__ key_out,
                                                      unsigned *__restrict__ id_out,
                                                      unsigned nfirst)
{
    __shared__ unsigned s_c[4][256];   // next slot per wave and digit
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const unsigned long long below = (1ull << lane) - 1ull;
#pragma unroll
    for (int i = 0; i < 4; ++i) s_c[i][threadIdx.x] = 0u;
    __syncthreads();
    const unsigned base = blockIdx.x * (256 * ROUNDS) + w * (64 * ROUNDS) + lane;
    unsigned k[ROUNDS], v[ROUNDS];
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
        const unsigned i = base + r * 64;
        k[r] = i < n ? key[i] : 0u;
        v[r] = i < n ? id[i] : 0u;
        if (i < n) atomicAdd(&s_c[w][(k[r] >> shift) & 255u], 1u);
    }
    __syncthreads();
    {
        unsigned b = hist[threadIdx.x * ntiles + blockIdx.x];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const unsigned c = s_c[i][threadIdx.x];
            s_c[i][threadIdx.x] = b;
            b += c;
        }
    }
    __syncthreads();
    // a wave's rounds in order; within a round, the lanes of one digit take
    // consecutive slots in lane order (only this wave touches s_c[w])
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
        const unsigned i = base + r * 64;
        const bool on = i < n;
        const unsigned d = (k[r] >> shift) & 255u;
        unsigned long long same = __ballot(on);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const unsigned long long m = __ballot((d >> b) & 1u);
            same &= ((d >> b) & 1u) ? m : ~m;
        }
        if (on) {
            const unsigned slot = s_c[w][d] + (unsigned)__popcll(same & below);
            if (LAST) {
                key_out[v[r]] = slot;
                if (slot < nfirst) id_out[slot] = v[r];
            } else {
                key_out[slot] = k[r];
                id_out[slot] = v[r];
            }
        }
        wave_sync();   // every lane has read its counter
        if (on && (same & below) == 0ull) s_c[w][d] += (unsigned)__popcll(same);
        wave_sync();
    }
}

// rank of each of n ids in the order of their 32-bit keys (k0 / v0), and the
// first nfirst ids in it; k1 / v1: as much scratch
template <int ROUNDS>
static void radix_rank(unsigned *k0, unsigned *v0, unsigned *k1, unsigned *v1, unsigned n,
                       unsigned *rank, unsigned *first, unsigned nfirst, unsigned *hist,
                       unsigned *sums, hipStream_t s)
{
    const unsigned tiles = (n + 256 * ROUNDS - 1) / (256 * ROUNDS);
    for (int shift = 0; shift < 32; shift += 8) {
        hipLaunchKernelGGL((k_sort_hist<ROUNDS>), dim3(tiles), dim3(256), 0, s,
                           (const unsigned *)k0, n, shift, hist, tiles);
        launch_scan_u32(hist, 256 * tiles, sums, s);
        if (shift < 24)
            hipLaunchKernelGGL((k_sort_scatter<ROUNDS, false>), dim3(tiles), dim3(256), 0, s,
                               (const unsigned *)k0, (const unsigned *)v0, n, shift,
                               (const unsigned *)hist, tiles, k1, v1, 0u);
        else
            hipLaunchKernelGGL((k_sort_scatter<ROUNDS, true>), dim3(tiles), dim3(256), 0, s,
                               (const unsigned *)k0, (const unsigned *)v0, n, shift,
                               (const unsigned *)hist, tiles, rank, first, nfirst);
        std::swap(k0, k1);
        std::swap(v0, v1);
    }
}

// 16 rounds of 64 pairs a wave, fewer where the chip would be idle and the
// 256 counts a tile still fit the one-workgroup scan: 42,000 pairs in 11
// workgroups of 4096 took 22 us a pass, in 42 of 1024 12
static int sort_rounds(int n) { return n <= 65536 ? 4 : (n <= 131072 ? 8 : 16); }

// ---------------------------------------------------------------------------
// Morton layout
// ---------------------------------------------------------------------------
__device__ __forceinline__ unsigned spread3(unsigned x)
{
    x &= 0x3ffu;
    x = (x | (x << 16)) & 0x030000FFu;
    x = (x | (x << 8)) & 0x0300F00Fu;
    x = (x | (x << 4)) & 0x030C30C3u;
    x = (x | (x << 2)) & 0x09249249u;
    return x;
}

// Morton keys of 10 bits an axis, originals before ghosts; ntet: zeroed
__global__ void k_morton_keys(const float4 *__restrict__ pts, int np, int norig, StageBox box,
                              unsigned *__restrict__ key, unsigned *__restrict__ id,
                              unsigned *__restrict__ ntet)
{
    const int p = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (p >= np) return;
    const float4 a = pts[p];
    const float x[3] = {a.x, a.y, a.z};
    unsigned q[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const double ext = (double)box.hi[i] - (double)box.lo[i];
        const double f = ext > 0 ? ((double)x[i] - (double)box.lo[i]) / ext : 0.0;
        double g = f * 1023.0;
        g = g > 0.0 ? g : 0.0;         // NaN to 0
        g = g < 1023.0 ? g : 1023.0;
        q[i] = (unsigned)g;
    }
    key[p] = spread3(q[0]) | (spread3(q[1]) << 1) | (spread3(q[2]) << 2) |
             (p < norig ? 0u : 1u << 30);
    id[p] = (unsigned)p;
    ntet[p] = 0u;
}

// each tet's first-ranked vertex (an original when it has one), and the tet's
// place among that vertex's (in no set order: no result depends on it).  One
// atomic per tet bounds it, 13.5M in 691 us; a stable sort by that vertex, a
// histogram, scan and scatter per 8 bits, took 744 and 256,000 tets 100
// against 40 with the scan
__global__ void k_tet_keys(const int4 *__restrict__ tets, int nt,
                           const unsigned *__restrict__ rank, unsigned *__restrict__ ntet,
                           uint2 *__restrict__ key)
{
    const int t = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (t >= nt) return;
    const int4 v = tets[2 * (long long)t];
    const unsigned r = min(min(rank[v.x], rank[v.y]), min(rank[v.z], rank[v.w]));
    key[t] = make_uint2(r, atomicAdd(&ntet[r], 1u));
}

__global__ void k_tet_new(const uint2 *__restrict__ key, const unsigned *__restrict__ start,
                          int nt, int *__restrict__ tnew, unsigned *__restrict__ id)
{
    const int t = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (t >= nt) return;
    const uint2 k = key[t];
    const unsigned m = start[k.x] + k.y;
    tnew[t] = (int)m;
    id[m] = (unsigned)t;
}

// tets in their new order with renumbered neighbours, vert_to_tet renumbered.
// Gathers by new id: by old id, scattering 32-byte records, 13.5M tets take
// 851 against 640 us
__global__ void k_renumber(const unsigned *__restrict__ id, int nt,
                           const int *__restrict__ tnew, const int4 *__restrict__ raw,
                           int4 *__restrict__ tets, const int *__restrict__ v2t_raw, int np,
                           int *__restrict__ v2t)
{
    const long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k < nt) {
        const long long t = id[k];
        const int4 n = raw[2 * t + 1];
        tets[2 * k] = raw[2 * t];
        tets[2 * k + 1] = make_int4(n.x < 0 ? n.x : tnew[n.x], n.y < 0 ? n.y : tnew[n.y],
                                    n.z < 0 ? n.z : tnew[n.z], n.w < 0 ? n.w : tnew[n.w]);
    }
    if (k < np) {
        const int t = v2t_raw[k];
        v2t[k] = t < 0 ? t : tnew[t];
    }
}

// scratch of launch_layout in unsigned words: the ranks and the tets per rank,
// two key and two id arrays of the particles or three words per tet, the digit
// counts and scan sums
static size_t layout_sort_words(int np, int nt)
{
    return std::max<size_t>(4 * (size_t)np, 3 * (size_t)nt);
}
static size_t layout_hist_words(int np)
{
    const size_t tile = 256 * (size_t)sort_rounds(np);
    return 256 * ((np + tile - 1) / tile);
}
size_t layout_scratch_words(int np, int nt)
{
    const size_t h = layout_hist_words(np);
    return layout_sort_words(np, nt) + 2 * (size_t)np + h +
           scan_sums_words(std::max<size_t>(h, (size_t)np)) + 1;
}

void launch_layout(const float4 *pts, int np, int norig, const StageBox &box, const int4 *raw,
                   int nt, const int *v2t_raw, unsigned *scratch, int *order, int4 *tets,
                   int *v2t, int *tnew, hipStream_t s)
{
    if (np <= 0) return;   // no particles, no tets
    unsigned *k0 = scratch, *v0 = k0 + np, *k1 = v0 + np, *v1 = k1 + np;
    uint2 *tkey = reinterpret_cast<uint2 *>(scratch);   // when the sort is over
    unsigned *tid = scratch + 2 * (size_t)nt;
    unsigned *rank = scratch + layout_sort_words(np, nt), *ntet = rank + np, *hist = ntet + np,
             *sums = hist + layout_hist_words(np);
    hipLaunchKernelGGL(k_morton_keys, dim3((np + 255) / 256), dim3(256), 0, s, pts, np, norig,
                       box, k0, v0, ntet);
    unsigned *first = reinterpret_cast<unsigned *>(order);
    const int rounds = sort_rounds(np);
    (rounds == 4 ? radix_rank<4> : (rounds == 8 ? radix_rank<8> : radix_rank<16>))(
        k0, v0, k1, v1, (unsigned)np, rank, first, (unsigned)norig, hist, sums, s);
    if (nt > 0) {
        const dim3 g((nt + 255) / 256);
        hipLaunchKernelGGL(k_tet_keys, g, dim3(256), 0, s, raw, nt, (const unsigned *)rank, ntet,
                           tkey);
        launch_scan_u32(ntet, (unsigned)np, sums, s);
        hipLaunchKernelGGL(k_tet_new, g, dim3(256), 0, s, (const uint2 *)tkey,
                           (const unsigned *)ntet, nt, tnew, tid);
    }
    const int m = std::max(np, nt);
    hipLaunchKernelGGL(k_renumber, dim3((m + 255) / 256), dim3(256), 0, s, (const unsigned *)tid, nt,
                       (const int *)tnew, raw, tets, v2t_raw, np, v2t);
}

// circumcenters as xyz triples in the caller's numbering (tnew null: the
// device numbering is the caller's)
__global__ void k_unpack_cc(const float4 *__restrict__ cc, const int *__restrict__ tnew, int nt,
                            float *__restrict__ out)
{
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nt) return;
    const float4 q = cc[tnew ? tnew[t] : (int)t];
    out[3 * t] = q.x;
    out[3 * t + 1] = q.y;
    out[3 * t + 2] = q.z;
}

void launch_unpack_cc(const float4 *cc, const int *tnew, int nt, float *out, hipStream_t s)
{
    if (nt <= 0) return;
    hipLaunchKernelGGL(k_unpack_cc, dim3((nt + 255) / 256), dim3(256), 0, s, cc, tnew, nt, out);
}

}  // namespace t2
