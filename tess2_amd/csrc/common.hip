// common.hip -- streaming kernels: circumcenters, fills, statistics.
#include "kernels.hpp"
#include "geom.hpp"

#include <algorithm>

namespace t2 {

// fill_circumcenters(): one lane per tet, src/volume.cpp:6-11.  The four
// vertex gathers are 16-byte loads of the padded particle array.
__global__ void k_circumcenters(const float4 *__restrict__ pts, const int4 *__restrict__ tets,
                                int ntets, float4 *__restrict__ cc)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= ntets) return;
    const int4 vv = tets[2 * t];
    const float4 a = pts[vv.x], b = pts[vv.y], c = pts[vv.z], d = pts[vv.w];
    float x, y, z;
    circumcenter(a.x, a.y, a.z, b.x, b.y, b.z, c.x, c.y, c.z, d.x, d.y, d.z, x, y, z);
    const float e = circumcenter_err(a.x, a.y, a.z, b.x, b.y, b.z, c.x, c.y, c.z, d.x, d.y, d.z,
                                     x, y, z);
    cc[t] = make_float4(x, y, z, e);
}

void launch_circumcenters(const float4 *pts, const int4 *tets, int ntets, float4 *cc,
                          hipStream_t s)
{
    if (ntets <= 0) return;
    hipLaunchKernelGGL(k_circumcenters, dim3((ntets + 255) / 256), dim3(256), 0, s, pts, tets,
                       ntets, cc);
}

// What a run starts with, in one launch: circumcenters of every staged block
// (workgroups below bt of row blockIdx.y = block), its density and count grids
// cleared, and up to four more arrays zeroed (first row).  Both halves are
// streams; apart they were three to six launches of ~4 us each (4,000 cells,
// exact assignment, 49^3, whole run with the fused last pass: 185 against
// 156 us).
__global__ __launch_bounds__(256) void k_run_prep(const BlockIn *__restrict__ ins,
                                                  const CellOut *__restrict__ outs, int bt,
                                                  ZeroList z)
{
    if ((int)blockIdx.x < bt) {
        const BlockIn &in = ins[blockIdx.y];
        for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < in.ntets; t += bt * blockDim.x) {
            const int4 vv = in.tets[2 * t];
            const float4 a = in.pts[vv.x], b = in.pts[vv.y], c = in.pts[vv.z], d = in.pts[vv.w];
            float x, y, z0;
            circumcenter(a.x, a.y, a.z, b.x, b.y, b.z, c.x, c.y, c.z, d.x, d.y, d.z, x, y, z0);
            const float e = circumcenter_err(a.x, a.y, a.z, b.x, b.y, b.z, c.x, c.y, c.z, d.x,
                                             d.y, d.z, x, y, z0);
            const_cast<float4 *>(in.cc)[t] = make_float4(x, y, z0, e);   // read-only downstream
        }
        return;
    }
    const CellOut &o = outs[blockIdx.y];
    const unsigned long long n = o.ngrid, n4 = n / 4;
    const unsigned long long stride = (unsigned long long)(gridDim.x - bt) * blockDim.x;
    const unsigned long long i0 = (unsigned long long)(blockIdx.x - bt) * blockDim.x + threadIdx.x;
    const uint4 zero = make_uint4(0u, 0u, 0u, 0u);
    for (unsigned long long i = i0; i < n4; i += stride) {
        reinterpret_cast<uint4 *>(o.density)[i] = zero;
        reinterpret_cast<uint4 *>(o.count)[i] = zero;
    }
    if (i0 < n - n4 * 4) {
        o.density[n4 * 4 + i0] = 0.0f;
        o.count[n4 * 4 + i0] = 0u;
    }
    if (blockIdx.y == 0)
#pragma unroll
        for (int k = 0; k < 4; ++k)
            for (unsigned long long i = i0; i < z.n[k]; i += stride) z.p[k][i] = 0u;
}

void launch_run_prep(const BlockIn *ins, const CellOut *outs, int nb, int max_tets,
                     unsigned long long max_grid, const ZeroList &z, hipStream_t s)
{
    if (nb <= 0) return;
    unsigned long long most = max_grid / 4;
    for (int k = 0; k < 4; ++k) most = std::max<unsigned long long>(most, z.n[k]);
    const unsigned bg = (unsigned)std::max<unsigned long long>(
        1, std::min<unsigned long long>(2048, (most + 255) / 256));
    const unsigned bt = (unsigned)std::min(16384, (max_tets + 255) / 256);
    hipLaunchKernelGGL(k_run_prep, dim3(bt + bg, nb), dim3(256), 0, s, ins, outs, (int)bt, z);
}

__global__ void k_fill_u32(uint4 *__restrict__ p4, size_t n4, unsigned *__restrict__ tail,
                           size_t ntail, unsigned v)
{
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    const uint4 q = make_uint4(v, v, v, v);
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += stride)
        p4[i] = q;
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < ntail) tail[i] = v;
}

// fill a 16-byte aligned buffer (a kernel rather than a memset so that the
// sequence stays valid inside a captured graph)
void launch_fill_u32(unsigned *p, size_t n, unsigned v, hipStream_t s)
{
    if (n == 0) return;
    const size_t n4 = n / 4, ntail = n - n4 * 4;
    size_t blocks = (n4 + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    if (blocks == 0) blocks = 1;
    hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)blocks), dim3(256), 0, s, (uint4 *)p, n4,
                       p + n4 * 4, ntail, v);
}

// One pass over a block that the caller keeps in device memory: xyz triples ->
// padded float4, circumcenters of its tets, zeroed counters, and the index
// ranges (every tet vertex in [0, np), every neighbour and vert_to_tet entry
// in [-1, nt)).  A tet is read only once its own indices are in range; a
// violation stores `token` in *stop, and the kernels behind this one that
// carry the token return at once.  One word that holds this call's token needs no
// clearing first, and no wait of the host between check and use.
__global__ void k_device_block(const float *__restrict__ xyz, int np,
                               const int4 *__restrict__ tets, int nt,
                               const int *__restrict__ v2t, float4 *__restrict__ pts,
                               float4 *__restrict__ cc, unsigned *__restrict__ ctrs,
                               unsigned *stop, unsigned token)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < C_NCTR) ctrs[i] = 0u;
    bool bad = false;
    if (i < np) {
        pts[i] = make_float4(xyz[3ll * i], xyz[3ll * i + 1], xyz[3ll * i + 2], 0.0f);
        const int t = v2t[i];
        bad = t < -1 || t >= nt;
    }
    if (i < nt) {
        const int4 v = tets[2ll * i], n = tets[2ll * i + 1];
        const bool out = (unsigned)v.x >= (unsigned)np || (unsigned)v.y >= (unsigned)np ||
                         (unsigned)v.z >= (unsigned)np || (unsigned)v.w >= (unsigned)np;
        bad = bad || out || n.x < -1 || n.x >= nt || n.y < -1 || n.y >= nt || n.z < -1 ||
              n.z >= nt || n.w < -1 || n.w >= nt;
        if (!out) {
            const float *a = xyz + 3ll * v.x, *b = xyz + 3ll * v.y, *c = xyz + 3ll * v.z,
                        *d = xyz + 3ll * v.w;
            float x, y, z;
            circumcenter(a[0], a[1], a[2], b[0], b[1], b[2], c[0], c[1], c[2], d[0], d[1], d[2],
                         x, y, z);
            cc[i] = make_float4(x, y, z, 0.0f);   // no error bound: volumes do not read it
        }
    }
    if (bad) *stop = token;
}

void launch_device_block(const float *xyz, int np, const int4 *tets, int nt, const int *v2t,
                         float4 *pts, float4 *cc, unsigned *ctrs, unsigned *stop, unsigned token,
                         hipStream_t s)
{
    const int n = std::max(std::max(np, nt), (int)C_NCTR);
    hipLaunchKernelGGL(k_device_block, dim3((n + 255) / 256), dim3(256), 0, s, xyz, np, tets, nt,
                       v2t, pts, cc, ctrs, stop, token);
}

// ---------------------------------------------------------------------------
// The end of a run, after the fold of points with three and more
// contributions: the points with exactly two (the common case: a point on
// the face between two cells) hold both next to the point and are added here,
// in the order the sort would give the pair (the second first unless its key
// is larger); sum and maximum of the density; cells per status and points
// of deposited cells.  Each workgroup leaves a record and k_run_stats combines
// them in a fixed order, so that the sum is the same on every run, without
// an atomic per workgroup on the block's counters.  A stream over count and
// density, bound by it and by the lines of first and second that hold pairs
// (16.8M points, 2M cells: 88 us; as passes of their own, pairs 78, sums 55
// and cells 21).  Four points per lane and iteration: a small grid is then
// over in one (117,000 points: 5 us, 8 with sixteen).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_run_finish(const CellOut *__restrict__ outs,
                                                    const GridP *__restrict__ gps,
                                                    RunPart *__restrict__ part, int bg)
{
    __shared__ double s_acc[4];
    __shared__ float s_mx[4];
    __shared__ unsigned long long s_c[4][6];
    const CellOut &o = outs[blockIdx.y];
    RunPart &out = part[(size_t)blockIdx.y * RUN_PARTS + blockIdx.x];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if ((int)blockIdx.x < bg) {
        const double dd = (double)gps[blockIdx.y].div;
        // 16-byte loads, four independent partial sums per lane (the grid
        // arrays are 256-byte aligned allocations); the last n mod 4 points
        // go to the first lanes of workgroup 0
        const unsigned long long n = o.ngrid, n4 = n >> 2;
        const unsigned *__restrict__ count = o.count;
        const uint2 *__restrict__ first = o.first, *__restrict__ second = o.second;
        float *__restrict__ density = o.density;
        auto pair = [&](uint2 f, uint2 q) {
            const bool sw = q.x > f.x;
            const unsigned m0 = sw ? f.y : q.y, m1 = sw ? q.y : f.y;
            const float x = (float)(0.0 + (double)__uint_as_float(m0) / dd);
            return (float)((double)x + (double)__uint_as_float(m1) / dd);
        };
        double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
        float mx = 0.0f;
        unsigned np = 0;
        for (unsigned long long i = (unsigned long long)blockIdx.x * 256 + threadIdx.x; i < n4;
             i += (unsigned long long)bg * 256) {
            const uint4 c4 = reinterpret_cast<const uint4 *>(count)[i];
            const float4 x4 = reinterpret_cast<const float4 *>(density)[i];
            const unsigned c[4] = {c4.x, c4.y, c4.z, c4.w};
            float x[4] = {x4.x, x4.y, x4.z, x4.w};
            uint2 f[4], q[4];
            bool any = false;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                f[k] = q[k] = make_uint2(0u, 0u);
                if (c[k] == 2u) {
                    f[k] = first[4 * i + k];
                    q[k] = second[4 * i + k];
                }
                any |= c[k] == 2u;
                np += c[k] >= 2u ? 1u : 0u;
            }
            if (any) {
#pragma unroll
                for (int k = 0; k < 4; ++k) x[k] = c[k] == 2u ? pair(f[k], q[k]) : x[k];
                reinterpret_cast<float4 *>(density)[i] = make_float4(x[0], x[1], x[2], x[3]);
            }
            a0 += (double)x[0];
            a1 += (double)x[1];
            a2 += (double)x[2];
            a3 += (double)x[3];
            mx = fmaxf(mx, fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])));
        }
        if (blockIdx.x == 0 && threadIdx.x < (unsigned)(n & 3ull)) {
            const unsigned long long g = (n4 << 2) + threadIdx.x;
            float x = density[g];
            if (count[g] == 2u) {
                x = pair(first[g], second[g]);
                density[g] = x;
            }
            np += count[g] >= 2u ? 1u : 0u;
            a0 += (double)x;
            mx = fmaxf(mx, x);
        }
        double acc = (a0 + a1) + (a2 + a3);
        for (int off = 32; off >= 1; off >>= 1) {
            acc += __shfl_xor(acc, off);
            mx = fmaxf(mx, __shfl_xor(mx, off));
            np += __shfl_xor(np, off);
        }
        if (lane == 0) {
            s_acc[w] = acc;
            s_mx[w] = mx;
            s_c[w][0] = np;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            out.sum = ((s_acc[0] + s_acc[1]) + s_acc[2]) + s_acc[3];
            out.mx = fmaxf(fmaxf(s_mx[0], s_mx[1]), fmaxf(s_mx[2], s_mx[3]));
            out.pairs = (unsigned)(s_c[0][0] + s_c[1][0] + s_c[2][0] + s_c[3][0]);
        }
        if (threadIdx.x < 6) out.c[threadIdx.x] = 0;
        return;
    }
    // cells per status counted by ballots (wave-uniform counters), points of
    // deposited cells summed per lane
    const int b = (int)blockIdx.x - bg, nbc = (int)gridDim.x - bg;
    unsigned long long c[5] = {0, 0, 0, 0, 0}, np = 0;
    for (int base = b * 256; base < o.ncells; base += nbc * 256) {
        const int i = base + threadIdx.x;
        int s = -1;
        if (i < o.ncells) {
            s = o.status[i];
            if (s == 0 || s == 1) np += (unsigned long long)o.npts[i];
        }
#pragma unroll
        for (int k = 0; k < 5; ++k) c[k] += (unsigned long long)__popcll(__ballot(s == k));
    }
    for (int off = 32; off >= 1; off >>= 1) np += __shfl_xor(np, off);
    if (lane == 0) {
#pragma unroll
        for (int k = 0; k < 5; ++k) s_c[w][k] = c[k];
        s_c[w][5] = np;
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        const int k = threadIdx.x;
        out.c[k] = s_c[0][k] + s_c[1][k] + s_c[2][k] + s_c[3][k];
    }
    if (threadIdx.x == 6) {
        out.sum = 0.0;
        out.mx = 0.0f;
        out.pairs = 0u;
    }
}

// one workgroup per block: its records into its statistics, four lanes' worth
// of a fixed tree per record
__global__ __launch_bounds__(256) void k_run_stats(const CellOut *__restrict__ outs,
                                                   const RunPart *__restrict__ part, int nparts)
{
    __shared__ RunPart s_p[256];
    RunPart a{};
    for (int k = threadIdx.x; k < nparts; k += 256) {
        const RunPart &q = part[(size_t)blockIdx.x * RUN_PARTS + k];
        a.sum += q.sum;
        a.mx = fmaxf(a.mx, q.mx);
        a.pairs += q.pairs;
#pragma unroll
        for (int i = 0; i < 6; ++i) a.c[i] += q.c[i];
    }
    s_p[threadIdx.x] = a;
    for (int off = 128; off >= 1; off >>= 1) {
        __syncthreads();
        if ((int)threadIdx.x < off) {
            const RunPart &q = s_p[threadIdx.x + off];
            a.sum += q.sum;
            a.mx = fmaxf(a.mx, q.mx);
            a.pairs += q.pairs;
#pragma unroll
            for (int i = 0; i < 6; ++i) a.c[i] += q.c[i];
            s_p[threadIdx.x] = a;
        }
    }
    if (threadIdx.x == 0) {
        BlockStats &st = *outs[blockIdx.x].st;
        st.gsum = a.sum;
        st.gmax = __float_as_uint(a.mx);
        st.ctrs[C_PAIRS] = a.pairs;
        for (int i = 0; i < 6; ++i) st.cstat[i] = a.c[i];
    }
}

void launch_run_finish(const CellOut *outs, const GridP *gps, RunPart *part, int nb, int max_cells,
                       unsigned long long max_grid, hipStream_t s)
{
    if (nb <= 0) return;
    // four items per lane, at most RUN_PARTS workgroups per block (a
    // single block fills the chip; many blocks share it)
    const long long cap = std::max<long long>(16, RUN_PARTS / std::max(1, nb / 4));
    const unsigned bc = (unsigned)std::max<long long>(
        1, std::min<long long>(cap / 8, ((long long)max_cells + 1023) / 1024));
    const unsigned bg = (unsigned)std::max<unsigned long long>(
        1, std::min<unsigned long long>(cap - cap / 8, (max_grid + 1023) / 1024));
    hipLaunchKernelGGL(k_run_finish, dim3(bg + bc, nb), dim3(256), 0, s, outs, gps, part, (int)bg);
    hipLaunchKernelGGL(k_run_stats, dim3(nb), dim3(256), 0, s, outs, (const RunPart *)part,
                       (int)(bg + bc));
}

}  // namespace t2
