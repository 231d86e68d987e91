// kernels.hpp -- device data layout and kernel declarations.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

#include "buckets.hpp"

namespace t2 {

// Grid and block parameters of one dense run on one block (host-computed
// with the reference's GridStepParams / BlockGridParams arithmetic).
struct GridP {
    float gmin[3];
    float step[3];
    float dmin[3];
    float dmax[3];
    float bmin[3];       // block bounds (the in-block deposit test)
    float bmax[3];
    int bmin_idx[3];
    int bnum_idx[3];
    float eps;
    float mass;
    float div;
    int project;         // 2-D x-y projection
};

// counters in device memory (ctrs[])
enum {
    C_OVF = 0,        // entries appended to the shared-point list
    C_OFFBLOCK = 1,   // points no block grid holds (dropped)
    C_SLOW = 2,       // cells queued for the large-capacity pass
    C_ERR = 3,        // bit 0: deferred-cell list full; bit 2: cell beyond all capacities;
                      // bit 3: a shared point beyond the fold's capacities
    C_DEFER = 4,      // grid points queued for the FP64 search of the exact assignment
    C_FALLBACK = 5,   // FP64 re-checks of the exact assignment
    C_ROUTED = 6,     // points deposited into another block's grid
    C_SEG = 7,        // contributions gathered into per-point segments for the fold
    C_FOLD0 = 8,      // shared points per fold class (C_FOLD0 + class, 3 classes)
    C_PAIRS = 11,     // points with a second contribution
    C_NCTR = 12
};

// fold classes by contributions per shared point
enum { FOLD_SMALL_MAX = 16, FOLD_MID_MAX = 2048 };

// Counters and statistics of one block; the records of all blocks of a
// context sit in one device array (cleared by one fill, copied to pinned host
// memory by one transfer).
struct BlockStats {
    unsigned ctrs[C_NCTR];
    unsigned pad0[16 - C_NCTR];
    unsigned long long cstat[6];   // cells per status 0..4, points of deposited cells
    double gsum;                   // sum of the block's density grid
    unsigned gmax;                 // bits of its maximum (non-negative float)
    unsigned pad1;
};
static_assert(sizeof(BlockStats) % 16 == 0, "BlockStats is cleared with 16-byte stores");

// Per-block device outputs of the density kernels.
struct CellOut {
    float *vol;        // [ncells] volume() or nullptr
    int *status;       // [ncells] TESS2_CELL_*
    int *npts;         // [ncells] points the cell deposits
    float *density;    // [grid]
    unsigned *count;   // [grid] contributions per point
    uint2 *first;      // [grid] first contribution (cell, mass bits)
    uint2 *second;     // [grid] second contribution (the list holds the third on)
    int *head;         // [grid] the point's fold record, -(1 + 4 index + class), written
                       // by the fold's gather for points with list entries
    int4 *ovf;         // shared-point list, third contribution on: {lidx, key, mass bits,
                       // ordinal among the point's contributions (2 for the third)};
                       // (3 * ovf_cap + 1) / 2 entries, the large fold's scratch
    unsigned ovf_cap;
    unsigned *ctrs;    // [C_NCTR]
    int *slow;         // cells for the large-capacity pass
    unsigned slow_cap;
    uint2 *seg;        // [3 * ovf_cap] contributions {key, mass bits}, one segment per point
    int4 *fold[3];     // shared points per fold class: {lidx, segment start, count, cursor}
    unsigned fold_cap[3];
    BlockStats *st;    // this block's record (st->ctrs == ctrs)
    unsigned long long ngrid;
    int ncells;
};

// Per-block grids and outputs of all blocks of a run, in staging order (the
// rank of a block = its position; blocks are staged in ascending gid), for
// deposits that leave their block.
struct Router {
    int nblocks;
    const GridP *gps;
    const CellOut *outs;
    // The ends of the blocks' 3-D grid ranges cut each axis into intervals:
    // rmap[roff[a] + g - rbase[a]] is the interval of global index g on
    // axis a (g in [rbase[a], rbase[a] + rlen[a])), rcand[(i0 * rn[1] + i1)
    // * rn[2] + i2] the first two blocks (staging order, -1 for none) whose
    // ranges hold the box of intervals (i0, i1, i2).
    const int *rmap;
    const int2 *rcand;
    int rbase[3], rlen[3], roff[3], rn[3];
};

// what one workgroup of the staging pass found in its part of a block's
// arrays; lo / hi: the bounding box of its particles (lo > hi: none)
struct StageInfo {
    unsigned err;          // an index out of range
    unsigned nonfinite;    // a coordinate that is infinite or NaN
    float lo[3], hi[3];
};
enum { STAGE_RECORDS = 1024 };   // workgroups of the pass at most

// the particles' bounding box (the Morton grid)
struct StageBox {
    float lo[3], hi[3];
};

// one chunk of cells of one block for the batched launch
struct Chunk {
    int block;
    int start;    // position in the block's cell order of the first cell
    int count;
    int stride;   // cells start, start + stride, ... (count of them)
};

// The chunk list split into 8 contiguous ranges, one per XCD (workgroup b
// runs on XCD b % 8): waves take chunks of their own range first, so that
// each XCD's L2 sees one compact part of the data, then help the others.
struct XcdQueues {
    int start[9];   // range x = chunks [start[x], start[x+1])
};

struct BlockIn {
    const float4 *pts;   // xyz + pad
    const int4 *tets;    // 2 int4 per tet: verts, neighbours
    const int *v2t;
    const float4 *cc;    // circumcenters (xyz + pad)
    const int *order;    // cells in processing (Morton) order, or nullptr
    int ncells;          // original particles
    int ntets;
    // set for a block whose indices are checked on the device: its kernels
    // return at once when *stop holds the token
    const unsigned *stop;
    unsigned token;
    __device__ __forceinline__ bool stopped() const { return stop && *stop == token; }
};

// 64 consecutive cells (of the Morton order) of one block; base: the position
// of the first in the buffers that run over all cells of a launch
enum { CELL_TILE = 64 };
struct CellTile {
    int block, start, count, base;
};

// The cells of a launch: one block given by value, or all blocks of a run by
// their descriptors in device memory and a tile list (no tile holds cells of
// two blocks).
template <bool MULTI> struct CellSet;
template <> struct CellSet<false> {
    BlockIn bin;
    CellOut bout;
    const GridP *gp;     // device memory, null without density
    int tile0, ntiles;   // the launch's tiles; positions count from the first
    __device__ __forceinline__ CellTile tile(int t) const
    {
        const int s = (tile0 + t) * CELL_TILE;
        return CellTile{0, s, min((int)CELL_TILE, bin.ncells - s), t * CELL_TILE};
    }
    __device__ __forceinline__ const BlockIn &in(int) const { return bin; }
    __device__ __forceinline__ const CellOut &out(int) const { return bout; }
    __device__ __forceinline__ const GridP &grid(int) const { return *gp; }
    __device__ __forceinline__ const Router *router() const { return nullptr; }
};
template <> struct CellSet<true> {
    const BlockIn *ins;
    const CellOut *outs;
    const GridP *gps;
    const Router *rt;
    const CellTile *tiles;
    int tile0, ntiles;
    __device__ __forceinline__ CellTile tile(int t) const
    {
        const CellTile q = tiles[tile0 + t];
        return CellTile{q.block, q.start, q.count, t * CELL_TILE};
    }
    __device__ __forceinline__ const BlockIn &in(int b) const { return ins[b]; }
    __device__ __forceinline__ const CellOut &out(int b) const { return outs[b]; }
    __device__ __forceinline__ const GridP &grid(int b) const { return gps[b]; }
    __device__ __forceinline__ const Router *router() const { return rt; }
};

// What the geometry kernel leaves for the scan, by position: bbox and face
// count (0: nothing to scan), {min xyz, faces}, {max xyz, cell}; the face
// planes {n, f0.x}, {f0.y, f0.z}, PLANE_STRIDE per cell
enum { PLANE_STRIDE = 26 };
struct PlaneBuf {
    float4 *hdr;
    float4 *fa;
    float2 *fb;
    int2 *big;         // {block, position} of the cells for one wave each
    unsigned *nbig;    // their number, cleared with the run's counters
};

// find or insert key (>= 0) in an open-addressing table of HS entries in
// LDS (-1 = empty); returns the entry, or -1 when HS probes found no room
template <int HS>
__device__ __forceinline__ int hash_find(int *hk, int key)
{
    unsigned h = ((unsigned)key * 0x9E3779B1u) >> 16;
    for (int n = 0; n < HS; ++n) {
        h &= HS - 1;
        const int old = atomicCAS(&hk[h], -1, key);
        if (old == -1 || old == key) return (int)h;
        ++h;
    }
    return -1;
}

// orders a wave's LDS accesses where its lanes exchange values through LDS (its
// LDS instructions execute in order; the fence keeps the compiler from
// reusing or moving a load across, which the barrier alone does not)
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Workgroup -> work item with XCD affinity: the dispatcher hands consecutive
// workgroups to the 8 XCDs in turn, so item k = (b % 8) * chunk + b / 8 gives
// each XCD (and its L2) one contiguous range of items.  Returns -1 for the
// padding workgroups of the last range.
__device__ __forceinline__ int xcd_item(int b, int n)
{
    const int chunk = (n + 7) >> 3;
    const int k = (b & 7) * chunk + (b >> 3);
    return k < n ? k : -1;
}
__host__ __forceinline__ int xcd_grid(int n) { return ((n + 7) >> 3) << 3; }

// copies between pageable host memory and device memory (transfer.hip), after
// the stream's earlier work.  copy_to_host is done when it returns; the array
// given to copy_to_device may be read until the stream has been waited for.
// The pinned slots behind them live while a context is open.
void transfer_open();
void transfer_close();
hipError_t copy_to_host(void *dst, const void *src, size_t bytes, hipStream_t s);
hipError_t copy_to_device(void *dst, const void *src, size_t bytes, hipStream_t s);
// circumcenters; cc.w = error bound of the float solve (inf when undefined)
void launch_circumcenters(const float4 *pts, const int4 *tets, int ntets, float4 *cc,
                          hipStream_t s);
// bucket hash of the np particles and the cells' deposit status; start, flags
// (3 * ncells bytes: incomplete, outside, defined) and the counts below are
// zero on entry
void launch_exact_setup(const BlockIn &in, const GridP &gp, int np, const HashP &h,
                        unsigned *start, unsigned *sums, int2 *bk, float4 *sorted, const int *key,
                        int *status, int prec, unsigned *ctrs, unsigned char *flags,
                        hipStream_t s);
// npts_tab / stex_tab (by rank) when several blocks share the assignment,
// else nullptr; defq: queue of defq_cap grid points for the FP64 re-search
// of the mixed precision (0: searched inline)
void launch_owner(const GridP &gp, const HashP &h, const unsigned *start, const float4 *hp,
                  int *owner, int prec, unsigned *ctrs, const int *status, int *npts,
                  int ncells, int *const *npts_tab, const int *const *stex_tab, unsigned *defq,
                  unsigned defq_cap, hipStream_t s);
// parts: 1 = densities of the owned points, 2 = CIC of cells that own none;
// every block's part 1 must precede any block's part 2
void launch_exact_tail(const BlockIn &in, const GridP &gp, const int *owner,
                       const int *status_ex, const CellOut &o, int prec, int *const *npts_tab,
                       const int *const *stex_tab, const Router *rt, int self, int parts,
                       hipStream_t s);
// exclusive scan of n counts in place; sums: scan_sums_words(n) words of
// scratch
size_t scan_sums_words(size_t n);
void launch_scan_u32(unsigned *a, unsigned n, unsigned *sums, hipStream_t s);
void launch_fill_u32(unsigned *p, size_t n, unsigned v, hipStream_t s);
// ghost selection (incomplete_cells): bit i of sends[p] for neighbour box i
// (6 floats each, [first, nnb)), for original particles p < norig
void launch_ghost_sends(const float4 *pts, const int4 *tets, int ntets, int norig,
                        const float *bmin, const float *bmax, const float *boxes, int nnb,
                        int first, unsigned long long *sends, hipStream_t s);
// staging (stage.hip): range checks, bounding box and float4 particles of a
// block as the caller gave it; then its cells in Morton order and its tets
// renumbered by their lowest-ranked vertex (raw, v2t_raw: the caller's
// numbering; scratch: layout_scratch_words(np, nt) words)
// (returns the records written)
int launch_stage_check(const float *xyz, int np, const int4 *tets, int nt, const int *v2t,
                       float4 *pts, StageInfo *info, hipStream_t s);
size_t layout_scratch_words(int np, int nt);
void launch_layout(const float4 *pts, int np, int norig, const StageBox &box, const int4 *raw,
                   int nt, const int *v2t_raw, unsigned *scratch, int *order, int4 *tets,
                   int *v2t, int *tnew, hipStream_t s);
// circumcenters as xyz triples in the caller's tet numbering
void launch_unpack_cc(const float4 *cc, const int *tnew, int nt, float *out, hipStream_t s);
// a block in the caller's device memory: float4 particles, circumcenters,
// zeroed counters; an index out of range stores token in *stop (BlockIn::stop)
void launch_device_block(const float *xyz, int np, const int4 *tets, int nt, const int *v2t,
                         float4 *pts, float4 *cc, unsigned *ctrs, unsigned *stop, unsigned token,
                         hipStream_t s);
// up to four arrays of n words to zero at the start of a run
struct ZeroList {
    unsigned *p[4];
    unsigned long long n[4];
};
// the start of a run: circumcenters of every block (max_tets > 0), density and
// count grids and the listed arrays zeroed
void launch_run_prep(const BlockIn *ins, const CellOut *outs, int nb, int max_tets,
                     unsigned long long max_grid, const ZeroList &z, hipStream_t s);
void launch_cells_ref(const BlockIn &in, const GridP &gp, const CellOut &o,
                      int want_density, hipStream_t s);
void launch_cells_ref_slow(const BlockIn &in, const GridP &gp, const CellOut &o,
                           int want_density, hipStream_t s);
// stars, faces, volumes of all tiles' cells (cells_geom.hip); with
// want_density also what the scan needs, in pb (else unused)
void launch_cell_geom(const CellSet<false> &set, const PlaneBuf &pb, int want_density,
                      hipStream_t s);
void launch_cell_geom(const CellSet<true> &set, const PlaneBuf &pb, int want_density,
                      hipStream_t s);
// scan and deposit of the cells whose planes are in pb (cells_scan.hip);
// eps >= 0
void launch_cell_scan(const CellSet<false> &set, const PlaneBuf &pb, hipStream_t s);
void launch_cell_scan(const CellSet<true> &set, const PlaneBuf &pb, hipStream_t s);
// several cells per wave in the geometry phase (cells_mc.hip); variant 1..2
// picks the verdict masks; returns -1 for an unknown variant.  gp is the
// block's grid descriptor in device memory (read only by the scan, so that
// its fields take no registers in the geometry phase; may be null without
// density)
int launch_cells_mc(const BlockIn &in, const GridP *gp, const CellOut &o, int want_density,
                    int variant, hipStream_t s);
// large-capacity pass over the cells every block's fast pass deferred
void launch_cells_ref_slow_batched(const BlockIn *ins, const Router *rt, int want_density,
                                   hipStream_t s);
// the two-cell kernel over all blocks in one persistent launch (the deferred
// cells then need launch_cells_ref_batched's large-capacity pass)
// the batched launch over an item list (two consecutive cells of one block
// per item), one workgroup per item, no work queue
void launch_cells_mc_items(const BlockIn *ins, const GridP *gps, const CellOut *outs,
                           const Router *rt, const Chunk *items, const XcdQueues &xr,
                           int want_density, hipStream_t s);
void launch_cells_mc_batched(const BlockIn *ins, const GridP *gps, const CellOut *outs,
                             const Router *rt, const Chunk *chunks, const XcdQueues &xq,
                             unsigned *queue, int waves, int want_density, hipStream_t s);
void launch_cic(const BlockIn &in, const GridP &gp, const CellOut &o, const Router *rt_dev,
                int self, hipStream_t s);
// spec: each star-search candidate loads its tet's record before the table
// decides whether it is new (the loads overlap the LDS work)
void launch_cells_ref_batched(const BlockIn *ins, const GridP *gps, const CellOut *outs,
                              const Router *rt, const Chunk *chunks, const XcdQueues &xq,
                              unsigned *queue, int waves, int want_density, hipStream_t s,
                              bool spec);
// ordered fold of the points with three and more contributions of nb blocks at
// once (outs/gps: device arrays; the capacities size the grids)
// nb <= 128; the sums are the list capacities of all blocks
void launch_fold(const CellOut *outs, const GridP *gps, int nb, unsigned max_ovf_cap,
                 const unsigned max_fold_cap[3], unsigned long long sum_ovf_cap,
                 unsigned long long sum_mid_cap, hipStream_t s);
// the end of a run: points with two contributions, statistics.  part: nb *
// RUN_PARTS records of scratch
enum { RUN_PARTS = 1024 };
struct RunPart {
    double sum;                  // of the density
    float mx;                    // its maximum
    unsigned pairs;              // points with two and more contributions
    unsigned long long c[6];     // cells per status 0..4, points of deposited cells
};
void launch_run_finish(const CellOut *outs, const GridP *gps, RunPart *part, int nb, int max_cells,
                       unsigned long long max_grid, hipStream_t s);

}  // namespace t2
