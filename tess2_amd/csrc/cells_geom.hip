// cells_geom.hip -- the geometry of every cell (star, faces, ring walks,
// volume, bbox), several cells per wave, for the scan kernel (cells_scan.hip)
// or for volumes alone.
//
// One 64-lane wave takes CPW consecutive cells of a block's Morton order,
// G = 64 / CPW lanes per cell for the star, all 64 lanes over the faces of
// its cells for the ring walks:
//   1. star (neighbor_edges' first-seen order, src/tet.cpp:228-270).  A star
//      tet has three link vertices (its vertices but the cell's) and three
//      neighbours in the star, one across each.  A tet met across a face of
//      its parent shares two link vertices with it, whose face numbers the
//      parent knows; only the third (the apex) can be new.  So each tet asks
//      the tet table twice (its parent is known) and the vertex table once.
//      The candidates (two per tet, three for the first) form one queue in
//      (slot, link vertex) order, G of which are resolved per round: the lowest
//      lane of those that meet a new tet takes it, the takers get the next
//      slots in lane order, then the takers with a new apex the next face
//      numbers: the order in which a walk through the queue first meets them.
//   2. the circumcenters of the star, one gather per tet, and the bbox
//      (src/dense.cpp:701-714).
//   3. ring walks (fill_edge_link, src/tet.cpp:389-409), one face per lane over
//      star slots and face numbers: Newell normal (src/dense.cpp:1131-1162),
//      fan area with the double square root (src/volume.cpp:32-46).
//   4. volume, the faces in neighbour order (src/volume.cpp:23-53).
//
// A table entry is one word: the low 26 bits of the id above six bits that
// hold a slot (or face number), or 48 + lane while a round decides who takes
// it; atomicMin leaves the lowest.  Each user then compares the slot's full id, so
// two ids that share 26 bits only defer the cell.
// What bounds it: vector instructions, 604 a cell, more than half of them in
// the star's rounds (2.1M cells of a GRF box with planes: 1.80 to 1.86 ms, one
// instruction per SIMD in 3.5 cycles; volumes of
// 216k cells 188 us, of 64k 64).
// Each table probe, index and mask in a round is therefore the cheapest form
// that holds: tables of 64 words that cannot fill up (with 32 words for the
// vertices and a probe count 2.04 ms, 219 and 74 us), 24-bit hash products,
// wrap-arounds by one subtraction, hull links seen when a tet is taken rather
// than when it is visited, a group's ballot in one register, the bbox by
// row exchanges instead of LDS.  Eight cells a wave (8 lanes each) has the
// same rate and a longer latency.
// Cells beyond SG star tets or FG faces, and stars whose links are not those
// of a tessellation, go to the large-capacity pass (k_cells_ref_slow).
#include "kernels.hpp"
#include "geom.hpp"
#include "cell_status.hpp"

namespace t2 {

namespace {

enum { G_RUN = 0, G_NONE = 1, G_HULL = 2, G_DEFER = 3 };

constexpr unsigned EMPTY = 0xffffffffu;
constexpr unsigned PENDING = 48;   // low six bits from here on: 48 + lane
constexpr int QUEUE = 24;          // tets met and not yet visited, at most

// Correctly rounded square root of a double holding a float value: the
// reciprocal square root refined by Goldschmidt's iteration with two Newton
// corrections, without the rescaling of inputs below 2^-767 that float
// values never need.
__device__ __forceinline__ double sqrt_of_float_g(double x)
{
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y;
    double h = y * 0.5;
    const double r = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, r, g);
    double d = __builtin_fma(-g, g, x);
    h = __builtin_fma(h, r, h);
    g = __builtin_fma(d, h, g);
    d = __builtin_fma(-g, g, x);
    g = __builtin_fma(d, h, g);
    return __builtin_amdgcn_class(x, 0x260) ? x : g;
}

__device__ __forceinline__ unsigned eq4(const int4 &q, int x)
{
    return (q.x == x ? 1u : 0u) | (q.y == x ? 2u : 0u) | (q.z == x ? 4u : 0u) |
           (q.w == x ? 8u : 0u);
}

// the component at the one bit of m, by masks
__device__ __forceinline__ int pick4(const int4 &q, unsigned m)
{
    return (q.x & -(int)(m & 1u)) | (q.y & -(int)((m >> 1) & 1u)) |
           (q.z & -(int)((m >> 2) & 1u)) | (q.w & -(int)((m >> 3) & 1u));
}

// x of the lane whose number differs by a mirror: quads' pairs, quads' halves,
// eights and sixteens, which together reach every lane of 16
template <int CTRL>
__device__ __forceinline__ float dpp_f(float x)
{
    return __int_as_float(
        __builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, false));
}
__device__ __forceinline__ float lesser(float x, float y) { return y < x ? y : x; }   // no NaN
__device__ __forceinline__ float min16(float x)
{
    x = lesser(x, dpp_f<0xb1>(x));    // quad_perm 1,0,3,2
    x = lesser(x, dpp_f<0x4e>(x));    // quad_perm 2,3,0,1
    x = lesser(x, dpp_f<0x141>(x));   // mirrored eights
    return lesser(x, dpp_f<0x140>(x));   // mirrored sixteens
}

// first entry to look at in a table of 64 words: the top bits of a 24-bit
// product (a full-rate multiplication; consecutive ids fall far apart)
__device__ __forceinline__ unsigned table_first(int id)
{
    return (__umul24((unsigned)id, 0x9E3779u) >> 18) & 63u;
}

// find id in the table of 64 words or put `want` (its tag above a pending
// code) there; the lowest pending code of an id stays.  Returns the entry.  A
// round starts with at most SG tets and FG vertices and adds at most one per
// lane of the group, so that there always is one.
__device__ __forceinline__ int table_take(unsigned *t, int id, unsigned want)
{
    unsigned h = table_first(id), old = atomicCAS(&t[h], EMPTY, want);
    while (old != EMPTY && (old >> 6) != (want >> 6)) {
        h = (h + 1) & 63u;
        old = atomicCAS(&t[h], EMPTY, want);
    }
    if (old != EMPTY && (old & 63u) >= PENDING) atomicMin(&t[h], want);
    return (int)h;
}

}  // namespace

// One cell's LDS: the tables and the queue of candidates, later the
// circumcenters; then the star.  F (words): the face numbers of a tet's link
// vertices in vertex order, a byte each, the apex's position in the top byte.
// NB (bytes): the star slots across them.
template <int SG, int FG>
struct GeomLayout {
    static constexpr int T = 0;                 // unsigned [64] tet table
    static constexpr int V = 256;               // unsigned [64] vertex table
    static constexpr int CAND = 512;            // int2 [QUEUE] neighbour ids to visit
    static constexpr int CC = 0;                // float [SG][3] circumcenters
    static constexpr int TID = CAND + 8 * QUEUE;   // int [SG] slot -> tet; then fvol
    static constexpr int F = TID + 4 * SG;      // unsigned [SG]
    static constexpr int FU = F + 4 * SG;       // int [FG] face -> vertex
    static constexpr int FLAG = FU + 4 * FG;    // int: a ring does not close
    static constexpr int NB = FLAG + 4;         // unsigned char [SG][3]
    static constexpr int FS = NB + 3 * SG;      // unsigned char [FG] face -> first slot
    static constexpr int BYTES = (FS + FG + 15) / 16 * 16;
    static_assert(12 * SG <= TID, "the circumcenters fit over tables and queue");
    static_assert(SG + 16 <= 64 && FG + 16 <= 64, "a round's new ids fit the tables");
};

template <int CPW, int SG, int FG, bool MULTI, bool PLANES>
__global__ __launch_bounds__(64) void k_cell_geom(CellSet<MULTI> set, PlaneBuf pb)
{
    using L = GeomLayout<SG, FG>;
    constexpr int G = 64 / CPW;
    static_assert(G * CPW == 64 && G >= 4 && G <= 16, "three lanes start a star; pending codes");
    static_assert(SG <= (int)PENDING && FG <= 32 && 4 * FG <= 4 * SG, "table codes; fvol room");
    __shared__ __align__(16) unsigned char smem[CPW * L::BYTES];

    const int lane = (int)(threadIdx.x & 63);
    const int g = lane / G, gl = lane % G;
    const unsigned long long gbits = ((1ull << G) - 1ull) << (g * G);
    // a ballot's half that holds the group, the group's bits there, and those
    // of its lower lanes
    const bool upper = lane >= 32;
    auto half = [upper](unsigned long long m) {
        return upper ? (unsigned)(m >> 32) : (unsigned)m;
    };
    const unsigned ghalf = half(gbits), gbelow = ghalf & ((1u << (lane & 31)) - 1u);

    constexpr int WPT = CELL_TILE / CPW;   // waves per tile
    const int item = xcd_item((int)blockIdx.x, set.ntiles * WPT);
    if (item < 0) return;
    const CellTile tile = set.tile(item / WPT);
    const BlockIn in = set.in(tile.block);
    if (!MULTI && !PLANES && in.stopped()) return;
    const int rel = (item % WPT) * CPW + g;   // this group's cell in the tile
    const bool have = rel < tile.count;
    const int v = have ? (in.order ? in.order[tile.start + rel] : tile.start + rel) : -1;

    unsigned char *R = smem + g * L::BYTES;
    unsigned *T = reinterpret_cast<unsigned *>(R + L::T);
    unsigned *V = reinterpret_cast<unsigned *>(R + L::V);
    int *cand = reinterpret_cast<int *>(R + L::CAND);
    int *tid = reinterpret_cast<int *>(R + L::TID);
    unsigned *fw = reinterpret_cast<unsigned *>(R + L::F);
    unsigned char *nb = R + L::NB;
    int *fu = reinterpret_cast<int *>(R + L::FU);
    unsigned char *fs = R + L::FS;

    const int vt = have ? in.v2t[v] : -1;
    int st = !have ? G_NONE : (vt < 0 ? G_HULL : G_RUN);

    // ---- 1. star ------------------------------------------------------------
    for (int i = gl; i < 128; i += G) T[i] = EMPTY;   // both tables
    if (gl == 0) *reinterpret_cast<int *>(R + L::FLAG) = 0;
    wave_sync();
    int rootn = -1;   // lanes 0..2: the first tet's neighbour across link vertex gl
    if (st == G_RUN) {
        const int4 rv = in.tets[2 * (long long)vt], rn = in.tets[2 * (long long)vt + 1];
        const unsigned mv = eq4(rv, v);
        bool ok = __popc(mv) == 1, inner = true;
        if (ok && gl < 3) {
            const unsigned mi = 1u << (gl + (gl >= __builtin_ctz(mv) ? 1 : 0));
            const int u = pick4(rv, mi);
            rootn = pick4(rn, mi);
            const unsigned want = ((unsigned)u << 6) | (unsigned)gl;
            inner = rootn >= 0;
            const int e = table_take(V, u, want);
            ok = V[e] == want;   // a vertex twice in the tet: not a tet
            fu[gl] = u;
            fs[gl] = 0;
        }
        if (ok && gl == 0) {
            T[table_first(vt)] = (unsigned)vt << 6;
            tid[0] = vt;
            fw[0] = 0u | (1u << 8) | (2u << 16) | (3u << 24);
        }
        if (__ballot(!inner) & gbits) st = G_HULL;
        if (__ballot(!ok) & gbits) st = G_DEFER;
    }
    wave_sync();
    int S = 1, F = 3, hc = 0;   // tets, faces, candidates resolved so far
    for (;;) {
        const int ncand = 2 * S + 1;
        const int q = hc + gl;
        bool mine = st == G_RUN && q < ncand;
        if (!__ballot(mine)) break;
        int s = 0, j = q, ni = rootn, fa = 0, fb = 0, ua = 0, ub = 0, ptid = 0;
        int4 rv = make_int4(0, 0, 0, 0), rn = make_int4(0, 0, 0, 0);
        if (mine) {
            if (q >= 3) {
                s = (q - 1) >> 1;
                ni = cand[q - 1 - (q > 2 * QUEUE ? 2 * QUEUE : 0)];
            }
            const unsigned w = fw[s];
            if (q >= 3) {
                const int c = (q - 1) & 1;
                j = c + (c >= (int)(w >> 24) ? 1 : 0);
            }
            // loaded before the table knows whether the tet is new, so that
            // the load is in flight while it decides
            const int4 *tp = in.tets + 2u * (unsigned)ni;
            rv = tp[0];
            rn = tp[1];
            // the link vertices shared across the face: the other two
            fa = (int)((w >> (j == 0 ? 8 : 0)) & 255u);
            fb = (int)((w >> (j == 2 ? 8 : 16)) & 255u);
            ua = fu[fa];
            ub = fu[fb];
            ptid = tid[s];
        }
        const unsigned code = PENDING + (unsigned)gl;
        int e = 0;
        if (mine) e = table_take(T, ni, ((unsigned)ni << 6) | code);
        bool bad = false, hull = false;
        wave_sync();
        const unsigned te = T[e];
        const bool lead = mine && (te & 63u) == code;
        const unsigned Lb = half(__ballot(lead));
        const int slot = S + __popc(Lb & gbelow);
        S += __popc(Lb & ghalf);
        if (S > SG || 2 * S - hc > 2 * QUEUE) st = G_DEFER;
        const bool take = lead && st == G_RUN;
        int jp = 0, ev = 0, up = 0;
        unsigned wnew = 0;
        if (take) {
            // the apex is the new tet's vertex besides the cell's and the two
            // shared ones; where it holds the three, and its neighbours there
            up = (int)((unsigned)rv.x + (unsigned)rv.y + (unsigned)rv.z + (unsigned)rv.w -
                       (unsigned)v - (unsigned)ua - (unsigned)ub);
            // its link vertices l and the neighbours m across them, in order
            const bool v0 = rv.x == v, v1 = v0 || rv.y == v, v2 = v1 || rv.z == v;
            const int l0 = v0 ? rv.y : rv.x, l1 = v1 ? rv.z : rv.y, l2 = v2 ? rv.w : rv.z;
            const int m0 = v0 ? rn.y : rn.x, m1 = v1 ? rn.z : rn.y, m2 = v2 ? rn.w : rn.z;
            const bool p0 = l0 == up, p2 = l2 == up;   // the apex: first, last, or second
            jp = p0 ? 0 : (p2 ? 2 : 1);
            const int first = p0 ? l1 : l0, second = p2 ? l1 : l2;
            const int np = p0 ? m0 : (p2 ? m2 : m1);
            const int na = p0 ? m1 : m0, nbb = p2 ? m1 : m2;
            const bool fwd = first == ua;
            // not a tet on that face, or one that does not link back (with
            // the cell's vertex and the shared two in it, the apex is the
            // fourth by its sum)
            bad = !(v2 || rv.w == v) || first != (fwd ? ua : ub) || second != (fwd ? ub : ua) ||
                  up == ua || up == ub || np != ptid;
            T[e] = (te & ~63u) | (unsigned)slot;
            tid[slot] = ni;
            const int at = 2 * (slot - (slot >= QUEUE ? QUEUE : 0));
            cand[at] = na;
            cand[at + 1] = nbb;
            wnew = ((unsigned)(fwd ? fa : fb) << (p0 ? 8 : 0)) |
                   ((unsigned)(fwd ? fb : fa) << (p2 ? 8 : 16)) | ((unsigned)jp << 24);
            hull = (na | nbb) < 0;   // a hull link: the cell is infinite
            nb[3 * slot + jp] = (unsigned char)s;
            ev = table_take(V, up, ((unsigned)up << 6) | code);
        }
        wave_sync();
        // new apexes: face numbers in slot (lane) order
        const unsigned ve = V[take && !bad ? ev : 0];
        const bool leadv = take && !bad && (ve & 63u) == code;
        const unsigned Lv = half(__ballot(leadv));
        const int fnew = F + __popc(Lv & gbelow);
        F += __popc(Lv & ghalf);
        if (F > FG) st = G_DEFER;
        if (leadv && st == G_RUN) {
            V[ev] = (ve & ~63u) | (unsigned)fnew;
            fu[fnew] = up;
            fs[fnew] = (unsigned char)slot;
        }
        wave_sync();
        if (mine && !bad && st == G_RUN) {
            if (take) {
                const int fp = (int)(V[ev] & 63u);
                fw[slot] = wnew | ((unsigned)fp << (8 * jp));
                bad = fu[fp] != up;        // another vertex with the same tag
            }
            const int sl = (int)(T[e] & 63u);
            nb[3 * s + j] = (unsigned char)sl;
            bad = bad || tid[sl] != ni;    // another tet with the same tag
        }
        if (__ballot(bad || hull)) {
            if (__ballot(hull) & gbits) st = G_HULL;
            if (__ballot(bad) & gbits) st = G_DEFER;
        }
        hc = min(hc + G, ncand);
        wave_sync();
    }

    // ---- 2. circumcenters and bbox -------------------------------------------
    float *cc = reinterpret_cast<float *>(R + L::CC);   // over the tables
    float mnx = INFINITY, mny = INFINITY, mnz = INFINITY;
    float mxx = -INFINITY, mxy = -INFINITY, mxz = -INFINITY;
    if (st == G_RUN) {
        for (int i = gl; i < S; i += G) {
            const float4 c = in.cc[tid[i]];
            cc[3 * i] = c.x;
            cc[3 * i + 1] = c.y;
            cc[3 * i + 2] = c.z;
            if (PLANES) {
                if (c.x < mnx) mnx = c.x;
                if (c.y < mny) mny = c.y;
                if (c.z < mnz) mnz = c.z;
                if (c.x > mxx) mxx = c.x;
                if (c.y > mxy) mxy = c.y;
                if (c.z > mxz) mxz = c.z;
            }
        }
    }
    if (PLANES) {
        static_assert(G == 16, "a group is a row of lanes");
        mnx = min16(mnx);
        mny = min16(mny);
        mnz = min16(mnz);
        mxx = -min16(-mxx);
        mxy = -min16(-mxy);
        mxz = -min16(-mxz);
    }
    wave_sync();
    if (PLANES && st == G_RUN) {
        // the first ring vertex of the first face seeds the reference's fold;
        // a NaN there survives every later comparison
        const float c00x = cc[0], c00y = cc[1], c00z = cc[2];
        if (isnan(c00x)) { mnx = c00x; mxx = c00x; }
        if (isnan(c00y)) { mny = c00y; mxy = c00y; }
        if (isnan(c00z)) { mnz = c00z; mxz = c00z; }
    }

    // ---- 3. ring walks, the faces of all cells of the wave over its lanes ----
    int pre[CPW + 1];   // faces of the groups below (wave-uniform)
    pre[0] = 0;
#pragma unroll
    for (int k = 0; k < CPW; ++k)
        pre[k + 1] = pre[k] + __builtin_amdgcn_readlane(st == G_RUN ? F : 0, k * G);
    const long long base = (long long)tile.base + (item % WPT) * CPW;
    for (int p0 = 0; p0 < pre[CPW]; p0 += 64) {
        const int p = p0 + lane;
        int k = 0, kp = 0;
#pragma unroll
        for (int i = 1; i < CPW; ++i)
            if (p >= pre[i]) {
                k = i;
                kp = pre[i];
            }
        const int vc = __shfl(v, k * G);
        if (p < pre[CPW]) {
            unsigned char *Q = smem + k * L::BYTES;
            const float *qc = reinterpret_cast<const float *>(Q + L::CC);
            const unsigned *qf = reinterpret_cast<const unsigned *>(Q + L::F);
            const unsigned char *qn = Q + L::NB;
            const int f = p - kp;
            const int u = reinterpret_cast<const int *>(Q + L::FU)[f];
            const float4 pu = in.pts[u], site = in.pts[vc];
            const int us = Q[L::FS + f];
            unsigned w = qf[us];
            const float3 c0 = make_float3(qc[3 * us], qc[3 * us + 1], qc[3 * us + 2]);
            float cx = c0.x, cy = c0.y, cz = c0.z;
            float abx = 0.0f, aby = 0.0f, abz = 0.0f;   // ring[L-1] - ring[0]
            float nx = 0.0f, ny = 0.0f, nz = 0.0f;
            float area = 0.0f;
            // circulate_start: the first link vertex that is not u
            int wi = (int)(w & 255u) == f ? 1 : 0;
            int behind = (int)((w >> (8 * wi)) & 255u);
            int t = us, Lr = 1;
            bool stuck = false;
            for (;;) {
                // circulate_next (src/tet.cpp:185-215): the next vertex is the
                // link vertex that is not u or behind
                const int nv = (int)__builtin_amdgcn_udot4(w, 0x010101u, (unsigned)(-f - behind),
                                                           false);
                const int nt = qn[3 * t + wi];
                if (nt == us) break;
                w = qf[nt];
                const float3 c = make_float3(qc[3 * nt], qc[3 * nt + 1], qc[3 * nt + 2]);
                // its position among the next tet's link vertices
                const unsigned x = w ^ ((unsigned)nv * 0x010101u);
                wi = (x & 0xffu) == 0u ? 0 : ((x & 0xff00u) == 0u ? 1 : 2);
                const bool lost = (x & 0xff0000u) != 0u && wi == 2;
                // Newell term for (ring[L-1], ring[L])
                nx += (cy - c.y) * (cz + c.z);
                ny += (cz - c.z) * (cx + c.x);
                nz += (cx - c.x) * (cy + c.y);
                const float acx = c.x - c0.x, acy = c.y - c0.y, acz = c.z - c0.z;
                if (Lr >= 2) {   // fan triangle (ring[0], ring[L-1], ring[L])
                    const float px = aby * acz - abz * acy;
                    const float py = abz * acx - abx * acz;
                    const float pz = abx * acy - aby * acx;
                    area = (float)((double)area +
                                   sqrt_of_float_g((double)nrm3(px, py, pz)) / 2.0);
                }
                cx = c.x;
                cy = c.y;
                cz = c.z;
                abx = acx;
                aby = acy;
                abz = acz;
                t = nt;
                behind = nv;
                if (++Lr > SG || lost) {
                    stuck = true;
                    break;
                }
            }
            if (stuck) *reinterpret_cast<int *>(Q + L::FLAG) = 1;
            const float ddx = pu.x - site.x, ddy = pu.y - site.y, ddz = pu.z - site.z;
            const float dist = sqrtf(nrm3(ddx, ddy, ddz));
            reinterpret_cast<float *>(Q + L::TID)[f] = area * dist / 6.0f;
            if (PLANES) {
                // closing Newell term (ring[L-1], ring[0])
                nx += (cy - c0.y) * (cz + c0.z);
                ny += (cz - c0.z) * (cx + c0.x);
                nz += (cx - c0.x) * (cy + c0.y);
                const float mag = sqrtf(nx * nx + ny * ny + nz * nz);
                nx = -(nx / mag);
                ny = -(ny / mag);
                nz = -(nz / mag);
                const float wx = c0.x - site.x, wy = c0.y - site.y, wz = c0.z - site.z;
                if (wx * nx + wy * ny + wz * nz < 0.0f) {
                    nx = -nx;
                    ny = -ny;
                    nz = -nz;
                }
                const long long at = (base + k) * PLANE_STRIDE + f;
                pb.fa[at] = make_float4(nx, ny, nz, c0.x);
                pb.fb[at] = make_float2(c0.y, c0.z);
            }
        }
    }
    wave_sync();

    // ---- 4. volumes and the cells' records ------------------------------------
    if (st == G_RUN && *reinterpret_cast<int *>(R + L::FLAG)) st = G_DEFER;
    if (gl == 0 && st != G_NONE) {
        const CellOut &o = set.out(tile.block);
        if (st == G_RUN) {
            if (o.vol) {
                const float *fvol = reinterpret_cast<const float *>(tid);
                float vol = 0.0f;
                for (int i = 0; i < F; i += 4) {
                    const float4 q = *reinterpret_cast<const float4 *>(fvol + i);
                    vol += q.x;
                    vol = i + 1 < F ? vol + q.y : vol;
                    vol = i + 2 < F ? vol + q.z : vol;
                    vol = i + 3 < F ? vol + q.w : vol;
                }
                o.vol[v] = vol;
            }
            if (!PLANES) {
                o.status[v] = ST_SCAN;
                o.npts[v] = 0;
            }
        } else if (st == G_HULL) {
            o.status[v] = ST_INCOMPLETE;
            o.npts[v] = 0;
            if (o.vol) o.vol[v] = -1.0f;
        } else {
            const unsigned kk = atomicAdd(&o.ctrs[C_SLOW], 1u);
            if (kk < o.slow_cap) o.slow[kk] = v;
            else atomicOr(&o.ctrs[C_ERR], 1u);   // list full: rerun with more room
        }
        if (PLANES) {
            pb.hdr[2 * (base + g)] =
                make_float4(mnx, mny, mnz, __int_as_float(st == G_RUN ? F : 0));
            pb.hdr[2 * (base + g) + 1] = make_float4(mxx, mxy, mxz, __int_as_float(v));
        }
    }
}

template <bool MULTI>
static void launch_geom(const CellSet<MULTI> &set, const PlaneBuf &pb, int want_density,
                        hipStream_t s)
{
    if (set.ntiles <= 0) return;
    constexpr int CPW = 4, SG = 48;
    const dim3 grid(xcd_grid(set.ntiles * (CELL_TILE / CPW)));
    if (want_density)
        hipLaunchKernelGGL((k_cell_geom<CPW, SG, PLANE_STRIDE, MULTI, true>), grid, dim3(64), 0,
                           s, set, pb);
    else
        hipLaunchKernelGGL((k_cell_geom<CPW, SG, PLANE_STRIDE, MULTI, false>), grid, dim3(64), 0,
                           s, set, pb);
}

void launch_cell_geom(const CellSet<false> &set, const PlaneBuf &pb, int want_density,
                      hipStream_t s)
{
    launch_geom<false>(set, pb, want_density, s);
}

void launch_cell_geom(const CellSet<true> &set, const PlaneBuf &pb, int want_density,
                      hipStream_t s)
{
    launch_geom<true>(set, pb, want_density, s);
}

}  // namespace t2
