// A HIP runtime without a GPU, for tests of the library's host code: device
// memory is host memory, kernels do nothing, and the test sets what fails and
// what each launch costs.  Linked with api.hip and transfer.hip compiled for
// the host only.
#include "../tess2_amd/csrc/kernels.hpp"

#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <set>
#include <vector>

namespace {

std::mutex mu;
std::map<char *, size_t> device;          // allocations
std::map<char *, size_t> pinned;
size_t used = 0, limit = ~size_t(0);      // bytes; hipMalloc fails beyond the limit
long fail_copy = -1;                      // copies until one fails (-1: none)
hipError_t last_error = hipSuccess;

struct Pending { const char *host; size_t bytes; };
std::vector<Pending> pending;             // pageable sources not waited for

// counters, by name in fake_count
long n_malloc, n_copy, n_graph, n_sync, n_slot_copy, n_async_down;
long n_bad;                               // launches with a buffer missing or too small
// launches: number and cost (ms) by kind
std::map<int, long> n_launch;
std::map<int, double> cost;
double now = 0.0;                         // the stream's clock
double drift = 1.0;                       // each launch costs so much of the one before
double speed = 1.0;
bool capturing = false;
double graph_ms = 0.0;

std::atomic<long> fail_new{-1};           // allocations until operator new throws

bool in(const std::map<char *, size_t> &m, const void *p)
{
    char *q = (char *)p;
    auto it = m.upper_bound(q);
    if (it == m.begin()) return false;
    --it;
    return q < it->first + it->second;
}

hipError_t ret(hipError_t e)
{
    if (e != hipSuccess) last_error = e;
    return e;
}

void launch(int kind)
{
    std::lock_guard<std::mutex> lk(mu);
    ++n_launch[kind];
    (capturing ? graph_ms : now) += (cost.count(kind) ? cost[kind] : 0.001) * speed;
    speed *= drift;
}

// whether p has room for so many bytes; counted when not
void need(const void *p, size_t bytes)
{
    std::lock_guard<std::mutex> lk(mu);
    auto it = device.upper_bound((char *)p);
    if (it != device.begin() && (--it, (char *)p + bytes <= it->first + it->second)) return;
    ++n_bad;
}

enum { K_OTHER = 0, K_GEOM = 1, K_SCAN = 2, K_REF_BATCHED = 3, K_MC_BATCHED = 4, K_MC_ITEMS = 5,
       K_REF = 6, K_MC = 7 };

}  // namespace

// ---- control ----------------------------------------------------------------
extern "C" {
void fake_reset()
{
    std::lock_guard<std::mutex> lk(mu);
    limit = ~size_t(0);
    fail_copy = -1;
    fail_new = -1;
    last_error = hipSuccess;
    pending.clear();
    n_malloc = n_copy = n_graph = n_sync = n_slot_copy = n_async_down = n_bad = 0;
    n_launch.clear();
    cost.clear();
    drift = speed = 1.0;
}
void fake_limit(size_t bytes) { limit = bytes == ~size_t(0) ? bytes : used + bytes; }
void fake_fail_copy(long n) { fail_copy = n; }
void fake_fail_new(long n) { fail_new = n; }
void fake_cost(int kind, double ms) { cost[kind] = ms; }
void fake_drift(double f) { drift = f; }
long fake_pending() { return (long)pending.size(); }
long fake_launches(int kind) { return n_launch[kind]; }
long fake_copies() { return n_copy; }
long fake_pinned_copies() { return n_slot_copy; }
long fake_graphs() { return n_graph; }
long fake_mallocs() { return n_malloc; }
long fake_async_downloads() { return n_async_down; }
long fake_bad_launches() { return n_bad; }
void *fake_pinned(size_t bytes)
{
    void *p = nullptr;
    return hipHostMalloc(&p, bytes, 0) == hipSuccess ? p : nullptr;
}
}

// ---- the runtime ------------------------------------------------------------
extern "C" {
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "injected"; }
hipError_t hipGetLastError()
{
    const hipError_t e = last_error;
    last_error = hipSuccess;
    return e;
}
hipError_t hipGetSymbolAddress(void **p, const void *)
{
    *p = nullptr;
    return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n)
{
    std::lock_guard<std::mutex> lk(mu);
    ++n_malloc;
    if (used + n > limit || !(*p = std::calloc(1, n))) return ret(hipErrorOutOfMemory);
    device[(char *)*p] = n;
    used += n;
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    std::lock_guard<std::mutex> lk(mu);
    auto it = device.find((char *)p);
    if (it == device.end()) return ret(hipErrorInvalidValue);
    used -= it->second;
    device.erase(it);
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    std::lock_guard<std::mutex> lk(mu);
    *p = std::calloc(1, n);
    pinned[(char *)*p] = n;
    return hipSuccess;
}
hipError_t hipHostFree(void *p)
{
    std::lock_guard<std::mutex> lk(mu);
    pinned.erase((char *)p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p)
{
    std::lock_guard<std::mutex> lk(mu);
    std::memset(a, 0, sizeof *a);
    if (in(pinned, p)) a->type = hipMemoryTypeHost;
    else if (in(device, p)) a->type = hipMemoryTypeDevice;
    else return ret(hipErrorInvalidValue);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t n, hipMemcpyKind kind, hipStream_t)
{
    std::lock_guard<std::mutex> lk(mu);
    ++n_copy;
    if (fail_copy >= 0 && fail_copy-- == 0) return ret(hipErrorUnknown);
    const void *host = kind == hipMemcpyHostToDevice ? src : dst;
    if (in(pinned, host)) ++n_slot_copy;
    else if (kind == hipMemcpyHostToDevice) pending.push_back({(const char *)src, n});
    else ++n_async_down;
    std::memmove(dst, src, n);
    return hipSuccess;
}
hipError_t hipMemcpy(void *dst, const void *src, size_t n, hipMemcpyKind kind)
{
    return hipMemcpyWithStream(dst, src, n, kind, nullptr);
}
hipError_t hipMemcpyWithStream(void *dst, const void *src, size_t n, hipMemcpyKind, hipStream_t s)
{
    {
        std::lock_guard<std::mutex> lk(mu);
        ++n_copy;
        if (fail_copy >= 0 && fail_copy-- == 0) return ret(hipErrorUnknown);
        std::memmove(dst, src, n);
    }
    return hipStreamSynchronize(s);
}
hipError_t hipStreamSynchronize(hipStream_t)
{
    std::lock_guard<std::mutex> lk(mu);
    ++n_sync;
    pending.clear();
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned)
{
    *s = (hipStream_t)std::calloc(1, 8);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) { std::free(s); return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = (hipEvent_t)std::calloc(1, 8); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { std::free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t)
{
    std::lock_guard<std::mutex> lk(mu);
    *(double *)e = now;
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b)
{
    *ms = (float)(*(double *)b - *(double *)a);
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode)
{
    capturing = true;
    graph_ms = 0.0;
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g)
{
    capturing = false;
    *g = (hipGraph_t)std::calloc(1, 8);
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t, hipGraphNode_t *, char *, size_t)
{
    ++n_graph;
    *x = (hipGraphExec_t)std::calloc(1, 8);
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t)
{
    now += graph_ms;
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) { std::free(g); return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t x) { std::free(x); return hipSuccess; }
void **__hipRegisterFatBinary(const void *) { static void *h; return &h; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
}

// the library's own allocations on the host
void *operator new(size_t n)
{
    if (fail_new >= 0 && fail_new-- == 0) throw std::bad_alloc();
    if (void *p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

// ---- the kernels ------------------------------------------------------------
namespace t2 {

int launch_stage_check(const float *xyz, int np, const int4 *, int, const int *, float4 *,
                       StageInfo *info, hipStream_t)
{
    launch(K_OTHER);
    StageInfo q{0u, 0u, {INFINITY, INFINITY, INFINITY}, {-INFINITY, -INFINITY, -INFINITY}};
    for (int p = 0; p < np; ++p)
        for (int a = 0; a < 3; ++a) {
            q.lo[a] = std::min(q.lo[a], xyz[3 * p + a]);
            q.hi[a] = std::max(q.hi[a], xyz[3 * p + a]);
        }
    info[0] = q;
    return 1;
}
size_t layout_scratch_words(int np, int nt) { return 6 * (size_t)np + 3 * (size_t)nt; }
size_t scan_sums_words(size_t n) { return n / 4096 + 2; }
void launch_layout(const float4 *, int, int, const StageBox &, const int4 *, int, const int *,
                   unsigned *, int *, int4 *, int *, int *, hipStream_t) { launch(K_OTHER); }
void launch_unpack_cc(const float4 *, const int *, int, float *, hipStream_t) { launch(K_OTHER); }
void launch_circumcenters(const float4 *, const int4 *, int, float4 *, hipStream_t) { launch(K_OTHER); }
void launch_exact_setup(const BlockIn &, const GridP &, int, const HashP &, unsigned *, unsigned *,
                        int2 *, float4 *, const int *, int *, int, unsigned *, unsigned char *,
                        hipStream_t) { launch(K_OTHER); }
void launch_owner(const GridP &gp, const HashP &, const unsigned *, const float4 *, int *owner, int,
                  unsigned *, const int *, int *, int, int *const *, const int *const *,
                  unsigned *defq, unsigned defq_cap, hipStream_t)
{
    launch(K_OTHER);
    need(owner, 4 * (size_t)gp.bnum_idx[0] * gp.bnum_idx[1] * gp.bnum_idx[2]);
    if (defq_cap) need(defq, 4 * (size_t)defq_cap);
}
void launch_exact_tail(const BlockIn &, const GridP &, const int *, const int *, const CellOut &,
                       int, int *const *, const int *const *, const Router *, int, int,
                       hipStream_t) { launch(K_OTHER); }
void launch_fill_u32(unsigned *p, size_t n, unsigned v, hipStream_t)
{
    launch(K_OTHER);
    need(p, 4 * n);
    std::fill(p, p + n, v);
}
void launch_ghost_sends(const float4 *, const int4 *, int, int, const float *, const float *,
                        const float *, int, int, unsigned long long *, hipStream_t) { launch(K_OTHER); }
void launch_device_block(const float *, int, const int4 *, int, const int *, float4 *, float4 *,
                         unsigned *, unsigned *, unsigned, hipStream_t) { launch(K_OTHER); }
void launch_run_prep(const BlockIn *, const CellOut *outs, int nb, int, unsigned long long,
                     const ZeroList &z, hipStream_t)
{
    launch(K_OTHER);
    for (int b = 0; b < nb; ++b) {
        const CellOut &o = outs[b];
        need(o.density, 4 * o.ngrid);
        need(o.count, 4 * o.ngrid);
        need(o.first, 8 * o.ngrid);
        need(o.second, 8 * o.ngrid);
        need(o.head, 4 * o.ngrid);
        need(o.slow, 4 * (size_t)o.slow_cap);
        need(o.ovf, 24 * (size_t)o.ovf_cap);
        need(o.seg, 24 * (size_t)o.ovf_cap);
        for (int k = 0; k < 3; ++k) need(o.fold[k], 16 * (size_t)o.fold_cap[k]);
    }
    for (int k = 0; k < 4; ++k)
        if (z.n[k]) {
            need(z.p[k], 4 * z.n[k]);
            std::fill(z.p[k], z.p[k] + z.n[k], 0u);
        }
}
void launch_cells_ref(const BlockIn &, const GridP &, const CellOut &, int, hipStream_t)
{
    launch(K_REF);
}
void launch_cells_ref_slow(const BlockIn &, const GridP &, const CellOut &, int, hipStream_t)
{
    launch(K_OTHER);
}
static void geom(int ntiles, const PlaneBuf &pb, int want_density)
{
    launch(K_GEOM);
    if (!want_density) return;
    const size_t n = (size_t)ntiles * CELL_TILE;
    need(pb.hdr, 32 * n);
    need(pb.fa, 16 * n * PLANE_STRIDE);
    need(pb.fb, 8 * n * PLANE_STRIDE);
    need(pb.big, 8 * n);
    need(pb.nbig, 4);
}
void launch_cell_geom(const CellSet<false> &set, const PlaneBuf &pb, int want_density, hipStream_t)
{
    geom(set.ntiles, pb, want_density);
}
void launch_cell_geom(const CellSet<true> &set, const PlaneBuf &pb, int want_density, hipStream_t)
{
    geom(set.ntiles, pb, want_density);
}
void launch_cell_scan(const CellSet<false> &, const PlaneBuf &, hipStream_t) { launch(K_SCAN); }
void launch_cell_scan(const CellSet<true> &, const PlaneBuf &, hipStream_t) { launch(K_SCAN); }
int launch_cells_mc(const BlockIn &, const GridP *, const CellOut &, int, int, hipStream_t)
{
    launch(K_MC);
    return 0;
}
void launch_cells_ref_slow_batched(const BlockIn *, const Router *, int, hipStream_t)
{
    launch(K_OTHER);
}
void launch_cells_mc_items(const BlockIn *, const GridP *, const CellOut *, const Router *,
                           const Chunk *, const XcdQueues &, int, hipStream_t)
{
    launch(K_MC_ITEMS);
}
void launch_cells_mc_batched(const BlockIn *, const GridP *, const CellOut *, const Router *,
                             const Chunk *, const XcdQueues &, unsigned *, int, int, hipStream_t)
{
    launch(K_MC_BATCHED);
}
void launch_cic(const BlockIn &, const GridP &, const CellOut &, const Router *, int, hipStream_t)
{
    launch(K_OTHER);
}
void launch_cells_ref_batched(const BlockIn *, const GridP *, const CellOut *, const Router *,
                              const Chunk *, const XcdQueues &, unsigned *, int, int, hipStream_t,
                              bool)
{
    launch(K_REF_BATCHED);
}
void launch_fold(const CellOut *, const GridP *, int, unsigned, const unsigned[3],
                 unsigned long long, unsigned long long, hipStream_t) { launch(K_OTHER); }
void launch_run_finish(const CellOut *, const GridP *, RunPart *, int, int, unsigned long long,
                       hipStream_t) { launch(K_OTHER); }

}  // namespace t2
