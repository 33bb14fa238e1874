// batch.hip -- many voxelizations in one graph launch (vox_batch_* C-ABI).
//
// vox_batch_create sorts the jobs into algorithm classes (fill, chunk,
// marker, direct surface/solid, tile surface/solid), uploads one device array of job
// descriptors per class together with the per-job prefix of each kernel's
// work units, allocates one workspace, and captures the whole pipeline --
// every kernel processing all jobs of its class at once -- into a HIP graph.
// vox_batch_launch then costs one hipGraphLaunch per batch, however many
// meshes it holds.
#include <hip/hip_runtime.h>

#include <cstring>
#include <mutex>
#include <new>
#include <string>
#include <vector>

#include "../../include/cuda_voxelizer_amd/vox_capi.h"
#include "vox_host.h"
#include "scratch.h"
#include "vox_kernels.h"

namespace voxamd {

struct JobClass {
    std::vector<ItemDev> items;
    std::vector<uint32_t> base_a, base_b, base_c;  // prefixes (class dependent)
    ItemMap m_a{}, m_b{}, m_c{};
    uint32_t total_a = 0, total_b = 0, total_c = 0;
    uint32_t max_tile_words = 0;
    bool loop = false;  // chunk class: some job takes several chunks per workgroup
    bool split = false; // chunk class: some job's triangles are shared by several lanes
    size_t off_items = 0, off_a = 0, off_b = 0, off_c = 0;
};

}  // namespace voxamd

struct vox_batch {
    int device = 0;
    bool use_graph = true;
    hipStream_t cap_stream = nullptr;
    hipStream_t side[4] = {};  // capture only: tile chain, marker chain, direct classes, fill and its chunk classes
    hipEvent_t ev[6] = {};     // capture only: fork, tables zeroed, and the four side branches' ends
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    void* dev_mem = nullptr;
    void* ws = nullptr;
    void* mws = nullptr;  // marker class: spill records and counters
    void* sws = nullptr;  // blocked chunk class: the jobs' scratch tables, all zero between launches
    uint64_t scratch_bytes = 0;
    // Launches on different streams share the workspaces, so each waits for the one
    // before.  Only a batch that has been launched on a second stream records an
    // event after each launch (48 mixed meshes: 396 us a launch, 400 with it).
    std::mutex use;
    voxamd::StreamKey last;
    bool launched = false;
    hipEvent_t done = nullptr;
    bool scratch_dirty = false;  // a launch failed between the scratch tables' use and their clearing
    voxamd::WorkspaceLayout L{};
    // chunk: one class per layout specialisation (ChunkSpec); chunkw: layout-generic jobs at 6 waves per SIMD
    voxamd::JobClass fill, chunk[voxamd::kBlockedSpecs], chunkw, unblock, marker, dsurf, dsolid, tsurf, tsolid;
    int count = 0;
    uint64_t total_triangles = 0;
};

namespace voxamd {

static void add_prefix(std::vector<uint32_t>& base, uint32_t& total, uint64_t units) {
    if (base.empty()) base.push_back(0);
    total += (uint32_t)units;
    base.push_back(total);
}

// The classes of a batch, by the launch that runs them.  Every job is in one
// algorithm class; the fill class zeroes the tables of the chunk, marker and
// direct jobs that do not accumulate (tile jobs write every word themselves).
static hipError_t launch_fill_class(vox_batch* b, hipStream_t s) {
    const ItemDev dummy{};
    if (!b->fill.total_a) return hipSuccess;
    return launch_fill_jobs(dummy, b->fill.m_a, b->fill.total_a, s);
}

// Which chunk classes a launch covers: those whose tables are zero-filled
// before, or the blocked one, whose scratch tables are zero already and whose
// tables the unblock pass then writes.
enum ChunkClassSet { kFilledChunkClasses, kBlockedChunkClass };

static hipError_t launch_chunk_classes(vox_batch* b, hipStream_t s, ChunkClassSet which) {
    const ItemDev dummy{};
    hipError_t e = hipSuccess;
    for (int sp = 0; sp < kBlockedSpecs; sp++) {
        if ((which == kBlockedChunkClass) != (sp == kSpecBlocked)) continue;
        const JobClass& c = b->chunk[sp];
        if (c.total_a && (e = launch_chunk_jobs(dummy, c.m_a, c.total_a, c.loop, s, 5, sp, c.split)) != hipSuccess)
            return e;
    }
    const JobClass& w = b->chunkw;
    if (which == kFilledChunkClasses && w.total_a &&
        (e = launch_chunk_jobs(dummy, w.m_a, w.total_a, w.loop, s, 6, kSpecAny, w.split)) != hipSuccess)
        return e;
    if (which == kBlockedChunkClass) return launch_unblock_jobs(dummy, b->unblock.m_a, b->unblock.total_a, s);
    return hipSuccess;
}

static hipError_t launch_marker_class(vox_batch* b, hipStream_t s) {
    if (b->marker.items.empty()) return hipSuccess;
    return launch_marker_jobs(b->marker.m_a, b->marker.m_b, b->marker.m_c, b->marker.total_a, b->marker.total_b,
                              b->mws, s);
}

static hipError_t launch_direct_classes(vox_batch* b, hipStream_t s) {
    const ItemDev dummy{};
    hipError_t e = hipSuccess;
    if (b->dsurf.total_a && (e = launch_direct_jobs(dummy, b->dsurf.m_a, b->dsurf.total_a, false, s)) != hipSuccess)
        return e;
    if (b->dsolid.total_a && (e = launch_direct_jobs(dummy, b->dsolid.m_a, b->dsolid.total_a, true, s)) != hipSuccess)
        return e;
    return hipSuccess;
}

// The two tile classes share the binning workspace: one after the other.
static hipError_t launch_tile_classes(vox_batch* b, hipStream_t s) {
    const ItemDev dummy{};
    hipError_t e = hipSuccess;
    if (!b->tsurf.items.empty() &&
        (e = launch_tiled_jobs(dummy, b->tsurf.m_a, b->tsurf.m_b, b->tsurf.m_c, b->tsurf.total_a, b->tsurf.total_b,
                               false, b->tsurf.max_tile_words, b->ws, b->L, s)) != hipSuccess)
        return e;
    if (!b->tsolid.items.empty() &&
        (e = launch_tiled_jobs(dummy, b->tsolid.m_a, b->tsolid.m_b, b->tsolid.m_c, b->tsolid.total_a,
                               b->tsolid.total_b, true, b->tsolid.max_tile_words, b->ws, b->L, s)) != hipSuccess)
        return e;
    return hipSuccess;
}

// Every class in stream order (eager launches and runners).
static hipError_t launch_all(vox_batch* b, hipStream_t s) {
    hipError_t e = hipSuccess;
    if ((e = launch_fill_class(b, s)) != hipSuccess) return e;
    if ((e = launch_chunk_classes(b, s, kBlockedChunkClass)) != hipSuccess) return e;
    if ((e = launch_chunk_classes(b, s, kFilledChunkClasses)) != hipSuccess) return e;
    if ((e = launch_marker_class(b, s)) != hipSuccess) return e;
    if ((e = launch_direct_classes(b, s)) != hipSuccess) return e;
    return launch_tile_classes(b, s);
}

// For graph capture on `m`: classes that touch different jobs run as
// concurrent branches, so one class's tail (its last workgroups) and the
// small latency-bound kernels (the tile chain's scans, the chunk loop of
// small dense tables, the marker chain's spill pass) overlap the others
// instead of leaving the GPU idle between kernels.  Nodes are created in the
// order the critical path wants them dispatched: the fill, then the longer of
// the two chunk chains on `m` (the classes that need the fill, or the blocked one
// and its unblock pass, which does not), the other on a branch, and the tile
// chain (no fill), the marker chain and the direct classes.  A launch of 13 mixed
// meshes whose longest job is a soup of 269,272 at 32^3 takes 125 us with the
// filled chain first, 157 with the blocked one; of 31 171 and 202; of 36 208 and
// 191, of 48 442 and 423.  `m` joins every branch at the end.  Tables of different
// jobs do not overlap, so the branches share no data (the out-of-row counters they
// add to are atomic).
static hipError_t launch_forked(vox_batch* b, hipStream_t m) {
    hipError_t e = hipSuccess;
    uint64_t filled = 0, blocked = 0;  // triangles of the two chunk chains
    for (int sp = 0; sp < kBlockedSpecs; sp++)
        for (const ItemDev& it : b->chunk[sp].items) (sp == kSpecBlocked ? blocked : filled) += it.info.n_triangles;
    for (const ItemDev& it : b->chunkw.items) filled += it.info.n_triangles;
    const bool filled_first = 2 * filled >= blocked;
    hipStream_t fs = filled_first ? m : b->side[3], bs = filled_first ? b->side[3] : m;
#define VOX_TRY(x) \
    if ((e = (x)) != hipSuccess) return e
    VOX_TRY(hipEventRecord(b->ev[0], m));
    VOX_TRY(hipStreamWaitEvent(b->side[3], b->ev[0], 0));
    VOX_TRY(launch_fill_class(b, fs));
    VOX_TRY(hipEventRecord(b->ev[1], fs));
    if (filled_first) VOX_TRY(launch_chunk_classes(b, fs, kFilledChunkClasses));
    VOX_TRY(launch_chunk_classes(b, bs, kBlockedChunkClass));
    VOX_TRY(hipStreamWaitEvent(b->side[0], b->ev[0], 0));
    VOX_TRY(launch_tile_classes(b, b->side[0]));
    VOX_TRY(hipEventRecord(b->ev[2], b->side[0]));
    VOX_TRY(hipStreamWaitEvent(b->side[1], b->ev[1], 0));
    VOX_TRY(launch_marker_class(b, b->side[1]));
    VOX_TRY(hipEventRecord(b->ev[3], b->side[1]));
    VOX_TRY(hipStreamWaitEvent(b->side[2], b->ev[1], 0));
    VOX_TRY(launch_direct_classes(b, b->side[2]));
    VOX_TRY(hipEventRecord(b->ev[4], b->side[2]));
    if (!filled_first) VOX_TRY(launch_chunk_classes(b, fs, kFilledChunkClasses));
    VOX_TRY(hipEventRecord(b->ev[5], b->side[3]));
    for (int k = 2; k < 6; k++) VOX_TRY(hipStreamWaitEvent(m, b->ev[k], 0));
#undef VOX_TRY
    return hipSuccess;
}

static void free_batch(vox_batch* b) {
    if (!b) return;
    if (b->exec) (void)hipGraphExecDestroy(b->exec);
    if (b->graph) (void)hipGraphDestroy(b->graph);
    if (b->cap_stream) (void)hipStreamDestroy(b->cap_stream);
    for (hipStream_t& st : b->side)
        if (st) (void)hipStreamDestroy(st);
    for (hipEvent_t& ev : b->ev)
        if (ev) (void)hipEventDestroy(ev);
    if (b->done) (void)hipEventDestroy(b->done);
    if (b->dev_mem) (void)hipFree(b->dev_mem);
    if (b->ws) (void)hipFree(b->ws);
    if (b->mws) (void)hipFree(b->mws);
    if (b->sws) (void)hipFree(b->sws);
    delete b;
}

// Host side of a batch: jobs sorted into algorithm classes, the packed
// device image of the descriptor and prefix arrays, and the workspace needed.
struct BatchPlan {
    std::vector<char> host;
    bool ws_needed = false;
    WorkspaceLayout L{};
    uint64_t scratch = 0;  // bytes of blocked scratch tables; the jobs hold their offsets until place_scratch
};

// A batch's scratch tables together; jobs beyond it go to their tables directly, as
// all do where the device has no room for them.
constexpr uint64_t kBatchScratch = 1ull << 30;

// Every chunk class and the others, in the order of the packed image.
constexpr int kClasses = kBlockedSpecs + 8;
struct ClassList {
    JobClass* c[kClasses];
    explicit ClassList(vox_batch* b) {
        int k = 0;
        c[k++] = &b->fill;
        for (JobClass& j : b->chunk) c[k++] = &j;
        for (JobClass* j : {&b->chunkw, &b->unblock, &b->marker, &b->dsurf, &b->dsolid, &b->tsurf, &b->tsolid}) c[k++] = j;
    }
    JobClass** begin() { return c; }
    JobClass** end() { return c + kClasses; }
};

// The scratch offsets in the packed image become pointers.
static void place_scratch(vox_batch* b, BatchPlan& plan) {
    for (JobClass* c : {&b->chunk[kSpecBlocked], &b->unblock}) {
        ItemDev* it = (ItemDev*)(plan.host.data() + c->off_items);
        for (size_t i = 0; i < c->items.size(); i++) it[i].scratch = (uint32_t*)((char*)b->sws + (uintptr_t)it[i].scratch);
    }
}

static void reset_classes(vox_batch* b) {
    ClassList classes(b);
    for (JobClass* c : classes) *c = JobClass{};
    b->count = 0;
    b->total_triangles = 0;
}

// Workgroups for which a job of large triangles shares them (0: not shared); see
// chunk_batch_shape.
static uint32_t shared_groups(const vox_batch_item* items, int count) {
    uint64_t triangles = 0, jobs = 0;
    for (int i = 0; i < count; i++) {
        if (items[i].solid) continue;
        triangles += items[i].info.n_triangles;
        jobs += chunk_large(items[i].info.gridsize[0], items[i].info.n_triangles) ? 1u : 0u;
    }
    if (triangles > kSharedBatch || jobs == 0) return 0u;
    const uint64_t groups = 1024u / jobs;
    return groups > 512u ? 512u : (groups < 64u ? 64u : (uint32_t)groups);
}

static vox_status plan_batch(const vox_batch_item* items, int count, vox_batch* b, BatchPlan& plan,
                             uint64_t scratch_limit) {
    if (count < 0 || (count > 0 && !items)) return fail(VOX_ERR_INVALID, "bad item array");
    reset_classes(b);
    b->count = count;
    uint64_t tri_sum_surf = 0, tri_sum_solid = 0;
    const uint32_t share = shared_groups(items, count);
    for (int i = 0; i < count; i++) {
        const vox_batch_item& it = items[i];
        vox_status s = validate(&it.info, it.d_tris, it.d_table, it.layout);
        if (s != VOX_OK) return fail(s, "item " + std::to_string(i) + ": " + vox_last_error());
        const unsigned algo =
            it.flags & (VOX_FLAG_ALGO_DIRECT | VOX_FLAG_ALGO_TILE | VOX_FLAG_ALGO_CHUNK | VOX_FLAG_ALGO_MARKER);
        const bool solid = it.solid != 0;
        if ((algo & (algo - 1)) || (solid && (algo & VOX_FLAG_ALGO_CHUNK)) || (!solid && (algo & VOX_FLAG_ALGO_MARKER)))
            return fail(VOX_ERR_INVALID, "item " + std::to_string(i) + ": bad algorithm flags");
        const uint32_t G = it.info.gridsize[0];
        const bool accumulate = (it.flags & VOX_FLAG_ACCUMULATE) != 0;
        TilePlan P;
        const bool have_plan =
            make_plan((int)G, it.layout, solid, P, tune_tile_scale(it.flags)) || make_plan((int)G, it.layout, solid, P);
        // the marker class tags spill records with the job index (below 2^22)
        const bool have_marker = solid && marker_batch_supported(G, it.layout, accumulate) && i < (1 << 22);
        enum { DIRECT, TILE, CHUNK, MARKER } a;
        if (algo & VOX_FLAG_ALGO_DIRECT) a = DIRECT;
        else if (algo & VOX_FLAG_ALGO_TILE) a = have_plan ? TILE : DIRECT;
        else if (algo & VOX_FLAG_ALGO_CHUNK) a = chunk_supported(G) ? CHUNK : DIRECT;
        else if (algo & VOX_FLAG_ALGO_MARKER) a = have_marker ? MARKER : (have_plan ? TILE : DIRECT);
        else if (solid && prefer_direct_solid(it.info.n_triangles, G)) a = DIRECT;
        else if (solid && have_plan && prefer_tile_solid(it.layout, accumulate, it.info.n_triangles, G)) a = TILE;
        else if (solid && have_marker) a = MARKER;
        else if (solid) a = have_plan ? TILE : DIRECT;
        else a = chunk_supported(G) ? CHUNK : (have_plan ? TILE : DIRECT);
        ItemDev d{};
        d.info = it.info;
        d.tris = it.d_tris;
        d.table = it.d_table;
        d.offrow = (unsigned long long*)it.d_offrow;
        d.layout = it.layout;
        d.solid = solid ? 1 : 0;
        d.accumulate = accumulate ? 1 : 0;
        d.big = tune_big(it.flags);
        const uint64_t n = it.info.n_triangles;
        b->total_triangles += n;
        const uint64_t table_bytes = blocked_bytes(G);
        // 48 mixed meshes, linear keys -> blocked: 740 -> 405 us a launch
        const bool blocked = a == CHUNK && !(it.flags & VOX_FLAG_NO_SCRATCH) && G <= kBatchBlockedGrid &&
                             chunk_blocked(it.layout, G, n, accumulate) &&
                             plan.scratch + table_bytes <= scratch_limit;
        if (a != TILE && !accumulate && !blocked) {
            b->fill.items.push_back(d);
            add_prefix(b->fill.base_a, b->fill.total_a, fill_units(G));
        }
        if (a == MARKER) {
            if ((uint64_t)b->marker.total_c + n > 0xFFFFFFFFull)
                return fail(VOX_ERR_UNSUPPORTED, "more than 2^32-1 triangles in one marker batch class");
            const uint32_t units = marker_block_units(d);
            b->marker.items.push_back(d);
            add_prefix(b->marker.base_a, b->marker.total_a, units);
            add_prefix(b->marker.base_b, b->marker.total_b, marker_row_units(G));
            add_prefix(b->marker.base_c, b->marker.total_c, n);  // triangles (spill overflow pass)
        } else if (a == CHUNK) {
            d.span = chunk_span(G, n, false);
            if (d.span <= 1u) chunk_batch_shape(d, share);
            // jobs that loop over chunks run in the 4-wave form (any layout): they stay in the 5-wave class;
            // a layout-specialised kernel runs at six waves per SIMD under either bound, so only
            // layout-generic jobs are split by the waves knob (each class is one more kernel)
            const bool loop = d.span > 1u && d.parts <= 1u;
            const int sp = blocked ? (int)kSpecBlocked : (loop ? (int)kSpecAny : chunk_spec(it.layout, G));
            if (blocked) {
                d.scratch = (uint32_t*)(uintptr_t)plan.scratch;
                plan.scratch += (table_bytes + 255u) & ~255ull;
                b->unblock.items.push_back(d);
                add_prefix(b->unblock.base_a, b->unblock.total_a, unblock_units(G, it.d_table));
            }
            const bool wide = tune_waves(it.flags) == 6 && !loop && sp == kSpecAny;
            JobClass& c = wide ? b->chunkw : b->chunk[sp];
            if (loop) c.loop = true;
            if (d.lg_split) c.split = true;
            c.items.push_back(d);
            add_prefix(c.base_a, c.total_a, chunk_units(n, d.span, d.parts, d.lg_split));
        } else if (a == DIRECT) {
            JobClass& c = solid ? b->dsolid : b->dsurf;
            c.items.push_back(d);
            add_prefix(c.base_a, c.total_a, direct_units(n));
        } else {
            JobClass& c = solid ? b->tsolid : b->tsurf;
            uint64_t& tri_sum = solid ? tri_sum_solid : tri_sum_surf;
            d.P = P;
            d.tile_base = c.total_b;
            d.tri_base = tri_sum;
            if (tri_sum + n > 0xFFFFFFFFull)
                return fail(VOX_ERR_UNSUPPORTED, "more than 2^32-1 triangles in one tiled batch class");
            tri_sum += n;
            c.items.push_back(d);
            add_prefix(c.base_a, c.total_a, (n + 255) / 256);  // bin blocks
            add_prefix(c.base_b, c.total_b, (uint64_t)P.ntiles);
            add_prefix(c.base_c, c.total_c, n);                 // triangles
            if ((uint32_t)P.tile_words > c.max_tile_words) c.max_tile_words = (uint32_t)P.tile_words;
        }
    }
    // one device allocation: per class the job array and its prefix arrays
    ClassList classes(b);
    size_t total = 0;
    auto reserve = [&](size_t bytes) {
        const size_t off = total;
        total = (total + bytes + 255) & ~(size_t)255;
        return off;
    };
    for (JobClass* c : classes) {
        c->off_items = reserve(c->items.size() * sizeof(ItemDev));
        c->off_a = reserve(c->base_a.size() * 4);
        c->off_b = reserve(c->base_b.size() * 4);
        c->off_c = reserve(c->base_c.size() * 4);
    }
    std::vector<char>& host = plan.host;
    host.assign(total > 0 ? total : 1, 0);
    for (JobClass* c : classes) {
        if (!c->items.empty()) std::memcpy(host.data() + c->off_items, c->items.data(), c->items.size() * sizeof(ItemDev));
        if (!c->base_a.empty()) std::memcpy(host.data() + c->off_a, c->base_a.data(), c->base_a.size() * 4);
        if (!c->base_b.empty()) std::memcpy(host.data() + c->off_b, c->base_b.data(), c->base_b.size() * 4);
        if (!c->base_c.empty()) std::memcpy(host.data() + c->off_c, c->base_c.data(), c->base_c.size() * 4);
    }
    if (!b->tsurf.items.empty() || !b->tsolid.items.empty()) {
        const uint64_t tiles = b->tsurf.total_b > b->tsolid.total_b ? b->tsurf.total_b : b->tsolid.total_b;
        const uint64_t tris = tri_sum_surf > tri_sum_solid ? tri_sum_surf : tri_sum_solid;
        plan.ws_needed = true;
        plan.L = workspace_layout((tiles + 4095) & ~4095ull, tris > 4096 ? tris : 4096, 8);
    }
    return VOX_OK;
}

// Point every class's job maps at a device copy of the packed image.
static void bind_maps(vox_batch* b, void* dev) {
    char* dm = (char*)dev;
    ClassList classes(b);
    for (JobClass* c : classes) {
        const ItemDev* it = (const ItemDev*)(dm + c->off_items);
        const int ni = (int)c->items.size();
        c->m_a = ItemMap{it, (const uint32_t*)(dm + c->off_a), ni, 0};
        c->m_b = ItemMap{it, (const uint32_t*)(dm + c->off_b), ni, 0};
        c->m_c = ItemMap{it, (const uint32_t*)(dm + c->off_c), ni, 0};
    }
}

}  // namespace voxamd

using namespace voxamd;

extern "C" {

static vox_status create_batch(const vox_batch_item* items, int count, unsigned flags, uint64_t scratch_limit,
                               uint64_t& scratch, vox_batch** out) {
    vox_batch* b = new (std::nothrow) vox_batch();
    if (!b) return fail(VOX_ERR_OOM, "host allocation");
    b->use_graph = !(flags & VOX_BATCH_NO_GRAPH);
    hipError_t e = hipGetDevice(&b->device);
    if (e != hipSuccess) {
        free_batch(b);
        return hip_fail(e, "hipGetDevice");
    }
    BatchPlan plan;
    vox_status s = plan_batch(items, count, b, plan, scratch_limit);
    if (s != VOX_OK) {
        free_batch(b);
        return s;
    }
    scratch = plan.scratch;
    if (plan.scratch) {
        e = hipMalloc(&b->sws, plan.scratch);
        if (e == hipSuccess) e = hipMemset(b->sws, 0, plan.scratch);
        if (e != hipSuccess) {
            free_batch(b);
            return fail(VOX_ERR_OOM, std::string("batch scratch tables: ") + hipGetErrorString(e));
        }
        b->scratch_bytes = plan.scratch;
        place_scratch(b, plan);
    }
    e = hipMalloc(&b->dev_mem, plan.host.size());
    if (e != hipSuccess) {
        free_batch(b);
        return fail(VOX_ERR_OOM, std::string("batch descriptors: ") + hipGetErrorString(e));
    }
    e = hipMemcpy(b->dev_mem, plan.host.data(), plan.host.size(), hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        free_batch(b);
        return hip_fail(e, "batch descriptor upload");
    }
    bind_maps(b, b->dev_mem);
    if (!b->marker.items.empty()) {
        e = hipMalloc(&b->mws, marker_ws_bytes());
        if (e == hipSuccess) e = hipMemset(b->mws, 0, marker_ws_bytes());  // counters start at zero
        if (e != hipSuccess) {
            free_batch(b);
            return fail(VOX_ERR_OOM, std::string("batch marker workspace: ") + hipGetErrorString(e));
        }
    }
    if (plan.ws_needed) {
        b->L = plan.L;
        e = hipMalloc(&b->ws, b->L.total);
        if (e == hipSuccess) e = hipMemset(b->ws, 0, b->L.total);
        if (e != hipSuccess) {
            free_batch(b);
            return fail(VOX_ERR_OOM, std::string("batch workspace: ") + hipGetErrorString(e));
        }
    }
    if (b->use_graph) {
        e = hipStreamCreateWithFlags(&b->cap_stream, hipStreamNonBlocking);
        for (hipStream_t& st : b->side)
            if (e == hipSuccess) e = hipStreamCreateWithFlags(&st, hipStreamNonBlocking);
        for (hipEvent_t& ev : b->ev)
            if (e == hipSuccess) e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
        if (e == hipSuccess) e = hipStreamBeginCapture(b->cap_stream, hipStreamCaptureModeThreadLocal);
        if (e == hipSuccess) {
            hipError_t le = launch_forked(b, b->cap_stream);
            e = hipStreamEndCapture(b->cap_stream, &b->graph);
            if (le != hipSuccess) e = le;
        }
        if (e == hipSuccess) e = hipGraphInstantiate(&b->exec, b->graph, nullptr, nullptr, 0);
        if (e != hipSuccess) {
            free_batch(b);
            return hip_fail(e, "batch graph capture");
        }
    }
    *out = b;
    return VOX_OK;
}

vox_status vox_batch_create(const vox_batch_item* items, int count, unsigned flags, vox_batch** out) {
    if (!out) return fail(VOX_ERR_INVALID, "out is NULL");
    *out = nullptr;
    uint64_t scratch = 0;
    vox_status s = create_batch(items, count, flags, kBatchScratch, scratch, out);
    if (s == VOX_ERR_OOM && scratch) {  // the scratch tables are optional
        (void)hipGetLastError();
        s = create_batch(items, count, flags, 0, scratch, out);
    }
    return s;
}

vox_status vox_batch_launch(vox_batch* b, void* stream) {
    if (!b) return fail(VOX_ERR_INVALID, "batch is NULL");
    hipStream_t st = (hipStream_t)stream;
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    hipError_t e = hipSuccess;
    std::lock_guard<std::mutex> lock(b->use);
    // a captured launch (of a batch without a graph) is ordered by its graph's user
    const bool shared = b->sws || b->ws || b->mws;
    if (shared) e = hipStreamIsCapturing(st, &cap);
    const bool ordered = shared && cap == hipStreamCaptureStatusNone;
    StreamKey key;
    if (e == hipSuccess && ordered) e = stream_key(st, key);
    if (e == hipSuccess && ordered && b->launched && !(key == b->last)) {
        if (b->done) {
            e = hipStreamWaitEvent(st, b->done, 0);
        } else {
            e = wait_for_device();
            if (e == hipErrorOutOfMemory) {  // it has none to free
                (void)hipGetLastError();
                e = hipDeviceSynchronize();
            }
            if (e == hipSuccess) e = hipEventCreateWithFlags(&b->done, hipEventDisableTiming);
        }
    }
    if (e == hipSuccess && ordered && b->scratch_dirty) e = hipMemsetAsync(b->sws, 0, b->scratch_bytes, st);
    if (e != hipSuccess) return hip_fail(e, "batch launch");
    e = b->use_graph ? hipGraphLaunch(b->exec, st) : launch_all(b, st);
    if (ordered) {  // also after a failure: some kernels may have been launched
        b->scratch_dirty = b->sws && e != hipSuccess;
        b->last = key;
        b->launched = true;
        if (b->done && hipEventRecord(b->done, st) != hipSuccess) (void)hipDeviceSynchronize();
    }
    if (e != hipSuccess) return hip_fail(e, "batch launch");
    return VOX_OK;
}

vox_status vox_batch_info(const vox_batch* b, int64_t out[8]) {
    if (!b || !out) return fail(VOX_ERR_INVALID, "NULL argument");
    out[0] = b->count;
    out[1] = (int64_t)b->total_triangles;
    out[2] = 0;
    for (const JobClass& c : b->chunk) out[2] += (int64_t)c.items.size();
    out[2] += (int64_t)b->chunkw.items.size();
    out[3] = (int64_t)b->tsurf.items.size();
    out[4] = (int64_t)b->tsolid.items.size();
    out[5] = (int64_t)(b->dsurf.items.size() + b->dsolid.items.size());
    out[6] = b->use_graph ? 1 : 0;
    out[7] = (int64_t)(b->L.total + b->scratch_bytes);
    return VOX_OK;
}

vox_status vox_batch_destroy(vox_batch* b) {
    if (!b) return VOX_OK;
    (void)hipDeviceSynchronize();  // launches of this batch may still be in flight on caller streams
    free_batch(b);
    return VOX_OK;
}

}  // extern "C"

// ---------------------------------------------------------------------------
// vox_runner: a re-fillable eager batch bound to one stream (serving)
// ---------------------------------------------------------------------------
struct vox_runner {
    vox_batch b;                 // classes, job maps, workspace (eager launches)
    hipStream_t stream = nullptr;
    void* dev_desc = nullptr;
    size_t dev_cap = 0;
    void* pinned[2] = {nullptr, nullptr};
    size_t pinned_cap[2] = {0, 0};
    hipEvent_t ev[2] = {nullptr, nullptr};
    int slot = 0;
    uint64_t tiles_cap = 0, n_cap = 0;
    uint64_t scratch_cap = 0;
    uint64_t scratch_limit = kBatchScratch;  // 0 once the device had no room
    uint64_t launches = 0;
};

extern "C" {

vox_status vox_runner_create(void* stream, vox_runner** out) {
    if (!out) return fail(VOX_ERR_INVALID, "out is NULL");
    *out = nullptr;
    vox_runner* r = new (std::nothrow) vox_runner();
    if (!r) return fail(VOX_ERR_OOM, "host allocation");
    r->stream = (hipStream_t)stream;
    r->b.use_graph = false;
    hipError_t e = hipGetDevice(&r->b.device);
    for (int i = 0; i < 2 && e == hipSuccess; i++) e = hipEventCreateWithFlags(&r->ev[i], hipEventDisableTiming);
    if (e != hipSuccess) {
        vox_runner_destroy(r);
        return hip_fail(e, "runner setup");
    }
    *out = r;
    return VOX_OK;
}

// The launch's plan, and the device buffers that it needs.
static vox_status prepare_launch(vox_runner* r, const vox_batch_item* items, int count, BatchPlan& plan) {
    vox_status s = plan_batch(items, count, &r->b, plan, r->scratch_limit);
    if (s != VOX_OK) return s;
    hipError_t e;
    // grow-only device buffers; growing waits for this runner's stream
    const uint64_t tiles = r->b.tsurf.total_b > r->b.tsolid.total_b ? r->b.tsurf.total_b : r->b.tsolid.total_b;
    uint64_t tris = 0;
    if (!r->b.tsurf.base_c.empty()) tris = r->b.tsurf.base_c.back();
    if (!r->b.tsolid.base_c.empty() && r->b.tsolid.base_c.back() > tris) tris = r->b.tsolid.base_c.back();
    const bool grow_ws = plan.ws_needed && (tiles > r->tiles_cap || tris > r->n_cap || !r->b.ws);
    const bool grow_desc = plan.host.size() > r->dev_cap;
    const bool grow_scratch = plan.scratch > r->scratch_cap;
    if (grow_ws || grow_desc || grow_scratch) {
        e = hipStreamSynchronize(r->stream);
        if (e != hipSuccess) return hip_fail(e, "hipStreamSynchronize");
    }
    if (grow_ws) {
        if (r->b.ws) (void)hipFree(r->b.ws);
        r->b.ws = nullptr;
        r->tiles_cap = ((tiles > r->tiles_cap ? tiles : r->tiles_cap) + 4095) & ~4095ull;
        r->n_cap = tris > r->n_cap ? tris : r->n_cap;
        if (r->n_cap < 4096) r->n_cap = 4096;
        r->b.L = workspace_layout(r->tiles_cap, r->n_cap, 8);
        e = hipMalloc(&r->b.ws, r->b.L.total);
        if (e == hipSuccess) e = hipMemset(r->b.ws, 0, r->b.L.total);
        if (e != hipSuccess) {
            r->tiles_cap = r->n_cap = 0;
            return fail(VOX_ERR_OOM, std::string("runner workspace: ") + hipGetErrorString(e));
        }
    }
    if (grow_scratch) {
        if (r->b.sws) (void)hipFree(r->b.sws);
        r->b.sws = nullptr;
        r->scratch_cap = 0;
        e = hipMalloc(&r->b.sws, plan.scratch);
        if (e != hipSuccess) {
            r->b.sws = nullptr;
            return fail(VOX_ERR_OOM, std::string("runner scratch tables: ") + hipGetErrorString(e));
        }
        r->scratch_cap = plan.scratch;
        r->b.scratch_dirty = true;
    }
    if (plan.scratch) {
        if (r->b.scratch_dirty) {
            e = hipMemsetAsync(r->b.sws, 0, r->scratch_cap, r->stream);
            if (e != hipSuccess) return hip_fail(e, "runner scratch tables");
        }
        place_scratch(&r->b, plan);
    }
    if (!r->b.marker.items.empty() && !r->b.mws) {  // fixed size, allocated once
        e = hipMalloc(&r->b.mws, marker_ws_bytes());
        if (e == hipSuccess) e = hipMemset(r->b.mws, 0, marker_ws_bytes());  // counters start at zero
        if (e != hipSuccess) {
            if (r->b.mws) (void)hipFree(r->b.mws);
            r->b.mws = nullptr;
            return fail(VOX_ERR_OOM, std::string("runner marker workspace: ") + hipGetErrorString(e));
        }
    }
    if (grow_desc) {
        if (r->dev_desc) (void)hipFree(r->dev_desc);
        r->dev_cap = plan.host.size() * 2;
        e = hipMalloc(&r->dev_desc, r->dev_cap);
        if (e != hipSuccess) {
            r->dev_cap = 0;
            r->dev_desc = nullptr;
            return fail(VOX_ERR_OOM, std::string("runner descriptors: ") + hipGetErrorString(e));
        }
    }
    return VOX_OK;
}

vox_status vox_runner_launch(vox_runner* r, const vox_batch_item* items, int count) {
    if (!r) return fail(VOX_ERR_INVALID, "runner is NULL");
    BatchPlan plan;
    vox_status s = prepare_launch(r, items, count, plan);
    if (s == VOX_ERR_OOM && (plan.scratch || r->b.sws)) {  // the scratch tables are optional
        (void)hipGetLastError();
        hipError_t w = hipStreamSynchronize(r->stream);
        if (w != hipSuccess) return hip_fail(w, "hipStreamSynchronize");
        if (r->b.sws) (void)hipFree(r->b.sws);
        r->b.sws = nullptr;
        r->scratch_cap = r->scratch_limit = 0;
        plan = BatchPlan{};
        s = prepare_launch(r, items, count, plan);
    }
    if (s != VOX_OK) return s;
    hipError_t e;
    // stage through a pinned slot whose previous copy has completed
    const int k = r->slot;
    r->slot ^= 1;
    e = hipEventSynchronize(r->ev[k]);
    if (e != hipSuccess) return hip_fail(e, "hipEventSynchronize");
    if (plan.host.size() > r->pinned_cap[k]) {
        if (r->pinned[k]) (void)hipHostFree(r->pinned[k]);
        r->pinned_cap[k] = plan.host.size() * 2;
        e = hipHostMalloc(&r->pinned[k], r->pinned_cap[k], hipHostMallocDefault);
        if (e != hipSuccess) {
            r->pinned[k] = nullptr;
            r->pinned_cap[k] = 0;
            return fail(VOX_ERR_OOM, std::string("runner pinned staging: ") + hipGetErrorString(e));
        }
    }
    std::memcpy(r->pinned[k], plan.host.data(), plan.host.size());
    e = hipMemcpyAsync(r->dev_desc, r->pinned[k], plan.host.size(), hipMemcpyHostToDevice, r->stream);
    if (e == hipSuccess) e = hipEventRecord(r->ev[k], r->stream);
    if (e != hipSuccess) return hip_fail(e, "runner descriptor upload");
    bind_maps(&r->b, r->dev_desc);
    if (plan.scratch) r->b.scratch_dirty = true;
    e = launch_all(&r->b, r->stream);
    if (e != hipSuccess) return hip_fail(e, "runner launch");
    if (plan.scratch) r->b.scratch_dirty = false;
    r->launches++;
    return VOX_OK;
}

vox_status vox_runner_destroy(vox_runner* r) {
    if (!r) return VOX_OK;
    if (r->stream || r->b.ws || r->b.mws || r->b.sws || r->dev_desc) (void)hipStreamSynchronize(r->stream);
    for (int i = 0; i < 2; i++) {
        if (r->ev[i]) (void)hipEventDestroy(r->ev[i]);
        if (r->pinned[i]) (void)hipHostFree(r->pinned[i]);
    }
    if (r->dev_desc) (void)hipFree(r->dev_desc);
    if (r->b.ws) (void)hipFree(r->b.ws);
    if (r->b.mws) (void)hipFree(r->b.mws);
    if (r->b.sws) (void)hipFree(r->b.sws);
    r->b.ws = nullptr;
    r->b.mws = nullptr;
    r->b.sws = nullptr;
    delete r;
    return VOX_OK;
}

}  // extern "C"
