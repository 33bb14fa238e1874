// scratch.hip -- the scratch memory that calls on one stream share (scratch.h).
#include "scratch.h"

#include <algorithm>
#include <atomic>
#include <map>
#include <mutex>
#include <utility>
#include <vector>

#include "vox_host.h"
#include "vox_kernels.h"

namespace voxamd {

struct DeviceScratch {
    uint64_t held = 0, leases = 0;  // bytes in tables, leases so far
    uint64_t graphs = 0;            // bytes that graphs have, or had
};

struct StreamScratch {
    DeviceScratch* dev = nullptr;
    void* table = nullptr;  // grow-only
    uint64_t bytes = 0;
    bool dirty = true;
    void* spills = nullptr;
    bool recorded = false;  // a graph holds the spills: they are never freed
    int holders = 0;    // leases that hold or await it
    uint64_t last = 0;  // the device's count of leases at its last one
    std::mutex use;
};

struct GraphMemory {
    void* ptr;
    uint64_t bytes;
    int device;
};

// All streams' scratch.  A device's tables together stay below an eighth of its
// memory (36 GB here: 36 streams at 2048^3), or are one stream's table: a call that
// would go beyond has none, unless a stream of the device that has not had a call
// for kIdle of the device's leases can give up its table -- a stream that was
// destroyed, above all.  What a thread's own stream had (hipStreamPerThread) goes
// once the thread has ended and another table grows.  What a graph had is kept for
// the next one, and freed by vox_release_scratch only: an executable that was updated
// from a graph does not hold what that graph had.  All graphs of a device have an
// eighth of its memory at most.
constexpr uint64_t kIdle = 64;
struct ScratchPool {
    std::mutex m;
    std::map<StreamKey, StreamScratch> streams;
    std::map<int, DeviceScratch> devices;
    std::vector<uint64_t> ended;           // threads
    std::mutex mr;                       // of returned; never held around a call of the runtime
    std::vector<GraphMemory*> returned;  // of graphs that are gone
};
static ScratchPool& pool() {
    static ScratchPool* p = new ScratchPool;  // threads may end after static objects have gone
    return *p;
}

struct ThreadNumber {
    uint64_t n;
    ThreadNumber() {
        static std::atomic<uint64_t> threads{0};
        n = ++threads;
    }
    ~ThreadNumber() {
        ScratchPool& P = pool();
        std::lock_guard<std::mutex> lock(P.m);
        P.ended.push_back(n);
    }
};

hipError_t stream_key(hipStream_t stream, StreamKey& key) {
    key.stream = stream;
    key.thread = 0;
    if (stream == hipStreamPerThread) {
        static thread_local ThreadNumber thread;
        key.thread = thread.n;
    }
    return hipGetDevice(&key.device);
}

hipError_t wait_for_device() {
    const RelaxedCapture relaxed;
    void* p = nullptr;
    const hipError_t e = hipMalloc(&p, 256);
    return e == hipSuccess ? hipFree(p) : e;
}

// Frees what an idle stream of the current device has; its last call may still run,
// and hipFree waits for the device.
static void give_back(StreamScratch& s) {
    if (s.table) (void)hipFree(s.table);
    s.dev->held -= s.bytes;
    s.table = nullptr;
    s.bytes = 0;
    s.dirty = true;
    if (s.spills && !s.recorded) {
        (void)hipFree(s.spills);
        s.spills = nullptr;
    }
}

// The runtime lets a graph's memory go: on any thread, where it must not be called.
static void graph_gone(void* memory) {
    ScratchPool& P = pool();
    std::lock_guard<std::mutex> lock(P.mr);
    P.returned.push_back((GraphMemory*)memory);
}

// Memory of at least `bytes` bytes, not above twice that, whose graph is gone; null if there is none.
static GraphMemory* take_returned(int device, uint64_t bytes) {
    ScratchPool& P = pool();
    std::lock_guard<std::mutex> lock(P.mr);
    auto best = P.returned.end();
    for (auto it = P.returned.begin(); it != P.returned.end(); ++it)
        if ((*it)->device == device && (*it)->bytes >= bytes && (*it)->bytes / 2 <= bytes &&
            (best == P.returned.end() || (*it)->bytes < (*best)->bytes))
            best = it;
    if (best == P.returned.end()) return nullptr;
    GraphMemory* g = *best;
    P.returned.erase(best);
    return g;
}

static hipError_t new_graph_memory(int device, uint64_t bytes, GraphMemory** out) {
    size_t total = 0;
    hipError_t e = hipDeviceTotalMem(&total, device);
    if (e != hipSuccess) return e;
    ScratchPool& P = pool();
    {
        std::lock_guard<std::mutex> lock(P.m);
        uint64_t& held = P.devices[device].graphs;
        if (held + bytes > total / 8) return hipErrorOutOfMemory;
        held += bytes;
    }
    void* p = nullptr;
    e = hipMalloc(&p, bytes);
    if (e != hipSuccess) {
        std::lock_guard<std::mutex> lock(P.m);
        P.devices[device].graphs -= bytes;
        return e;
    }
    *out = new GraphMemory{p, bytes, device};
    return hipSuccess;
}

hipError_t graph_memory(hipStream_t stream, uint64_t bytes, void** out) {
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess) return e;
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    unsigned long long id = 0;
    hipGraph_t graph = nullptr;
    const hipGraphNode_t* deps = nullptr;
    size_t ndeps = 0;
    e = hipStreamGetCaptureInfo_v2(stream, &status, &id, &graph, &deps, &ndeps);
    if (e != hipSuccess) return e;
    if (status != hipStreamCaptureStatusActive || !graph) return hipErrorIllegalState;
    const RelaxedCapture relaxed;
    GraphMemory* g = take_returned(device, bytes);
    // a graph that is gone may still run
    e = g ? wait_for_device() : new_graph_memory(device, bytes, &g);
    hipUserObject_t owner = nullptr;
    if (e == hipSuccess) e = hipUserObjectCreate(&owner, g, graph_gone, 1, hipUserObjectNoDestructorSync);
    if (e != hipSuccess) {
        if (g) graph_gone(g);
        return e;
    }
    *out = g->ptr;
    e = hipGraphRetainUserObject(graph, owner, 1, hipGraphUserObjectMove);
    if (e != hipSuccess) (void)hipUserObjectRelease(owner, 1);
    return e;
}

// Counts `bytes` instead of s.bytes among the device's tables, if they fit.
static bool reserve(int device, StreamScratch& s, uint64_t bytes) {
    size_t total = 0;
    if (hipDeviceTotalMem(&total, device) != hipSuccess) return false;
    ScratchPool& P = pool();
    std::lock_guard<std::mutex> lock(P.m);
    for (size_t i = 0; i < P.ended.size(); i++) {
        const uint64_t n = P.ended[i];
        bool left = false;
        for (auto it = P.streams.begin(); it != P.streams.end();) {
            const bool own = it->first.thread == n;
            if (own && it->first.device == device && it->second.holders == 0) {
                give_back(it->second);
                if (!it->second.spills) {
                    it = P.streams.erase(it);
                    continue;
                }
            }
            left = left || own;
            ++it;
        }
        if (!left) P.ended.erase(P.ended.begin() + (long)i--);
    }
    const uint64_t limit = total / 8, now = s.dev->leases;
    while (s.dev->held - s.bytes + bytes > limit && s.dev->held > s.bytes) {
        auto idle = P.streams.end();
        for (auto it = P.streams.begin(); it != P.streams.end(); ++it)
            if (it->first.device == device && it->second.holders == 0 && it->second.table &&
                now - it->second.last >= kIdle &&
                (idle == P.streams.end() || it->second.last < idle->second.last))
                idle = it;
        if (idle == P.streams.end()) return false;
        give_back(idle->second);
        if (!idle->second.spills) P.streams.erase(idle);
    }
    s.dev->held += bytes - s.bytes;
    return true;
}

ScratchLease::ScratchLease(hipStream_t stream) : stream_(stream) {
    StreamKey key;
    if (stream_key(stream, key) != hipSuccess) {
        (void)hipGetLastError();
        return;
    }
    device_ = key.device;
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &cap) == hipSuccess)
        recording_ = cap != hipStreamCaptureStatusNone;
    else
        (void)hipGetLastError();
    ScratchPool& P = pool();
    {
        std::lock_guard<std::mutex> lock(P.m);
        s_ = &P.streams[key];
        if (!s_->dev) s_->dev = &P.devices[device_];
        s_->holders++;
        s_->last = ++s_->dev->leases;
    }
    s_->use.lock();
}

ScratchLease::~ScratchLease() {
    if (!s_) return;
    s_->use.unlock();
    std::lock_guard<std::mutex> lock(pool().m);
    s_->holders--;
}

uint32_t* ScratchLease::table(uint64_t bytes) {
    if (!s_ || recording_) return nullptr;
    hipError_t e = hipSuccess;
    if (s_->bytes < bytes) {
        const RelaxedCapture relaxed;
        if (!reserve(device_, *s_, bytes)) return nullptr;
        if (s_->table) {
            e = hipStreamSynchronize(stream_);  // a previous call on this stream may still use it
            if (e == hipSuccess) e = hipFree(s_->table);
            if (e == hipSuccess) {
                s_->table = nullptr;
                s_->bytes = 0;
            }
        }
        if (e == hipSuccess) {
            void* p = nullptr;
            e = hipMalloc(&p, bytes);
            if (e == hipSuccess) {
                s_->table = p;
                s_->bytes = bytes;
                s_->dirty = true;
            }
        }
        if (e != hipSuccess) {
            std::lock_guard<std::mutex> lock(pool().m);
            s_->dev->held -= bytes - s_->bytes;
        }
    }
    if (e == hipSuccess && s_->dirty) e = hipMemsetAsync(s_->table, 0, s_->bytes, stream_);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    s_->dirty = true;
    return (uint32_t*)s_->table;
}

void ScratchLease::clean() { s_->dirty = false; }

hipError_t ScratchLease::spills(void** out) {
    if (!s_) return hipErrorInvalidDevice;
    if (recording_) {
        if (!s_->spills) return hipErrorStreamCaptureUnsupported;  // the counters could not be cleared
        s_->recorded = true;
    }
    if (!s_->spills) {
        const RelaxedCapture relaxed;
        void* p = nullptr;
        hipError_t e = hipMalloc(&p, marker_ws_bytes());
        if (e != hipSuccess) return e;
        e = hipMemsetAsync(p, 0, 256, stream_);  // the counters start at zero
        if (e != hipSuccess) {
            (void)hipFree(p);
            return e;
        }
        s_->spills = p;
    }
    *out = s_->spills;
    return hipSuccess;
}

}  // namespace voxamd

using namespace voxamd;

extern "C" vox_status vox_release_scratch(void) {
    int device = 0;
    const hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess) return hip_fail(e, "hipGetDevice");
    const RelaxedCapture relaxed;
    ScratchPool& P = pool();
    std::vector<GraphMemory*> gone;
    {
        std::lock_guard<std::mutex> lock(P.mr);
        for (GraphMemory*& g : P.returned)
            if (g->device == device) gone.push_back(std::exchange(g, nullptr));
        P.returned.erase(std::remove(P.returned.begin(), P.returned.end(), nullptr), P.returned.end());
    }
    std::lock_guard<std::mutex> lock(P.m);
    for (GraphMemory* g : gone) {
        (void)hipFree(g->ptr);
        P.devices[device].graphs -= g->bytes;
        delete g;
    }
    for (auto it = P.streams.begin(); it != P.streams.end();) {
        if (it->first.device == device && it->second.holders == 0) {
            give_back(it->second);
            if (!it->second.spills) {
                it = P.streams.erase(it);
                continue;
            }
        }
        ++it;
    }
    return VOX_OK;
}
