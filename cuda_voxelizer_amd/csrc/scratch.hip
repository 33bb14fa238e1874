// scratch.hip -- the scratch memory that calls on one stream share (scratch.h).
#include "scratch.h"

#include <atomic>
#include <map>
#include <mutex>

#include "vox_kernels.h"

namespace voxamd {

struct StreamScratch {
    void* table = nullptr;  // grow-only
    uint64_t bytes = 0;
    bool dirty = true;
    void* spills = nullptr;
    std::mutex use;
};

hipError_t stream_key(hipStream_t stream, StreamKey& key) {
    static std::atomic<uint64_t> threads{0};
    static thread_local const uint64_t thread = ++threads;
    key.stream = stream;
    key.thread = stream == hipStreamPerThread ? thread : 0;
    return hipGetDevice(&key.device);
}

static std::mutex g_scratch_mutex;
static std::map<StreamKey, StreamScratch> g_scratch;

ScratchLease::ScratchLease(hipStream_t stream) : stream_(stream) {
    StreamKey key;
    if (stream_key(stream, key) != hipSuccess) {
        (void)hipGetLastError();
        return;
    }
    {
        std::lock_guard<std::mutex> lock(g_scratch_mutex);
        s_ = &g_scratch[key];
    }
    s_->use.lock();
}

ScratchLease::~ScratchLease() {
    if (s_) s_->use.unlock();
}

uint32_t* ScratchLease::table(uint64_t bytes) {
    if (!s_) return nullptr;
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    hipError_t e = hipStreamIsCapturing(stream_, &cap);
    if (e == hipSuccess && cap != hipStreamCaptureStatusNone) return nullptr;
    if (e == hipSuccess && s_->bytes < bytes) {
        if (s_->table) {
            e = hipStreamSynchronize(stream_);  // a previous call on this stream may still use it
            if (e == hipSuccess) e = hipFree(s_->table);
            if (e == hipSuccess) {
                s_->table = nullptr;
                s_->bytes = 0;
            }
        }
        if (e == hipSuccess) e = hipMalloc(&s_->table, bytes);
        if (e == hipSuccess) {
            s_->bytes = bytes;
            s_->dirty = true;
        } else if (!s_->bytes) {
            s_->table = nullptr;
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
    if (!s_->spills) {
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
