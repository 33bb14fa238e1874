// scratch.h -- the scratch memory that calls on one stream share.
//
// Per device and stream: a table for blocked surface words, blocked or linear
// solid markers, all zero between calls, and the counters and records of spilled
// runs (marker.hip), whose counters are zero between calls.  Both are worked on by
// several launches of a call in a row, so a call holds the stream's scratch from
// before its first launch until its last is queued; a second thread's call on the
// stream waits for that, and the stream's order does the rest.  (A new stream may
// have the handle of one that was destroyed; hipStreamDestroy waits for a stream's
// work.)  Calls on the stream's other workspaces (tile, slab, region, triangle
// order) hold it too.  A call that is recorded into a graph uses none of it but
// memory of the graph's (graph_memory), the region algorithm's records apart.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <tuple>

namespace voxamd {

// What a stream's workspaces are kept under.  hipStreamPerThread is one handle for
// a stream of each thread, so there the thread is part of the key (0 otherwise; a
// thread's number is never given to another).
struct StreamKey {
    int device = 0;
    hipStream_t stream = nullptr;
    uint64_t thread = 0;
    bool operator<(const StreamKey& o) const {
        return std::tie(device, stream, thread) < std::tie(o.device, o.stream, o.thread);
    }
    bool operator==(const StreamKey& o) const { return !(*this < o) && !(o < *this); }
};
hipError_t stream_key(hipStream_t stream, StreamKey& key);  // on the current device

// Memory is allocated and freed in the relaxed capture mode: no stream that is being
// captured is touched, and the default mode refuses it while any thread captures one.
struct RelaxedCapture {
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    const bool set;
    RelaxedCapture() : set(hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess) {}
    ~RelaxedCapture() {
        if (set) (void)hipThreadExchangeStreamCaptureMode(&mode);
    }
};

// Waits for all work of the device that has been queued, as hipFree does; unlike
// hipDeviceSynchronize it leaves other threads' captures valid.  It needs 256 bytes.
hipError_t wait_for_device();

// Device memory for the graph into which calls on `stream` are being recorded, its
// own until it and all that was cloned or instantiated from it are gone.  The contents
// are undefined.  An error where the device's limit does not allow it.
hipError_t graph_memory(hipStream_t stream, uint64_t bytes, void** out);

struct StreamScratch;

class ScratchLease {
   public:
    explicit ScratchLease(hipStream_t stream);
    ~ScratchLease();
    ScratchLease(const ScratchLease&) = delete;
    ScratchLease& operator=(const ScratchLease&) = delete;

    // Calls on the stream are being recorded into a graph (or, for the null stream,
    // another stream's capture keeps it from being used).
    bool recording() const { return recording_; }
    // A zero table of at least `bytes` bytes; null while the stream is being
    // captured (a later call may replace the table that the graph would hold),
    // without memory, and where the device's tables would grow beyond their limit.
    uint32_t* table(uint64_t bytes);
    // All launches are queued that leave the table zero.  Without it the next
    // holder zero-fills it.
    void clean();
    // marker_ws_bytes() bytes: counters and records of spilled runs.
    hipError_t spills(void** out);

   private:
    hipStream_t stream_;
    int device_ = 0;
    bool recording_ = true;
    StreamScratch* s_ = nullptr;
};

}  // namespace voxamd
