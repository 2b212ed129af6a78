// transfer.hpp -- large copies between device memory and a caller's pageable
// host memory.
//
// The runtime's own copy of pageable memory runs on one host thread: 28 GB/s
// to the device, 17 GB/s back, and 10 GB/s back into memory that is touched
// for the first time (a fresh result array), where that thread also takes
// every page fault.  Here LANES host threads each own a pinned chunk and take
// every LANES-th chunk of the copy: while one lane's chunk is on the bus the
// others move theirs between pinned and pageable memory and fault its pages
// in.  Measured: the 703 MB state of 256^3 hydro, download into fresh memory
// 67.7 -> 16.1 ms, upload 25.1 -> 14.8 ms; 92 MB 9.1 -> 2.3 and 3.4 -> 2.2 ms;
// 12.6 MB 0.85 -> 0.46 ms.  Chunks of 1 and 4 MiB and a stream per lane are no
// faster; one stream for all takes 18 % longer, and each stream costs a
// millisecond or two to make.  Downloads below THRESHOLD stay with the runtime
// (5.6 MB takes 0.36 ms there, about what the threads would), and uploads
// below UP_THRESHOLD: 12.3 MB takes 0.38 ms there, 0.45 ms by the threads, and
// a block that is only uploaded to should not pay for the set.
//
// Pinned chunks and streams are kept for the next copy while any block
// exists: at most KEEP sets (32 MiB) idle, all given back with the last block.
// A copy in progress owns its set, so copies of several threads run side by
// side.
#pragma once

#include <hip/hip_runtime.h>

#include <cstring>
#include <mutex>
#include <new>
#include <system_error>
#include <thread>
#include <vector>

namespace mara {
namespace host {

constexpr int LANES = 8;
constexpr int STREAMS = 2;  // shared by the lanes
constexpr size_t CHUNK = 2u << 20;
constexpr size_t THRESHOLD = 8u << 20;
constexpr size_t UP_THRESHOLD = 32u << 20;
constexpr size_t KEEP = 2;

struct LaneSet
{
    int device = -1;
    char* pinned = nullptr;  // LANES chunks
    hipStream_t stream[STREAMS] = {};
    hipEvent_t done[LANES] = {};
};

class LanePool
{
public:
    // one more, or one less, block that may copy
    void add_user()
    {
        std::lock_guard<std::mutex> lock(mutex_);
        ++users_;
    }
    void drop_user()
    {
        std::vector<LaneSet*> rest;
        {
            std::lock_guard<std::mutex> lock(mutex_);
            if (--users_ == 0) rest.swap(idle_);
        }
        for (LaneSet* s : rest) destroy(s);
    }
    // a set on the device, or null
    LaneSet* take(int device)
    {
        {
            std::lock_guard<std::mutex> lock(mutex_);
            for (size_t k = 0; k < idle_.size(); ++k)
                if (idle_[k]->device == device)
                {
                    LaneSet* s = idle_[k];
                    idle_.erase(idle_.begin() + k);
                    return s;
                }
        }
        LaneSet* s = new (std::nothrow) LaneSet();
        if (!s) return nullptr;
        s->device = device;
        bool made = hipHostMalloc((void**)&s->pinned, LANES * CHUNK, hipHostMallocDefault) == hipSuccess;
        for (int l = 0; made && l < STREAMS; ++l)
            made = hipStreamCreateWithFlags(&s->stream[l], hipStreamNonBlocking) == hipSuccess;
        for (int l = 0; made && l < LANES; ++l)
            made = hipEventCreateWithFlags(&s->done[l], hipEventDisableTiming) == hipSuccess;
        if (made) return s;
        (void)hipGetLastError();
        destroy(s);
        return nullptr;
    }
    void give(LaneSet* s)
    {
        {
            std::lock_guard<std::mutex> lock(mutex_);
            if (users_ > 0 && idle_.size() < KEEP)
            {
                idle_.push_back(s);  // capacity reserved below: does not throw
                return;
            }
        }
        destroy(s);
    }
    LanePool() { idle_.reserve(KEEP); }

private:
    static void destroy(LaneSet* s)
    {
        for (int l = 0; l < LANES; ++l)
            if (s->done[l]) (void)hipEventDestroy(s->done[l]);
        for (int l = 0; l < STREAMS; ++l)
            if (s->stream[l]) (void)hipStreamDestroy(s->stream[l]);
        if (s->pinned) (void)hipHostFree(s->pinned);
        delete s;
    }
    std::mutex mutex_;
    std::vector<LaneSet*> idle_;
    int users_ = 0;
};

// never destroyed: the runtime may be gone by then
inline LanePool& lane_pool()
{
    static LanePool* pool = new LanePool();
    return *pool;
}

// Copies `bytes` between device and host memory on the current device, whose
// work on `dev` the caller has waited for; complete on return.
inline hipError_t copy_large(char* dev, char* hst, size_t bytes, bool to_device)
{
    const hipMemcpyKind kind = to_device ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost;
    int device = 0;
    LaneSet* set = nullptr;
    if (bytes >= THRESHOLD && hipGetDevice(&device) == hipSuccess) set = lane_pool().take(device);
    if (!set) return hipMemcpy(to_device ? dev : hst, to_device ? hst : dev, bytes, kind);
    hipError_t status[LANES] = {};
    const auto lane = [&](int l) {
        hipError_t e = hipSetDevice(device);
        char* const pinned = set->pinned + l * CHUNK;
        const hipStream_t stream = set->stream[l % STREAMS];
        for (size_t off = l * CHUNK; e == hipSuccess && off < bytes; off += LANES * CHUNK)
        {
            const size_t len = bytes - off < CHUNK ? bytes - off : CHUNK;
            if (to_device)
            {
                std::memcpy(pinned, hst + off, len);
                e = hipMemcpyAsync(dev + off, pinned, len, kind, stream);
            }
            else
                e = hipMemcpyAsync(pinned, dev + off, len, kind, stream);
            if (e == hipSuccess) e = hipEventRecord(set->done[l], stream);
            if (e == hipSuccess) e = hipEventSynchronize(set->done[l]);
            if (e == hipSuccess && !to_device) std::memcpy(hst + off, pinned, len);
        }
        status[l] = e;
    };
    std::thread threads[LANES];
    int started = 1;
    try
    {
        for (; started < LANES; ++started) threads[started] = std::thread(lane, started);
    }
    catch (const std::system_error&)
    {
    }
    lane(0);
    for (int l = 1; l < started; ++l) threads[l].join();
    for (int l = started; l < LANES; ++l) lane(l);  // threads the system did not give
    lane_pool().give(set);
    for (hipError_t e : status)
        if (e != hipSuccess) return e;
    return hipSuccess;
}

} // namespace host
} // namespace mara
