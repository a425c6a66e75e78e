// matmul_ws.h -- lkhip_matmul's workspaces (X planes, split-K partials), kept
// per stream: calls on one stream run in order, so they share one buffer, and a
// call holds the lock until its launches are enqueued, so another thread's cannot
// come between.  hipMallocAsync + hipFreeAsync cost 13 us per call, more than a
// small product takes.  Kept only for streams whose end is seen: the null stream
// and those of lkhip_stream_create; other streams (and a stream that is being
// captured, whose graph may replay beside later calls) allocate in stream order.
// At most kMost buffers of kBytes each; all are freed with the last weight handle.
// Host code only.
#pragma once
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <mutex>
#include <new>
#include <vector>

namespace lkws {

constexpr size_t kBytes = (size_t)256 << 20, kMost = 16;

struct Kept {
    int device;
    hipStream_t stream;
    void* p;
    size_t bytes;
};

struct Pool {
    Pool() { kept.reserve(kMost); }  // nothing below throws through the C entry points
    std::mutex mu;
    std::vector<Kept> kept;
    std::vector<std::pair<int, hipStream_t>> streams;  // made by lkhip_stream_create, by device
    size_t weights = 0;                                // live weight handles
};

// hipMallocAsync that leaves no error behind for a later hipGetLastError (the launch checks) to return
inline void* alloc(size_t bytes, hipStream_t st) {
    void* p = nullptr;
    if (hipMallocAsync(&p, bytes, st) == hipSuccess) return p;
    (void)hipGetLastError();
    return nullptr;
}

// The kept buffer of (current device, st) with room for `bytes`, or null; pool.mu is held.
// It asks for more than the call needs so that it grows seldom, and, where that much is
// not to be had, for the call's own size, the old buffer given back first.
inline void* room(Pool& pool, hipStream_t st, size_t bytes) {
    int dev = 0;
    if (bytes > kBytes || hipGetDevice(&dev) != hipSuccess) return nullptr;
    if (st) {
        if (std::find(pool.streams.begin(), pool.streams.end(), std::make_pair(dev, st)) == pool.streams.end())
            return nullptr;
        hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(st, &cs) != hipSuccess || cs != hipStreamCaptureStatusNone) return nullptr;
    }
    for (size_t i = 0; i < pool.kept.size(); i++) {
        Kept& w = pool.kept[i];
        if (w.device != dev || w.stream != st) continue;
        if (w.bytes >= bytes) return w.p;
        size_t want = std::max(bytes, std::min(kBytes, 2 * w.bytes));
        void* p = alloc(want, st);
        (void)hipFreeAsync(w.p, st);  // after the calls that use it
        if (!p) p = alloc(want = bytes, st);
        if (!p) {
            pool.kept.erase(pool.kept.begin() + i);
            return nullptr;
        }
        w.p = p;
        w.bytes = want;
        return p;
    }
    if (pool.kept.size() >= kMost) return nullptr;
    size_t want = std::max<size_t>(bytes, (size_t)4 << 20);
    void* p = alloc(want, st);
    if (!p) p = alloc(want = bytes, st);
    if (p) pool.kept.push_back({dev, st, p, want});
    return p;
}

// Frees the buffers of one stream (device, st), or of all; pool.mu is held.
inline void drop(Pool& pool, bool all, int device, hipStream_t st) {
    for (size_t i = 0; i < pool.kept.size();)
        if (all || (pool.kept[i].device == device && pool.kept[i].stream == st)) {
            (void)hipFree(pool.kept[i].p);  // waits for the device
            pool.kept[i] = pool.kept.back();
            pool.kept.pop_back();
        } else {
            i++;
        }
}

inline void weight_created(Pool& pool) {
    std::lock_guard<std::mutex> lk(pool.mu);
    pool.weights++;
}
inline void weight_destroyed(Pool& pool) {
    std::lock_guard<std::mutex> lk(pool.mu);
    if (--pool.weights == 0) drop(pool, true, 0, nullptr);
}
inline void stream_created(Pool& pool, hipStream_t st) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return;
    std::lock_guard<std::mutex> lk(pool.mu);
    try {
        pool.streams.emplace_back(dev, st);
    } catch (const std::bad_alloc&) {  // as a stream that was made elsewhere
    }
}
inline void stream_destroyed(Pool& pool, hipStream_t st) {
    std::lock_guard<std::mutex> lk(pool.mu);
    for (size_t i = 0; i < pool.streams.size();)
        if (pool.streams[i].second == st) {
            drop(pool, false, pool.streams[i].first, st);
            pool.streams.erase(pool.streams.begin() + i);
        } else {
            i++;
        }
}

// One call's workspace: the stream's kept buffer, locked, or an allocation in stream order.
class Scratch {
public:
    Scratch(Pool& pool, hipStream_t st) : pool_(pool), st_(st) {}
    // `bytes` of device memory until this object ends, or null where there are none.
    void* get(size_t bytes) {
        lk_ = std::unique_lock<std::mutex>(pool_.mu);
        if (void* p = room(pool_, st_, bytes)) return p;
        lk_.unlock();
        return own_ = alloc(bytes, st_);
    }
    ~Scratch() {
        if (own_) (void)hipFreeAsync(own_, st_);
    }
    Scratch(const Scratch&) = delete;
    Scratch& operator=(const Scratch&) = delete;

private:
    Pool& pool_;
    hipStream_t st_;
    std::unique_lock<std::mutex> lk_;
    void* own_ = nullptr;
};

}  // namespace lkws
