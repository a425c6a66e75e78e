// matmul_ws.h -- lkhip_matmul's workspaces (X planes, split-K partials), kept
// per stream: calls on one stream run in order, so they share one buffer, and a
// call holds that stream's lock until its launches are enqueued, so another
// thread's cannot come between; calls on other streams are not held up.
// hipMallocAsync + hipFreeAsync cost 13 us per call, more than a small product
// takes.  Kept only for streams whose end is seen: the null stream and those of
// lkhip_stream_create; other streams (and a stream that is being captured,
// whose graph may replay beside later calls) allocate in stream order.  At most
// kMost buffers of kBytes each (a call that needs more takes longer than its
// allocation); a stream's is freed, in its order, when it is destroyed, and all
// (but those of streams being captured) with the last weight handle.  Host code only.
#pragma once
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <memory>
#include <mutex>
#include <new>
#include <vector>

namespace lkws {

constexpr size_t kBytes = (size_t)64 << 20, kMost = 16;

struct Kept {
    int device = 0;
    hipStream_t stream = nullptr;
    std::mutex mu;  // the rest
    void* p = nullptr;
    size_t bytes = 0;
    bool ended = false;
};

struct Pool {
    Pool() { kept.reserve(kMost); }  // nothing below throws through the C entry points
    std::mutex mu;                   // never taken with a Kept's held
    std::vector<std::shared_ptr<Kept>> kept;
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

inline bool capturing(hipStream_t st) {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (!st) return false;
    if (hipStreamIsCapturing(st, &cs) == hipSuccess) return cs != hipStreamCaptureStatusNone;
    (void)hipGetLastError();
    return true;
}

// The entry of (current device, st), or null where none is kept.
inline std::shared_ptr<Kept> find(Pool& pool, hipStream_t st) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    std::lock_guard<std::mutex> lk(pool.mu);
    if (st && (std::find(pool.streams.begin(), pool.streams.end(), std::make_pair(dev, st)) == pool.streams.end() ||
               capturing(st)))
        return nullptr;
    for (const auto& k : pool.kept)
        if (k->device == dev && k->stream == st) return k;
    if (pool.kept.size() >= kMost) return nullptr;
    try {
        auto k = std::make_shared<Kept>();
        k->device = dev;
        k->stream = st;
        pool.kept.push_back(k);
        return k;
    } catch (const std::bad_alloc&) {
        return nullptr;
    }
}

// The entry's buffer with room for `bytes`, or null; its lock is held.  It asks for
// more than the call needs so that it grows seldom, and, where that much is not to
// be had, for the call's own size, the old buffer given back first.
inline void* room(Kept& k, size_t bytes) {
    if (k.ended || k.bytes >= bytes) return k.ended ? nullptr : k.p;
    size_t want = std::max(bytes, std::min(kBytes, std::max((size_t)4 << 20, 2 * k.bytes)));
    void* p = alloc(want, k.stream);
    if (k.p) (void)hipFreeAsync(k.p, k.stream);  // after the calls that use it
    if (!p) p = alloc(want = bytes, k.stream);
    k.p = p;
    k.bytes = p ? want : 0;
    return p;
}

// Gives the entry's buffer back after the calls on its stream that use it; other
// streams are not waited for, nor a capture on one of them disturbed.  On a stream that
// is being captured itself the free would become a node of its graph: false, and the
// entry stays, unless the stream is to be `gone`.
inline bool end(Kept& k, bool gone) {
    std::lock_guard<std::mutex> lk(k.mu);
    const bool cap = capturing(k.stream);
    if (cap && !gone) return false;
    k.ended = true;
    if (!k.p) return true;
    int dev = 0;
    const bool other = hipGetDevice(&dev) == hipSuccess && dev != k.device;
    if (other) (void)hipSetDevice(k.device);
    if (cap) (void)hipFree(k.p);
    else (void)hipFreeAsync(k.p, k.stream);
    if (other) (void)hipSetDevice(dev);
    k.p = nullptr;
    k.bytes = 0;
    return true;
}

inline void weight_created(Pool& pool) {
    std::lock_guard<std::mutex> lk(pool.mu);
    pool.weights++;
}
inline void weight_destroyed(Pool& pool) {
    std::lock_guard<std::mutex> lk(pool.mu);
    if (--pool.weights) return;
    auto& k = pool.kept;  // keeps its capacity
    k.erase(std::remove_if(k.begin(), k.end(), [](auto& e) { return end(*e, false); }), k.end());
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
// Before the stream is destroyed.
inline void stream_destroyed(Pool& pool, hipStream_t st) {
    std::shared_ptr<Kept> gone;
    {
        std::lock_guard<std::mutex> lk(pool.mu);
        const auto s = std::find_if(pool.streams.begin(), pool.streams.end(), [&](auto& v) { return v.second == st; });
        if (s == pool.streams.end()) return;
        pool.streams.erase(s);
        for (size_t i = 0; i < pool.kept.size(); i++)
            if (pool.kept[i]->stream == st) {
                gone = std::move(pool.kept[i]);
                pool.kept.erase(pool.kept.begin() + i);
                break;
            }
    }
    if (gone) end(*gone, true);
}

// One call's workspace: the stream's kept buffer, locked, or an allocation in stream order.
class Scratch {
public:
    Scratch(Pool& pool, hipStream_t st) : pool_(pool), st_(st) {}
    // whether the stream has a kept buffer
    bool keeps() {
        if (!kept_) kept_ = find(pool_, st_);
        return kept_ != nullptr;
    }
    // `bytes` of device memory until this object ends, or null where there are none.
    void* get(size_t bytes) {
        if (bytes <= kBytes && keeps()) {
            lk_ = std::unique_lock<std::mutex>(kept_->mu);
            if (void* p = room(*kept_, bytes)) return p;
            lk_.unlock();
        }
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
    std::shared_ptr<Kept> kept_;
    std::unique_lock<std::mutex> lk_;  // released before kept_ goes
    void* own_ = nullptr;
};

}  // namespace lkws
