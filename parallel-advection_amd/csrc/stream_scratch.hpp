// Device buffers that the runs of one plan write: one per stream, so that a
// plan's runs may overlap on several streams (and host threads) as if it kept
// nothing.
#pragma once

#include <mutex>
#include <thread>
#include <vector>

#include "common.hpp"

namespace bkma {

class StreamScratch {
public:
    // Streams, and captures, that may have a buffer of their own.  A buffer
    // stays with its stream until the plan goes; further streams get none, or take
    // over the one that was used longest ago.
    static constexpr size_t kStreams = 8, kCaptures = 8;

    StreamScratch() = default;
    StreamScratch(const StreamScratch &) = delete;
    StreamScratch &operator=(const StreamScratch &) = delete;
    ~StreamScratch() {
        for (const Buffer &b : buffers_) (void)hipFree(b.data);
    }

    // Buffers of `bytes` each.  The first one, for the first stream or capture
    // that asks, has `first` bytes and is allocated here, and so are `more` others
    // as far as there is memory; false: none for the first.
    bool create(u64 bytes, u64 first, int more) {
        bytes_ = bytes;
        Buffer b;
        if (!allocate(&b.data, first)) return false;
        buffers_.push_back(b);
        for (; more > 0 && allocate(&b.data, bytes); --more) buffers_.push_back(b);
        return true;
    }
    bool first(const void *data) const { return !buffers_.empty() && buffers_[0].data == data; }

    // Held from get() until the run is enqueued: a buffer may change hands.
    std::unique_lock<std::mutex> lock() { return std::unique_lock<std::mutex>(mutex_); }

    // The buffer of a run on stream s, or null.  A stream under capture takes a
    // buffer per capture, since its graph may run beside others later.  Where
    // none is left: without `grow` the answer is null; with it another is
    // allocated, and where there is no memory or there are too many streams, a run
    // outside a capture waits for the device and takes over a buffer (a capture
    // takes over that of an older one).
    void *get(hipStream_t s, bool grow) {
        Key k;
        k.stream = s;
        if (s == hipStreamPerThread) k.thread = std::this_thread::get_id();
        hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
        unsigned long long id = 0;
        if (hipStreamGetCaptureInfo(s, &st, &id) != hipSuccess) (void)hipGetLastError();  // the default stream beside a capture
        if (st == hipStreamCaptureStatusActive) {
            k.capture = id;
            k.captured = true;
        }
        size_t alike = 0;
        Buffer *oldest = nullptr;
        for (Buffer &b : buffers_) {
            if (b.taken && b.key == k) return use(b);
            if (!b.taken) {
                b.taken = true;
                b.key = k;
                return use(b);
            }
            if (b.key.captured != k.captured) continue;
            ++alike;
            if (!oldest || b.used < oldest->used) oldest = &b;
        }
        if (!grow) return nullptr;
        if (alike < (k.captured ? kCaptures : kStreams)) {
            Buffer b;
            if (allocate(&b.data, bytes_)) {
                b.taken = true;
                b.key = k;
                buffers_.push_back(b);
                return use(buffers_.back());
            }
        }
        if (!oldest) return nullptr;
        if (!k.captured && hipDeviceSynchronize() != hipSuccess) {
            (void)hipGetLastError();
            return nullptr;
        }
        oldest->key = k;
        return use(*oldest);
    }

private:
    struct Key {
        hipStream_t stream = nullptr;
        std::thread::id thread;          // of the per-thread default stream
        unsigned long long capture = 0;  // under capture: which
        bool captured = false;
        bool operator==(const Key &o) const {
            return stream == o.stream && thread == o.thread && capture == o.capture && captured == o.captured;
        }
    };
    struct Buffer {
        void *data = nullptr;
        bool taken = false;
        Key key;
        u64 used = 0;
    };

    void *use(Buffer &b) {
        b.used = ++clock_;
        return b.data;
    }
    // Also while this or another thread captures: an allocation is no part of it.
    static bool allocate(void **p, u64 bytes) {
        hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
        const bool swapped = hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess;
        const bool ok = hipMalloc(p, bytes ? bytes : 16) == hipSuccess;
        if (!ok) {
            (void)hipGetLastError();
            *p = nullptr;
        }
        if (swapped) (void)hipThreadExchangeStreamCaptureMode(&mode);
        return ok;
    }

    std::mutex mutex_;
    std::vector<Buffer> buffers_;
    u64 bytes_ = 0, clock_ = 0;
};

}  // namespace bkma
