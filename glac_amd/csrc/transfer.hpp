// transfer.hpp -- host arrays to and from the device through pinned slices.
//
// A copy from or to ordinary host memory runs at 30 and 17 GB/s through the
// runtime's own staging, and into pages not yet touched at 10.  Here a few host
// threads copy between the array and pinned slices while the slices before
// them travel at 46 GB/s of the link's 57, and the page faults of a fresh
// array are taken by all of them: 382 MB (24^3 x 48) up 12.7 -> 8.5 ms, down into
// a fresh array 36 -> 9.3 ms.  Four threads of two 4 MiB slices each: with 2 and
// 1 MiB slices the per-copy cost shows (41 and 32 GB/s), with two threads the
// page faults do (15 ms down), eight gain nothing.  The line lies at 16 MiB:
// 24 MB still go faster (up 0.71 -> 0.68 ms, down 1.35 -> 0.73), 4.7 MB go up no
// faster (0.21 and 0.23 ms) and would not earn back the pinned memory's
// allocation (0.75 ms, once per context).  Arrays that the runtime knows (pinned
// or managed ones) it copies by itself at the link's rate.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstddef>
#include <cstring>
#include <thread>

namespace glacx {

// A stretch of host memory and the device memory it is copied to or from.
struct HostSpan {
    char *host;
    char *dev;
    size_t bytes;
};

class Transfer {
public:
    static constexpr size_t kSlice = (size_t)4 << 20, kLeast = (size_t)16 << 20;
    static constexpr int kThreads = 4, kMostSpans = 4;

    Transfer() = default;
    Transfer(const Transfer &) = delete;
    Transfer &operator=(const Transfer &) = delete;
    ~Transfer() { release(); }

    // Copies `n` spans (kMostSpans at most) on `stream`, to the device (`up`) or to
    // the host, behind the work already there.  A copy to the host is complete on
    // return; one to the device may be used by what is launched on the stream
    // afterwards.  Allocates no host memory that could fail: the C entries above it
    // have nothing to catch an exception with.
    hipError_t run(const HostSpan *spans, int n, bool up, int device, hipStream_t stream) noexcept
    {
        size_t total = 0;
        for (int k = 0; k < n; k++) total += spans[k].bytes;
        Slices sliced;
        if (total >= kLeast)
            for (int k = 0; k < n; k++)
                if (ordinary(spans[k].host)) sliced.add(spans[k]);
        if (sliced.bytes < kLeast || !acquire()) sliced = Slices();
        for (int k = 0; k < n; k++) {
            const HostSpan &s = spans[k];
            if (sliced.holds(s)) continue;
            const hipError_t e = up ? hipMemcpyAsync(s.dev, s.host, s.bytes, hipMemcpyHostToDevice, stream)
                                    : hipMemcpyAsync(s.host, s.dev, s.bytes, hipMemcpyDeviceToHost, stream);
            if (e != hipSuccess) return e;
        }
        if (sliced.n == 0) return up ? hipSuccess : hipStreamSynchronize(stream);
        std::atomic<size_t> next{0};
        std::atomic<int> status{hipSuccess};
        auto work = [&](int w) {
            int e = hipSetDevice(device);
            if (e == hipSuccess)
                e = up ? send(sliced, next, status, w, stream) : receive(sliced, next, status, w, stream);
            if (e != hipSuccess) status = e;
        };
        std::thread helpers[kThreads - 1];
        int started = 0;
        try {
            for (; started < kThreads - 1; started++) helpers[started] = std::thread(work, started + 1);
        } catch (...) {
            // fewer helpers than wanted: the slices are dealt out as threads ask for them
        }
        work(0);
        for (int k = 0; k < started; k++) helpers[k].join();
        // the slices are free again when the stream has passed the copies
        const hipError_t e = hipStreamSynchronize(stream);
        return status != hipSuccess ? (hipError_t)status.load() : e;
    }

private:
    // Spans cut into slices, each span from its start.
    struct Slices {
        HostSpan span[kMostSpans];
        int n = 0;
        size_t bytes = 0, count = 0;

        static size_t of(const HostSpan &s) { return (s.bytes + kSlice - 1) / kSlice; }
        void add(const HostSpan &s)
        {
            span[n++] = s;
            bytes += s.bytes;
            count += of(s);
        }
        bool holds(const HostSpan &s) const
        {
            for (int k = 0; k < n; k++)
                if (span[k].dev == s.dev) return true;
            return false;
        }
        size_t size() const { return count; }
        HostSpan operator[](size_t i) const
        {
            int k = 0;
            for (; i >= of(span[k]); k++) i -= of(span[k]);
            const size_t o = i * kSlice;
            return {span[k].host + o, span[k].dev + o, std::min(kSlice, span[k].bytes - o)};
        }
    };

    // Memory that the runtime knows nothing of: from malloc, the stack, a mapped file.
    static bool ordinary(const void *p)
    {
        hipPointerAttribute_t a;
        if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type == hipMemoryTypeUnregistered;
        (void)hipGetLastError();
        return true;
    }

    char *slice(int w, int k) { return pinned_ + (size_t)(2 * w + k) * kSlice; }
    hipEvent_t event(int w, int k) { return events_[2 * w + k]; }

    int send(const Slices &slices, std::atomic<size_t> &next, std::atomic<int> &status, int w,
             hipStream_t stream)
    {
        bool busy[2] = {false, false};
        for (int k = 0;; k ^= 1) {
            const size_t i = next++;
            if (i >= slices.size() || status != hipSuccess) return hipSuccess;
            hipError_t e = busy[k] ? hipEventSynchronize(event(w, k)) : hipSuccess;
            if (e != hipSuccess) return e;
            const HostSpan s = slices[i];
            std::memcpy(slice(w, k), s.host, s.bytes);
            e = hipMemcpyAsync(s.dev, slice(w, k), s.bytes, hipMemcpyHostToDevice, stream);
            if (e != hipSuccess) return e;
            if ((e = hipEventRecord(event(w, k), stream)) != hipSuccess) return e;
            busy[k] = true;
        }
    }

    int receive(const Slices &slices, std::atomic<size_t> &next, std::atomic<int> &status, int w,
                hipStream_t stream)
    {
        size_t held[2];
        auto issue = [&](int k) -> hipError_t {
            const size_t i = held[k] = next++;
            if (i >= slices.size()) return hipSuccess;
            const HostSpan s = slices[i];
            const hipError_t e = hipMemcpyAsync(slice(w, k), s.dev, s.bytes, hipMemcpyDeviceToHost, stream);
            return e != hipSuccess ? e : hipEventRecord(event(w, k), stream);
        };
        hipError_t e = issue(0);
        if (e == hipSuccess) e = issue(1);
        for (int k = 0; e == hipSuccess && held[k] < slices.size() && status == hipSuccess; k ^= 1) {
            const HostSpan s = slices[held[k]];
            if ((e = hipEventSynchronize(event(w, k))) != hipSuccess) break;
            std::memcpy(s.host, slice(w, k), s.bytes);
            e = issue(k);
        }
        return e;
    }

    bool acquire()
    {
        if (pinned_) return true;
        if (hipHostMalloc((void **)&pinned_, 2 * kThreads * kSlice, hipHostMallocDefault) != hipSuccess) {
            pinned_ = nullptr;
            (void)hipGetLastError();
            return false;
        }
        for (int k = 0; k < 2 * kThreads; k++)
            if (hipEventCreateWithFlags(&events_[k], hipEventDisableTiming) != hipSuccess) {
                events_[k] = nullptr;
                (void)hipGetLastError();
                release();
                return false;
            }
        return true;
    }

    void release()
    {
        for (hipEvent_t &v : events_) {
            if (v) (void)hipEventDestroy(v);
            v = nullptr;
        }
        if (pinned_) (void)hipHostFree(pinned_);
        pinned_ = nullptr;
    }

    char *pinned_ = nullptr;
    hipEvent_t events_[2 * kThreads] = {};
};

} // namespace glacx
