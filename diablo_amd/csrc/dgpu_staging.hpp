// dgpu_staging.hpp -- host arrays of the caller in chunks through pinned memory.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <exception>
#include <mutex>
#include <system_error>
#include <thread>

namespace dgpu {

// The caller's arrays are pageable: one copy of a whole array runs at 14-22
// GB/s, and nothing else meanwhile.  Here up to kWorkers host threads take the
// array's chunks in turn, each with its own pinned slot, so the host copies and
// the DMA of different chunks overlap, and the host side can leave out what the
// device does not keep.  Copies on one stream follow each other at 21 GB/s, so
// the workers of a large array take turns on kStreams streams (53 GB/s; the
// same with a stream a worker).  A process's first streams cost 2.7 ms each to
// make, which a small array does not earn back in a few calls: below kSpread
// bytes all use the caller's.
// Slots and streams are made on first use, kept with the context and given back
// by release(); threads live for one call, and an array of one chunk starts
// none.  The members of an ensemble share one (a set of slots each is 16 MB of
// pinned memory a member, 1 GB for 64); calls that come together follow each
// other.
class Staging {
public:
    // planes of `bytes` each that make a chunk
    static int planes(size_t bytes) { return (int)std::max<size_t>(1, kChunk / bytes); }

    // Chunks 0..n-1: `in(chunk, slot, stream)` fills the slot and enqueues, and
    // when that work is done `out(chunk, slot)` reads the slot.  The work starts
    // after what `main` holds and is complete on return.  in and out run on
    // several threads at once and must not throw.
    template <typename In, typename Out>
    hipError_t run(hipStream_t main, int n, size_t bytes, In in, Out out)
    {
        std::lock_guard<std::mutex> one(call_);
        int workers = 0, streams = 1;
        if (hipError_t e = reserve(n, bytes, workers, streams)) return e;
        int dev = 0;
        if (hipError_t e = hipGetDevice(&dev)) return e;
        if (streams > 1) {
            if (hipError_t e = hipEventRecord(done_[0], main)) return e;
            for (int q = 1; q < streams; ++q)
                if (hipError_t e = hipStreamWaitEvent(stream_[q], done_[0], 0)) return e;
        }
        std::atomic<int> next{0}, err{hipSuccess};
        auto work = [&](int w) {
            hipError_t e = hipSuccess;
            const hipStream_t s = w % streams ? stream_[w % streams] : main;
            if (w) e = hipSetDevice(dev);
            for (int i; !e && err.load() == hipSuccess && (i = next.fetch_add(1)) < n;) {
                e = in(i, slot_[w], s);
                hipError_t f = hipEventRecord(done_[w], s);
                f = f ? hipStreamSynchronize(s) : hipEventSynchronize(done_[w]);
                if (!e) e = f;
                if (!e) out(i, slot_[w]);
            }
            if (e) err.store(e);
        };
        std::thread t[kWorkers];
        for (int w = 1; w < workers; ++w) {
            try {
                t[w] = std::thread(work, w);
            } catch (const std::exception &) {
                break;  // no more threads to be had: those that run take the rest
            }
        }
        work(0);
        for (int w = 1; w < workers; ++w)
            if (t[w].joinable()) t[w].join();
        return (hipError_t)err.load();
    }

    void release()
    {
        for (int w = 0; w < kWorkers; ++w) {
            if (slot_[w]) (void)hipHostFree(slot_[w]);
            if (done_[w]) (void)hipEventDestroy(done_[w]);
            slot_[w] = nullptr;
            done_[w] = nullptr;
        }
        for (auto &s : stream_)
            if (s) {
                (void)hipStreamDestroy(s);
                s = nullptr;
            }
        size_ = 0;
    }

private:
    static constexpr int kWorkers = 8;
    static constexpr size_t kChunk = size_t(2) << 20;

    static constexpr int kStreams = 3;
    static constexpr size_t kSpread = size_t(32) << 20;

    // as many workers as there is pinned memory for, one at least
    hipError_t reserve(int n, size_t bytes, int &got, int &streams)
    {
        const int want = std::min(n, kWorkers);
        const bool spread = n * bytes >= kSpread;
        if (bytes > size_) {
            for (auto &s : slot_)
                if (s) {
                    (void)hipHostFree(s);
                    s = nullptr;
                }
            size_ = bytes;
        }
        for (got = 0; got < want; ++got) {
            hipError_t e = hipSuccess;
            if (!slot_[got]) e = hipHostMalloc(reinterpret_cast<void **>(&slot_[got]), size_, hipHostMallocDefault);
            if (!e && !done_[got]) e = hipEventCreateWithFlags(&done_[got], hipEventDisableTiming);
            if (e) {
                (void)hipGetLastError();
                if (!got) return e;
                break;
            }
        }
        for (streams = 1; spread && streams < std::min(got, kStreams); ++streams)
            if (!stream_[streams])
                if (hipError_t e = hipStreamCreateWithFlags(&stream_[streams], hipStreamNonBlocking)) return e;
        return hipSuccess;
    }

    std::mutex call_;
    char *slot_[kWorkers] = {};
    hipEvent_t done_[kWorkers] = {};
    size_t size_ = 0;
    hipStream_t stream_[kStreams] = {};  // 0: the caller's
};

}  // namespace dgpu
