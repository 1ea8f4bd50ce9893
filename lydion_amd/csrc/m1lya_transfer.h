// m1lya_transfer.h -- large device-to-host copies into pageable memory (both C interfaces).
//
// A plain copy into an array that the caller has just allocated is bound by one host thread,
// which moves the data out of the runtime's staging buffer and takes the page faults of the
// destination: 10.6 GB/s, and 5.7 GB/s of FP64 values where that thread also widened the batch's
// FP32 state.  The copy engine alone does 56 GB/s.  Here a few threads, the caller's among them,
// each bring chunks into a pinned buffer of their own and widen or copy them from there, so the
// engine, the faults and the conversion of different chunks overlap (64 MiB of FP64: 2.0 ms, was
// 6.3; the batch's FP32 state widened to the same size: 1.5 ms, was 11.8).
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

namespace m1t {

constexpr int kWorkers = 8;
constexpr size_t kChunkBytes = 1 << 21;
// Below this the threads cost about what they save (8 MiB: 0.40 ms, 0.51 by a plain copy; 2 MiB: 0.16
// by a plain copy).
constexpr size_t kMinBytes = 8u << 20;

// The pinned buffers of one context or batch: kWorkers chunks at most, allocated with the first
// large copy and kept until the owner goes.  Copies of one owner take turns.
class Download {
    std::mutex lock;
    void* buf[kWorkers] = {};
    hipEvent_t ev[kWorkers] = {};

    static void put(double* dst, const double* src, size_t n, double) { std::memcpy(dst, src, n * sizeof(double)); }
    static void put(double* dst, const float* src, size_t n, double scale)
    {
        for (size_t t = 0; t < n; ++t) dst[t] = (double)src[t] * scale;
    }

public:
    Download() = default;
    Download(const Download&) = delete;
    Download& operator=(const Download&) = delete;

    // With the owner's device current and its stream idle
    void release()
    {
        for (int w = 0; w < kWorkers; ++w) {
            if (ev[w]) (void)hipEventDestroy(ev[w]);
            if (buf[w]) (void)hipHostFree(buf[w]);
            ev[w] = nullptr;
            buf[w] = nullptr;
        }
    }

    // host[0 .. n) = src[0 .. n), FP32 values times scale, once the stream's work so far is done;
    // returns when the copy is complete, its outcome in result.  False: there is no pinned memory to
    // be had, and nothing was copied.
    template <class T>
    bool run(double* host, const T* src, size_t n, double scale, int device, hipStream_t stream, hipError_t& result)
    {
        std::lock_guard<std::mutex> hold(lock);
        constexpr size_t kElems = kChunkBytes / sizeof(T);
        const size_t chunks = (n + kElems - 1) / kElems;
        const unsigned cpus = std::max(1u, std::thread::hardware_concurrency());
        const int most = (int)std::min<size_t>(std::min<size_t>(kWorkers, cpus), chunks);
        int current = device;
        (void)hipGetDevice(&current);
        result = current != device ? hipSetDevice(device) : hipSuccess;
        int workers = 0;
        while (result == hipSuccess && workers < most && slot(workers)) ++workers;
        if (result == hipSuccess && workers > 0) result = copy(host, src, n, scale, device, stream, workers, chunks);
        if (current != device) (void)hipSetDevice(current);
        return result != hipSuccess || workers > 0;
    }

private:
    // Worker w's buffer and event
    bool slot(int w)
    {
        if (!buf[w] && hipHostMalloc(&buf[w], kChunkBytes, hipHostMallocDefault) != hipSuccess) buf[w] = nullptr;
        if (buf[w] && !ev[w] && hipEventCreateWithFlags(&ev[w], hipEventDisableTiming) != hipSuccess) ev[w] = nullptr;
        if (buf[w] && ev[w]) return true;
        (void)hipGetLastError();
        return false;
    }

    template <class T>
    hipError_t copy(double* host, const T* src, size_t n, double scale, int device, hipStream_t stream, int workers,
                    size_t chunks)
    {
        constexpr size_t kElems = kChunkBytes / sizeof(T);
        std::atomic<size_t> next{0};
        std::atomic<int> error{hipSuccess};
        auto work = [&](int w) {
            hipError_t e = hipSetDevice(device);
            for (size_t c; e == hipSuccess && error == hipSuccess && (c = next.fetch_add(1)) < chunks;) {
                const size_t o = c * kElems, m = std::min(kElems, n - o);
                e = hipMemcpyAsync(buf[w], src + o, m * sizeof(T), hipMemcpyDeviceToHost, stream);
                if (e == hipSuccess) e = hipEventRecord(ev[w], stream);
                if (e == hipSuccess) e = hipEventSynchronize(ev[w]);
                if (e == hipSuccess) put(host + o, static_cast<const T*>(buf[w]), m, scale);
            }
            if (e != hipSuccess) error = e;
        };
        std::vector<std::thread> threads;
        try {
            threads.reserve(workers);
            for (int w = 1; w < workers; ++w) threads.emplace_back(work, w);
        } catch (const std::exception&) {
            // no more threads to be had: those there are take every chunk
        }
        work(0);
        for (std::thread& t : threads) t.join();
        const hipError_t e = static_cast<hipError_t>(error.load());
        if (e != hipSuccess) (void)hipStreamSynchronize(stream);   // no copy into a buffer outlives the call
        return e;
    }
};

// Memory that the runtime knows (pinned, managed or a device's) takes a plain copy at full speed.
inline bool pageable(const void* p)
{
    hipPointerAttribute_t at;
    if (hipPointerGetAttributes(&at, p) != hipSuccess) {
        (void)hipGetLastError();   // an ordinary pointer
        return true;
    }
    return at.type == hipMemoryTypeUnregistered;
}

}  // namespace m1t
