// nb_hostcopy.h -- device arrays into a caller's pageable host memory.
//
// hipMemcpyAsync into pageable memory takes 9 to 21 us per call and runs at 8 to
// 18 GB/s, bound by one thread that faults in and fills the caller's pages.  Here
// the arrays go through pinned memory owned by the context or ensemble:
//  - small copies (up to kSmall) by one kernel that stores them there, one wait,
//    and a memcpy per array;
//  - large ones (from kLarge) are cut into chunks that pass through a ring of
//    pinned slots by DMA (56 GB/s), and several threads fill the caller's pages
//    while later chunks are on their way.
// In between, the runtime's copies into pageable memory are as fast or the fastest:
// six arrays of 21,846 bodies (1 MiB) 0.100 ms and by the kernel 0.061, of 43,690
// (2 MiB) 0.146 and 0.107, but into the caller's pinned memory 0.095 and 0.098; of
// 131,073 bodies 0.40 ms, of 349,525 (16 MiB) 0.93, through the ring in chunks
// of 256 KiB 0.59 and 1.38; of 360,000 0.94 and, in chunks of 1 MiB, 0.75.
// Six arrays of 1024 bodies: 25 us instead of 105; of 1,048,576 bodies (50 MB)
// 2.5 ms instead of 6.4; of 4,194,304 7.9 ms instead of 21.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstring>
#include <thread>
#include <vector>

namespace nb {

// arrays of doubles stored into pinned host memory (dst is a host address that
// the device can write)
struct CopyOut {
    const double *src[6];
    double *dst[6];
    size_t n[6];
};
hipError_t launch_copy_out(const CopyOut &c, int count, hipStream_t s);

class HostCopier {
  public:
    struct Array {
        double *dst;
        const double *src;  // device
        size_t n;
    };
    static constexpr int kArrays = 6;

    // Pinned memory for the copies of six arrays (a state) or three (accelerations) of
    // n doubles, made with its owner: a first copy would pay for the allocation and
    // for a fault per page (1.6 us).  The first accelerations of 30,001 bodies took
    // 83 us that way, 52 now; the first state of 360,000 1.4 ms, 0.9 now.
    void reserve_for(size_t n) noexcept {
        if (6 * n * sizeof(double) >= kLarge) {
            if (reserve(kSlots * kChunk)) (void)make_events();
            return;
        }
        for (size_t arrays : {6, 3}) {
            const size_t bytes = arrays * n * sizeof(double);
            if (bytes > kSmall) continue;
            if (!reserve(bytes)) return;
            for (size_t o = 0; o < bytes; o += 4096) ring_[o] = 0;
            return;
        }
    }

    ~HostCopier() {
        for (uint32_t k = 0; k < nevents_; ++k) (void)hipEventDestroy(events_[k]);
        if (ring_) (void)hipHostFree(ring_);
    }

    // Copies the arrays behind the work already issued on `stream`; returns when
    // they have arrived.  Its callers are C entry points: nothing here throws (the
    // threads are the only host memory asked for, and copying goes on without them).
    hipError_t copy(hipStream_t stream, const Array *a, int count) noexcept {
        size_t total = 0;
        for (int k = 0; k < count; ++k) total += a[k].n * sizeof(double);
        if (total == 0) return hipStreamSynchronize(stream);
        const OnDevice device(stream);
        if (total <= (count == 1 ? kOne : kSmall) && reserve(total)) return small(stream, a, count);
        if (total < kLarge) return runtime(stream, a, count);
        // Pinned memory of the caller's takes a DMA itself: six arrays of 360,000
        // bodies 0.36 ms, through the ring 0.75; of 1,048,576 0.94 and 1.77.
        Array paged[kArrays], pinned[kArrays];
        int npaged = 0, npinned = 0;
        size_t bytes = 0;
        for (int k = 0; k < count; ++k) {
            if (is_pinned(a[k].dst)) {
                pinned[npinned++] = a[k];
            } else {
                paged[npaged++] = a[k];
                bytes += a[k].n * sizeof(double);
            }
        }
        if (npinned) {
            const hipError_t e = runtime(stream, pinned, npinned);
            if (e != hipSuccess) return e;
        }
        if (bytes >= kLarge && reserve(kSlots * kChunk) && make_events())
            return large(stream, paged, npaged);
        return runtime(stream, paged, npaged);  // a few, or no ring to be had
    }

  private:
    // The stream's device is current while this lives, whatever the caller's is: an
    // event is recorded, and a kernel launched, on the stream of its own device.
    struct OnDevice {
        int before = -1;
        explicit OnDevice(hipStream_t stream) {
            int own = 0, now = 0;
            if (hipStreamGetDevice(stream, &own) == hipSuccess && hipGetDevice(&now) == hipSuccess &&
                own != now && hipSetDevice(own) == hipSuccess)
                before = now;
        }
        ~OnDevice() {
            if (before >= 0) (void)hipSetDevice(before);
        }
    };

    static constexpr size_t kSmall = size_t(7) << 18;
    // One array alone: the runtime takes 21 us up to 16 KiB and 9.1 us just above (64
    // KiB 11.4, 1 MiB 64), the kernel 13.4 and as much (14.5, 66).
    static constexpr size_t kOne = size_t(16) << 10;
    static constexpr size_t kLarge = size_t(16) << 20;
    static constexpr size_t kChunk = size_t(1) << 20;
    static constexpr uint32_t kSlots = 8;
    static constexpr unsigned kThreads = 8;

    uint8_t *ring_ = nullptr;
    size_t ring_bytes_ = 0;
    hipEvent_t events_[kSlots] = {};
    uint32_t nevents_ = 0;

    // false: refused, with the runtime's last error cleared (the caller has another way)
    bool reserve(size_t bytes) {
        if (ring_bytes_ >= bytes) return true;
        if (ring_) (void)hipHostFree(ring_);
        ring_ = nullptr;
        ring_bytes_ = 0;
        if (hipHostMalloc((void **)&ring_, bytes, hipHostMallocDefault) != hipSuccess) {
            ring_ = nullptr;
            (void)hipGetLastError();
            return false;
        }
        ring_bytes_ = bytes;
        return true;
    }

    bool make_events() {
        for (; nevents_ < kSlots; ++nevents_)
            if (hipEventCreateWithFlags(&events_[nevents_], hipEventDisableTiming) != hipSuccess) {
                (void)hipGetLastError();
                return false;
            }
        return true;
    }

    static bool is_pinned(const void *p) {
        hipPointerAttribute_t at;
        if (hipPointerGetAttributes(&at, p) != hipSuccess) {
            (void)hipGetLastError();
            return false;
        }
        return at.type == hipMemoryTypeHost;
    }

    hipError_t runtime(hipStream_t stream, const Array *a, int count) {
        hipError_t e = hipSuccess;
        for (int k = 0; k < count && e == hipSuccess; ++k)
            e = hipMemcpyAsync(a[k].dst, a[k].src, a[k].n * sizeof(double), hipMemcpyDeviceToHost,
                               stream);
        const hipError_t s = hipStreamSynchronize(stream);
        return e != hipSuccess ? e : s;
    }

    // ring_ holds the arrays
    hipError_t small(hipStream_t stream, const Array *a, int count) {
        CopyOut arg{};
        size_t at = 0;
        for (int k = 0; k < count; ++k) {
            arg.src[k] = a[k].src;
            arg.dst[k] = (double *)ring_ + at;
            arg.n[k] = a[k].n;
            at += a[k].n;
        }
        const hipError_t e = launch_copy_out(arg, count, stream);
        const hipError_t s = hipStreamSynchronize(stream);
        if (e != hipSuccess) return e;
        if (s != hipSuccess) return s;
        for (int k = 0; k < count; ++k)
            std::memcpy(a[k].dst, arg.dst[k], a[k].n * sizeof(double));
        return hipSuccess;
    }

    // ring_ holds kSlots chunks and the events are there
    hipError_t large(hipStream_t stream, const Array *a, int count) {
        hipError_t e = hipSuccess;
        struct Chunk {
            uint8_t *dst;
            const uint8_t *src;
            size_t bytes;
        };
        // array k has the chunks [first[k], first[k + 1])
        uint32_t first[kArrays + 1] = {};
        for (int k = 0; k < count; ++k)
            first[k + 1] = first[k] + (uint32_t)((a[k].n * sizeof(double) + kChunk - 1) / kChunk);
        const uint32_t n = first[count];
        const auto chunk_at = [&](uint32_t i) {
            int k = 0;
            while (i >= first[k + 1]) ++k;
            const size_t o = (size_t)(i - first[k]) * kChunk;
            return Chunk{(uint8_t *)a[k].dst + o, (const uint8_t *)a[k].src + o,
                         std::min(kChunk, a[k].n * sizeof(double) - o)};
        };
        // Chunk i goes through slot i mod kSlots.  This thread issues the DMAs and
        // waits for them in order; arrived: chunks that lie in their slots;
        // filled[s]: chunks that have left slot s.  With threads they fill the
        // caller's pages (no HIP calls there), without this one does.
        std::atomic<uint32_t> arrived{0}, next{0};
        std::atomic<uint32_t> filled[kSlots];
        for (auto &f : filled) f.store(0);
        std::atomic<bool> failed{false};
        auto fill = [&](uint32_t i) {
            const Chunk c = chunk_at(i);
            std::memcpy(c.dst, ring_ + (i % kSlots) * kChunk, c.bytes);
            filled[i % kSlots].store(i / kSlots + 1, std::memory_order_release);
        };
        auto worker = [&] {
            for (;;) {
                const uint32_t i = next.fetch_add(1);
                if (i >= n) return;
                while (arrived.load(std::memory_order_acquire) <= i) {
                    if (failed.load()) return;
                    std::this_thread::yield();
                }
                fill(i);
            }
        };
        std::vector<std::thread> threads;
        const unsigned cores = std::max(1u, std::thread::hardware_concurrency());
        try {
            threads.reserve(kThreads);
            for (unsigned t = 0; t < std::min(cores, kThreads); ++t)
                threads.emplace_back(worker);
        } catch (...) {  // fewer threads, or none
        }
        for (uint32_t issued = 0, got = 0; got < n && e == hipSuccess;) {
            if (issued < n && issued - got < kSlots &&
                filled[issued % kSlots].load(std::memory_order_acquire) >= issued / kSlots) {
                const Chunk c = chunk_at(issued);
                e = hipMemcpyAsync(ring_ + (issued % kSlots) * kChunk, c.src, c.bytes,
                                   hipMemcpyDeviceToHost, stream);
                if (e == hipSuccess) e = hipEventRecord(events_[issued % kSlots], stream);
                ++issued;
            } else if (got < issued) {
                e = hipEventSynchronize(events_[got % kSlots]);
                if (e != hipSuccess) break;
                arrived.store(++got, std::memory_order_release);
                if (threads.empty()) fill(got - 1);
            } else {
                std::this_thread::yield();  // every slot waits to be filled
            }
        }
        if (e != hipSuccess) failed.store(true);
        for (auto &t : threads) t.join();
        const hipError_t s = hipStreamSynchronize(stream);
        return e != hipSuccess ? e : s;
    }
};

}  // namespace nb
