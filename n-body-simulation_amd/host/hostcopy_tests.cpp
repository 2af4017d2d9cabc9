// hostcopy_tests.cpp -- the read-back of csrc/nb_hostcopy.h on the CPU.
//
// The few HIP calls that it makes are stand-ins here (copies are memcpy, pinned
// memory is malloc), so no GPU is needed and a failing call can be asked for.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <new>
#include <vector>

#include "../csrc/nb_hostcopy.h"

namespace {

bool no_heap = false;    // operator new fails
bool no_pinned = false;  // hipHostMalloc fails
bool no_events = false;  // hipEventCreateWithFlags fails
hipError_t last_error = hipSuccess;
const void *pinned_from = nullptr, *pinned_to = nullptr;  // the caller's pinned memory
int allocations = 0;  // of pinned memory and events, since it was reset
int copies = 0;  // runtime copies since it was reset
int device = 0;        // the current one
int stream_device = 0;  // the stream's
bool wrong_device = false;  // an event or a launch of another device than the stream's

int failures = 0;
void check(bool ok, const char *name, size_t n) {
    if (!ok) ++failures;
    std::printf("%s %s n=%zu\n", ok ? "PASS" : "FAIL", name, n);
}

}  // namespace

void *operator new(size_t bytes) {
    void *p = no_heap ? nullptr : std::malloc(bytes ? bytes : 1);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

extern "C" {
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) {
    ++allocations;
    if (no_pinned) return last_error = hipErrorOutOfMemory;
    *p = std::malloc(bytes);
    return hipSuccess;
}
hipError_t hipHostFree(void *p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
    ++allocations;
    if (no_events) return last_error = hipErrorOutOfMemory;
    wrong_device |= device != stream_device;
    *e = (hipEvent_t)std::malloc(1);
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    std::free((void *)e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetDevice(int *d) {
    *d = device;
    return hipSuccess;
}
hipError_t hipSetDevice(int d) {
    device = d;
    return hipSuccess;
}
hipError_t hipStreamGetDevice(hipStream_t, hipDevice_t *d) {
    *d = stream_device;
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *at, const void *p) {
    *at = hipPointerAttribute_t{};
    at->type = p >= pinned_from && p < pinned_to ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
    return hipSuccess;
}
hipError_t hipGetLastError() {
    const hipError_t e = last_error;
    last_error = hipSuccess;
    return e;
}
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t bytes, hipMemcpyKind, hipStream_t) {
    ++copies;
    std::memcpy(dst, src, bytes);
    return hipSuccess;
}
}

namespace nb {
hipError_t launch_copy_out(const CopyOut &c, int count, hipStream_t) {
    wrong_device |= device != stream_device;
    for (int k = 0; k < count; ++k) std::memcpy(c.dst[k], c.src[k], c.n[k] * sizeof(double));
    return hipSuccess;
}
}  // namespace nb

namespace {

// Copies `count` arrays of n doubles; true if every one arrived and nothing past its end.
bool copied(nb::HostCopier &copier, size_t n, int count) {
    std::vector<std::vector<double>> src(count), dst(count);
    std::vector<nb::HostCopier::Array> a;
    for (int k = 0; k < count; ++k) {
        src[k].resize(n);
        for (size_t i = 0; i < n; ++i) src[k][i] = 1.0 + (double)i + 1e7 * k;
        dst[k].assign(n + 1, -1.0);
        a.push_back({dst[k].data(), src[k].data(), n});
    }
    bool ok = copier.copy(nullptr, a.data(), count) == hipSuccess;
    for (int k = 0; k < count; ++k) {
        ok = ok && std::memcmp(dst[k].data(), src[k].data(), n * sizeof(double)) == 0;
        ok = ok && dst[k][n] == -1.0;
    }
    return ok;
}

// A host that refuses memory: the copy goes on with this thread alone, and no
// exception leaves it (its callers are C entry points).
void without_heap(size_t n) {
    std::vector<double> src(6 * n), dst(6 * n, -1.0);
    for (size_t i = 0; i < src.size(); ++i) src[i] = (double)i;
    nb::HostCopier::Array a[6];
    for (int k = 0; k < 6; ++k) a[k] = {dst.data() + k * n, src.data() + k * n, n};
    bool ok = false;
    {
        nb::HostCopier copier;
        no_heap = true;
        try {
            ok = copier.copy(nullptr, a, 6) == hipSuccess;
        } catch (...) {
        }
        no_heap = false;
    }
    check(ok && dst == src, "HostCopier.withoutHeap", n);
}

// The first `own` of six arrays lie in pinned memory of the caller's.
void pinned_destinations(size_t n, int own) {
    std::vector<double> src(6 * n), dst(6 * n, -1.0);
    for (size_t i = 0; i < src.size(); ++i) src[i] = (double)i;
    nb::HostCopier::Array a[6];
    for (int k = 0; k < 6; ++k) a[k] = {dst.data() + k * n, src.data() + k * n, n};
    pinned_from = dst.data();
    pinned_to = dst.data() + own * n;
    nb::HostCopier copier;
    copies = 0;
    const bool ok = copier.copy(nullptr, a, 6) == hipSuccess && dst == src;
    const int chunks = (int)((n * sizeof(double) + (1 << 20) - 1) >> 20);
    const bool ring = (6 - own) * n * sizeof(double) >= 16u << 20;
    check(ok && copies == own + (6 - own) * (ring ? chunks : 1), "HostCopier.pinned", n);
    pinned_from = pinned_to = nullptr;
}

}  // namespace

int main() {
    // edges of the small copies (1.75 MiB in all), the chunked ones (16 MiB) and a
    // chunk's end (six arrays, or one)
    for (size_t n : {1, 38229, 38230, 131071, 131072, 131073, 163840, 349525, 349526, 400001}) {
        nb::HostCopier copier;
        check(copied(copier, n, 6) && copied(copier, n, 3) && copied(copier, n, 1),
              "HostCopier.everyArray", n);
    }
    for (size_t n : {21845, 131072, 400001}) without_heap(n);
    // up to 1.75 MiB in all: no runtime copy; to 16 MiB one per array; from there on,
    // one per MiB
    for (size_t n : {21846, 38229, 38230, 131072, 131073, 349525, 349526, 400001}) {
        nb::HostCopier copier;
        const int chunks = (int)((n * sizeof(double) + (1 << 20) - 1) >> 20);
        copies = 0;
        const bool ok = copied(copier, n, 6);
        check(ok && copies == 6 * (n < 38230 ? 0 : n < 349526 ? 1 : chunks), "HostCopier.copiesPerArray", n);
    }
    // without pinned memory, or without events: the runtime's own copies, and no
    // error left behind for a later call
    for (size_t n : {1, 21845, 131072, 400001}) {
        for (bool *refused : {&no_pinned, &no_events}) {
            nb::HostCopier copier;
            *refused = true;
            copier.reserve_for(n);
            const bool ok = copied(copier, n, 6) && copied(copier, n, 3) && last_error == hipSuccess;
            *refused = false;
            check(ok && copied(copier, n, 6), "HostCopier.refused", n);
        }
    }
    // an error that an older call left in the runtime is not this copy's, and stays
    for (size_t n : {1, 21845, 131072, 400001}) {
        nb::HostCopier copier;
        last_error = hipErrorInvalidValue;
        const bool ok = copied(copier, n, 6);
        check(ok && last_error == hipErrorInvalidValue, "HostCopier.olderError", n);
        last_error = hipSuccess;
    }
    // one array alone: without a runtime copy up to 16 KiB
    for (size_t n : {1, 2048, 2049, 131072, 131073}) {
        nb::HostCopier copier;
        copies = 0;
        const bool ok = copied(copier, n, 1);
        check(ok && copies == (n <= 2048 ? 0 : 1), "HostCopier.oneArray", n);
    }
    // what the copies of a state and of accelerations need is made with the owner
    for (size_t n : {1, 21846, 38229, 38230, 76458, 76459, 349525, 349526, 700000}) {
        nb::HostCopier copier;
        copier.reserve_for(n);
        allocations = 0;
        const bool ok = copied(copier, n, 6) && copied(copier, n, 3);
        check(ok && allocations == 0, "HostCopier.madeWithOwner", n);
    }
    for (int own : {1, 3, 6}) pinned_destinations(400001, own);
    // another device than the stream's is current: it is again afterwards
    for (size_t n : {1, 131072, 400001}) {
        nb::HostCopier copier;
        stream_device = 1;
        const bool ok = copied(copier, n, 6);
        check(ok && !wrong_device && device == 0, "HostCopier.otherDevice", n);
        stream_device = 0;
    }
    return failures ? 1 : 0;
}
