// cn_readback.cpp on the CPU: its HIP calls are stood in for by host memory,
// and allocations and copies can be made to fail one by one. Compiled together
// with cenote_amd/csrc/cn_readback.cpp and run by tests/test_readback_host.py:
// prints a line per call and exits with 0 when all went as they should.

#include <atomic>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <vector>

#include "cn_handles.h"
#include "cn_readback.h"

namespace {
thread_local long allocations_left = -1;  // -1: none fails
std::atomic<long> copies_left{-1};
std::atomic<int> in_flight{0};
bool pinned = true;
long pinned_bytes = 0, streams = 0;

bool spend(std::atomic<long>& left) { return left.load() >= 0 && left.fetch_sub(1) == 0; }
}  // namespace

void* operator new(size_t n) {
    if (allocations_left >= 0 && allocations_left-- == 0) throw std::bad_alloc();
    if (void* p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

extern "C" {
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "made to fail"; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned int) {
    *p = pinned ? std::malloc(n) : nullptr;
    pinned_bytes += n;
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void* p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipFree(void*) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned int) {
    *s = reinterpret_cast<hipStream_t>(std::malloc(1));
    ++streams;
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    std::free(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipMemcpy(void* dst, const void* src, size_t n, hipMemcpyKind) {
    std::memcpy(dst, src, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind, hipStream_t) {
    in_flight.fetch_add(1);
    const bool fails = spend(copies_left);
    if (!fails) std::memcpy(dst, src, n);
    in_flight.fetch_sub(1);
    return fails ? hipErrorUnknown : hipSuccess;
}
}

namespace cn {
int fail(int status, const char*, ...) { return status; }
}  // namespace cn

namespace {

struct Call {
    std::vector<float> src, dst;
    int run(cn::Readback& rb, size_t count, float divisor) {
        src.resize(count);
        dst.assign(count, -1.0f);
        for (size_t i = 0; i < count; ++i) src[i] = float(i % 65521);
        const cn::ReadArray a{src.data(), dst.data(), count, divisor};
        return cn::read_back(0, rb, &a, 1);
    }
    bool whole(float divisor) const {
        for (size_t i = 0; i < src.size(); ++i)
            if (dst[i] != src[i] / divisor) return false;
        return true;
    }
};

int failures = 0;
void check(bool ok, const char* what, long k) {
    std::printf("%s %s %ld\n", ok ? "ok" : "FAILED", what, k);
    std::fflush(stdout);
    failures += !ok;
}

}  // namespace

int main() {
    constexpr size_t SLOT = cn::Readback::SLOT / sizeof(float);
    cn::Readback rb;
    Call call;
    // A context's first small image takes no staging, the next ones what one
    // worker needs, and a large one the rest.
    check(call.run(rb, 1000, 3.0f) == CN_OK && call.whole(3.0f) && pinned_bytes == 0 && streams == 0, "first", 1000);
    check(call.run(rb, 1000, 3.0f) == CN_OK && call.whole(3.0f) && pinned_bytes <= 2 << 20 && streams == 1, "next", 1000);
    check(call.run(rb, 4 * SLOT, 3.0f) == CN_OK && pinned_bytes <= 4 << 20 && streams == 1, "next", 4 * SLOT);
    check(call.run(rb, 40 * SLOT, 3.0f) == CN_OK && pinned_bytes <= 16 << 20 && streams == 8, "next", 40 * SLOT);
    // One piece, several in one copy each, several workers, all of them; last pieces not full.
    for (size_t count : {size_t(1), SLOT, SLOT + 1, 4 * SLOT, 4 * SLOT + 1, 9 * SLOT + 7, 40 * SLOT + 3})
        for (float divisor : {1.0f, 3.0f})
            check(call.run(rb, count, divisor) == CN_OK && call.whole(divisor), "values", long(count));
    // Each allocation of the calling thread fails in turn, those that start a
    // worker among them: the call then fails as a whole or leaves the share to
    // the workers it has, and the staging serves the next call.
    const size_t count = 40 * SLOT + 3;
    for (long k = 0;; ++k) {
        call.src.reserve(count);
        call.dst.reserve(count);
        allocations_left = k;
        const int status = call.run(rb, count, 3.0f);
        const bool all = allocations_left >= 0;  // none failed any more
        allocations_left = -1;
        check(status == CN_E_ALLOC || (status == CN_OK && call.whole(3.0f)), "allocation", k);
        if (all) break;
    }
    check(call.run(rb, count, 3.0f) == CN_OK && call.whole(3.0f), "after failed allocations", 0);
    // Each copy fails in turn.
    for (long k = 0; k < 41; k += 5) {
        copies_left = k;
        const int status = call.run(rb, count, 3.0f);
        copies_left = -1;
        check(status != CN_OK && in_flight.load() == 0, "copy", k);
    }
    check(call.run(rb, count, 3.0f) == CN_OK && call.whole(3.0f), "after failed copies", 0);
    // No pinned memory: by way of pageable copies.
    cn::Readback bare;
    pinned = false;
    check(call.run(bare, count, 3.0f) == CN_OK && call.whole(3.0f), "without pinned memory", 0);
    return failures ? 1 : 0;
}
