// cn_readback.h — results from device memory into the caller's arrays.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <hip/hip_runtime.h>

#include <mutex>

namespace cn {

// A context's pinned staging for read-backs: 16 MiB in SLOTS slots and
// a stream per worker, taken at the first read-back and given back with
// the context. One read-back uses it at a time.
struct Readback {
    std::mutex busy;
    char* slots = nullptr;
    static constexpr size_t SLOT = size_t(1) << 20;
    static constexpr int WORKERS = 8;
    static constexpr int SLOTS = 2 * WORKERS;
    hipStream_t streams[WORKERS] = {};
    hipError_t prepare();
    ~Readback();
};

// One array to read back: `count` f32 from device memory `src`, each divided
// by `divisor` where that is not 1; with `width`, the values are `lanes`-wide
// pixels in band order (band_pixel) and land row-major.
struct ReadArray {
    const float* src;
    float* dst;  // null: skipped
    size_t count;
    float divisor = 1.0f;
    uint32_t lanes = 1, width = 0, height = 0;
};

// Reads the arrays back; what wrote them must have finished. CN_OK or a
// failing status.
int read_back(int device, Readback& rb, const ReadArray* arrays, int n);

}  // namespace cn
