// cn_readback.h — results from device memory into the caller's arrays.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <hip/hip_runtime.h>

#include <mutex>

namespace cn {

// A context's pinned staging for read-backs: two 1 MiB slots and a stream per
// worker, each taken by the first read-back that needs it and given back with
// the context. The first read-back of a context, if it is one worker's, goes
// without: making one worker's share takes 3 ms and all of it 8, which a
// program that reads one small image back would not see again (that call 14 ms
// with all of the staging made for it, 5 to 7 without, and 8 with a worker's;
// later calls of 16 x 16 to 256 x 256 pixels are up to 45 us faster staged).
// One read-back uses it at a time.
struct Readback {
    std::mutex busy;
    bool used = false;
    static constexpr size_t SLOT = size_t(1) << 20;
    static constexpr int WORKERS = 8;
    char* slots[WORKERS] = {};  // two each
    hipStream_t streams[WORKERS] = {};
    // Makes the first `pairs` workers' slots and the first `workers` ones' streams.
    hipError_t prepare(int pairs, int workers);
    char* slot(int i) const { return slots[i / 2] + SLOT * (i % 2); }
    ~Readback();
};

// One array to read back: `count` f32 from device memory `src`, each divided
// by `divisor` where that is not 1; with `width`, the values are pixels of
// `lanes` (4 or 1) values in band order (band_pixel) and land row-major.
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
