// The host BVH builder behind a C call, for tests of its limits: compiled
// together with cenote_amd/csrc/cn_bvh.cpp (tests/bvh_host.py).

#include <cstdio>
#include <cstring>

#include "cn_bvh.h"

extern "C" int bvh_host_build(const float* corners, uint32_t count, uint32_t max_stack, uint32_t most4,
                              uint32_t most8, uint32_t* nodes4, uint32_t* depth4, uint32_t* nodes8, uint32_t* depth8,
                              char* error, size_t capacity) {
    std::vector<cn::WorldTriangle> input(count);
    for (uint32_t i = 0; i < count; ++i) {
        const float* p = corners + 9 * size_t(i);
        input[i] = {cn::V3(p[0], p[1], p[2]), cn::V3(p[3], p[4], p[5]), cn::V3(p[6], p[7], p[8]), 0, i, 0};
    }
    cn::Bvh4 out;
    std::string message;
    const bool ok = cn::build_bvh4(input, {max_stack, most4, most8}, &out, &message);
    *nodes4 = uint32_t(out.nodes.size());
    *depth4 = out.max_depth;
    *nodes8 = uint32_t(out.nodes8.size());
    *depth8 = out.max_depth8;
    std::snprintf(error, capacity, "%s", ok ? "" : message.c_str());
    return ok ? 0 : 1;
}
