// cn_readback.cpp — results from device memory into the caller's arrays.
//
// A 1080p film with its guides is 108 MB. Copied array by array into pageable
// memory by one thread, and divided by the sample count by the same thread
// afterwards, it took 11 ms of a 30 ms frame: the runtime's staging copies,
// the first-touch faults of the caller's fresh arrays and the division follow
// one another. Here the arrays are cut into pieces of at most 1 MiB, and
// workers (one up to 4 MiB, then up to eight) copy pieces into pinned slots,
// each worker's next copy in flight while it divides the piece it has into the
// caller's array.

#include "cn_readback.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <new>
#include <system_error>
#include <thread>
#include <vector>

#include "cn_handles.h"

namespace cn {

hipError_t Readback::prepare(int pairs, int workers) {
    for (int w = 0; w < pairs; ++w)
        if (!slots[w]) {
            const hipError_t e = hipHostMalloc(reinterpret_cast<void**>(&slots[w]), 2 * SLOT, hipHostMallocDefault);
            if (e != hipSuccess) {
                slots[w] = nullptr;
                return e;
            }
        }
    for (int w = 0; w < workers; ++w)
        if (!streams[w]) {
            const hipError_t e = hipStreamCreateWithFlags(&streams[w], hipStreamNonBlocking);
            if (e != hipSuccess) return e;
        }
    return hipSuccess;
}

Readback::~Readback() {
    for (hipStream_t s : streams)
        if (s) (void)hipStreamDestroy(s);
    for (char* p : slots)
        if (p) (void)hipHostFree(p);
}

namespace {

// `count` values of an array from value `first` on.
struct Piece {
    const ReadArray* a;
    size_t first, count;
};

// One band's pixels of LANES values, walked column by column from `src`, into
// rows of `row` values from `dst` on. (The size of a pixel's copy is fixed: as a
// call of memcpy each, an image's pixels took up to 10% longer or shorter by
// where the compiler put the loop.)
template <uint32_t LANES>
void land_band(float* dst, const float* src, uint32_t width, uint32_t rows, size_t row) {
    for (uint32_t x = 0; x < width; ++x)
        for (uint32_t y = 0; y < rows; ++y, src += LANES)
            std::memcpy(dst + size_t(y) * row + size_t(x) * LANES, src, LANES * sizeof(float));
}

// The values of one piece, staged at `in`, into the caller's array.
void land(const Piece& p, const float* in) {
    const ReadArray& a = *p.a;
    if (a.width == 0) {
        float* out = a.dst + p.first;
        if (a.divisor == 1.0f) {
            std::memcpy(out, in, p.count * sizeof(float));
        } else {
            for (size_t i = 0; i < p.count; ++i) out[i] = in[i] / a.divisor;
        }
        return;
    }
    // Whole bands: 8 rows (fewer in the last), walked column by column.
    const size_t row = size_t(a.width) * a.lanes, band = row * 8;
    for (size_t at = 0; at < p.count; at += band) {
        const uint32_t y0 = uint32_t((p.first + at) / band) * 8;
        const uint32_t rows = std::min(8u, a.height - y0);
        float* const dst = a.dst + size_t(y0) * row;
        if (a.lanes == 4) land_band<4>(dst, in + at, a.width, rows, row);
        else land_band<1>(dst, in + at, a.width, rows, row);
    }
}

}  // namespace

static int read_pieces(int device, Readback& rb, const ReadArray* arrays, int n) {
    constexpr size_t SLOT_VALUES = Readback::SLOT / sizeof(float);
    // An array by way of one pageable copy.
    auto whole = [](const ReadArray& a) {
        std::vector<float> values(a.count);
        CN_HIP(hipMemcpy(values.data(), a.src, a.count * sizeof(float), hipMemcpyDeviceToHost));
        land({&a, 0, a.count}, values.data());
        return int(CN_OK);
    };
    std::vector<Piece> pieces;
    for (int i = 0; i < n; ++i) {
        const ReadArray& a = arrays[i];
        if (!a.dst) continue;
        size_t step = SLOT_VALUES;
        if (a.width) {
            const size_t band = size_t(a.width) * 8 * a.lanes;
            if (band > SLOT_VALUES) {
                // A band that fills more than a slot.
                if (int e = whole(a)) return e;
                continue;
            }
            step = SLOT_VALUES / band * band;
        }
        for (size_t first = 0; first < a.count; first += step)
            pieces.push_back({&a, first, std::min(step, a.count - first)});
    }
    if (pieces.empty()) return CN_OK;
    const bool one = pieces.size() <= 4;  // copied by one stream, each piece into a slot of its own
    const int workers = one ? 1 : int(std::min<size_t>(Readback::WORKERS, pieces.size() / 2));
    std::lock_guard<std::mutex> lock(rb.busy);
    const bool first = !rb.used;
    rb.used = true;
    if ((one && first) || rb.prepare(one ? int(pieces.size() + 1) / 2 : workers, workers) != hipSuccess) {
        // A context's first small read-back, or no pinned memory (or streams) to be had.
        (void)hipGetLastError();
        const ReadArray* last = nullptr;
        for (const Piece& p : pieces) {
            if (p.a == last) continue;
            last = p.a;
            if (int e = whole(*last)) return e;
        }
        return CN_OK;
    }
    auto copy = [&](int worker, int slot, const Piece& p) {
        return hipMemcpyAsync(rb.slot(slot), p.a->src + p.first, p.count * sizeof(float),
                              hipMemcpyDeviceToHost, rb.streams[worker]);
    };
    auto staged = [&](int slot) { return reinterpret_cast<const float*>(rb.slot(slot)); };
    if (one) {
        hipError_t e = hipSuccess;
        for (size_t k = 0; k < pieces.size() && e == hipSuccess; ++k) e = copy(0, int(k), pieces[k]);
        const hipError_t done = hipStreamSynchronize(rb.streams[0]);  // also before the slots are let go
        CN_HIP(e != hipSuccess ? e : done);
        for (size_t k = 0; k < pieces.size(); ++k) land(pieces[k], staged(int(k)));
        return CN_OK;
    }
    std::atomic<size_t> next{0};
    std::atomic<int> failed{int(hipSuccess)};
    auto work = [&](int w) {
        hipError_t e = hipSetDevice(device);
        size_t k = next.fetch_add(1);
        int slot = 2 * w;
        if (e == hipSuccess && k < pieces.size()) e = copy(w, slot, pieces[k]);
        while (e == hipSuccess && k < pieces.size()) {
            e = hipStreamSynchronize(rb.streams[w]);
            if (e != hipSuccess) break;
            const size_t then = next.fetch_add(1);
            const int other = slot ^ 1;
            if (then < pieces.size()) e = copy(w, other, pieces[then]);
            land(pieces[k], staged(slot));
            k = then;
            slot = other;
        }
        if (e != hipSuccess) {
            (void)hipStreamSynchronize(rb.streams[w]);
            failed.store(int(e));
        }
    };
    // The calling thread is worker 0; a thread that cannot be had (the system's
    // limit, or no memory for its state) leaves its share to the others. Nothing
    // may leave this scope before they are joined.
    std::vector<std::thread> threads;
    threads.reserve(workers);
    for (int w = 1; w < workers; ++w) {
        try {
            threads.emplace_back(work, w);
        } catch (const std::system_error&) {
            break;
        } catch (const std::bad_alloc&) {
            break;
        }
    }
    work(0);
    for (std::thread& t : threads) t.join();
    CN_HIP(hipError_t(failed.load()));
    return CN_OK;
}

int read_back(int device, Readback& rb, const ReadArray* arrays, int n) {
    try {
        return read_pieces(device, rb, arrays, n);
    } catch (const std::bad_alloc&) {
        return fail(CN_E_ALLOC, "out of host memory reading results back");
    }
}

}  // namespace cn
