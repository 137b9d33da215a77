// readback.h -- state reads: per-item doubles computed on the device into the caller's arrays.
//
// A direct copy into pageable memory runs at 5-15 GB/s: the runtime bounces it through its own
// buffer with one host thread, which also takes the page faults of a fresh array.  Here the
// kernels fill the handle's device buffer by halves, copies of 2 MiB bring it to page-locked
// slots (up to four under way), and a team of host threads moves each slot on as it arrives.
// Before the first one the team touches all pages of the caller's arrays, beside the first four
// copies only: the link then waits for it through most of a long read's touching.  Measured on
// fresh arrays, before -> now: a dense velocity and density of 208 MB 20.6 -> 7.9 ms, a
// colour-gradient state of 135 MB 12.2 -> 4.8 ms, a state of 29 MB 1.77 -> 0.87 ms, one of 0.8 MB with
// its run of ten steps 198 -> 180 us.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace lbm {

// Page-locked slots of the reads under way, shared by the handles of the process: a read takes a
// set for its duration, with as many slots as its bytes fill.  Idle sets are kept, at most one for each
// handle alive: making and freeing a set of four slots costs 0.2 ms.  There are PIN_SETS at most (128
// MiB); further reads at the same time copy straight into the caller's arrays.  Thread-safe.
constexpr int PIN_SETS = 16;
constexpr int PIN_SLOTS = 4;
constexpr size_t PIN_BYTES = size_t(2) << 20;
struct PinnedSet {
    void *slot[PIN_SLOTS] = {nullptr};
    hipEvent_t done[PIN_SLOTS] = {nullptr};
    int device = -1;   // the events' device
};
// a set for a read on the device, with its first `slots` slots; false where all are in use or page-locked
// memory cannot be had (no error is left pending)
bool pinned_take(int device, int slots, PinnedSet &out);
void pinned_return(PinnedSet &s);
// a member of every handle that reads back
struct PinnedUser {
    PinnedUser();
    ~PinnedUser();
    PinnedUser(const PinnedUser &) = delete;
    PinnedUser &operator=(const PinnedUser &) = delete;
};

// one output: `width` doubles an item, to dst (nullptr: not wanted)
struct ReadPart {
    double *dst;
    int width;
};
constexpr int READ_PARTS = 6;

// host side of a read: `bytes` bytes at byte offset `at` of the device chunk that holds items
// [i0, i1) of the parts, one after the other
void read_scatter(const ReadPart *parts, int np, int64_t i0, int64_t i1, size_t at, size_t bytes, const void *from);
// write to every page of the parts' arrays, with a team of threads, leaving what is in them
void read_touch(const ReadPart *parts, int np, int64_t items);

// the wanted parts of items [i0, i1) in device memory from base on, one after the other, to p; their bytes
inline size_t place_parts(const ReadPart *parts, int np, int64_t i0, int64_t i1, char *base, double **p)
{
    size_t at = 0;
    for (int k = 0; k < np; ++k) {
        p[k] = parts[k].dst ? (double *)(base + at) : nullptr;
        if (parts[k].dst) at += sizeof(double) * (size_t)parts[k].width * (size_t)(i1 - i0);
    }
    return at;
}

// read_back without page-locked slots or an allocation: each chunk straight into the caller's arrays
template <typename F>
hipError_t read_direct(hipStream_t s, int64_t n, const ReadPart *parts, int np, void *buf, size_t buf_bytes, size_t item,
                       int64_t step, F &&fill)
{
    const int64_t chunk = std::max<int64_t>(step, (int64_t)(buf_bytes / item) / step * step);
    hipError_t e = hipSuccess;
    for (int64_t i0 = 0; i0 < n && e == hipSuccess; i0 += chunk) {
        const int64_t i1 = std::min(n, i0 + chunk);
        double *p[READ_PARTS] = {nullptr};
        place_parts(parts, np, i0, i1, (char *)buf, p);
        e = fill(i0, i1, p);
        for (int k = 0; k < np && e == hipSuccess; ++k)
            if (p[k])
                e = hipMemcpyAsync(parts[k].dst + i0 * parts[k].width, p[k],
                                   sizeof(double) * (size_t)parts[k].width * (size_t)(i1 - i0), hipMemcpyDeviceToHost, s);
    }
    const hipError_t es = hipStreamSynchronize(s);
    return e == hipSuccess ? es : e;
}

// Read items 0 .. n-1 of the parts.  fill(i0, i1, p) queues on s the work that writes items
// [i0, i1) of each wanted part k to p[k].  buf: device memory, buf_bytes.  step: items per chunk
// are a multiple of it.  Every copy has ended when the call returns, with an error too.
template <typename F>
hipError_t read_back(int device, hipStream_t s, int64_t n, const ReadPart *parts, int np, void *buf, size_t buf_bytes,
                     int64_t step, F &&fill)
{
    int width = 0;
    for (int k = 0; k < np; ++k) width += parts[k].dst ? parts[k].width : 0;
    if (width == 0 || n <= 0) return hipSuccess;
    const size_t item = sizeof(double) * (size_t)width;
    PinnedSet set;
    const int slots = (int)std::min<size_t>(PIN_SLOTS, ((size_t)n * item + PIN_BYTES - 1) / PIN_BYTES);
    if (!pinned_take(device, slots, set)) return read_direct(s, n, parts, np, buf, buf_bytes, item, step, fill);
    hipError_t e = hipSuccess;
    const int64_t chunk = std::max<int64_t>(step, (int64_t)(buf_bytes / 2 / item) / step * step);
    struct Piece {
        int64_t i0, i1;
        size_t at, bytes;
    } ring[PIN_SLOTS];
    int64_t queued = 0, taken = 0;
    bool touched = false;
    auto take = [&]() {   // the oldest piece under way
        if (!touched) {
            touched = true;
            read_touch(parts, np, n);
        }
        const int k = (int)(taken++ % slots);
        const hipError_t w = hipEventSynchronize(set.done[k]);
        if (w == hipSuccess) read_scatter(parts, np, ring[k].i0, ring[k].i1, ring[k].at, ring[k].bytes, set.slot[k]);
        return w;
    };
    int half = 0;
    for (int64_t i0 = 0; i0 < n && e == hipSuccess; i0 += chunk, half ^= 1) {
        const int64_t i1 = std::min(n, i0 + chunk);
        // the half's last copies are ahead of this chunk's kernels on the stream
        char *base = (char *)buf + (half ? buf_bytes / 2 : 0);
        double *p[READ_PARTS] = {nullptr};
        const size_t at = place_parts(parts, np, i0, i1, base, p);
        e = fill(i0, i1, p);
        for (size_t o = 0; o < at && e == hipSuccess; o += PIN_BYTES) {
            if (queued - taken == slots) e = take();
            if (e != hipSuccess) break;
            const int k = (int)(queued % slots);
            ring[k] = Piece{i0, i1, o, std::min(PIN_BYTES, at - o)};
            e = hipMemcpyAsync(set.slot[k], base + o, ring[k].bytes, hipMemcpyDeviceToHost, s);
            if (e == hipSuccess) e = hipEventRecord(set.done[k], s);
            if (e == hipSuccess) ++queued;
        }
    }
    while (taken < queued && e == hipSuccess) e = take();
    const hipError_t es = hipStreamSynchronize(s);   // after an error, copies may be under way
    pinned_return(set);
    return e == hipSuccess ? es : e;
}

}  // namespace lbm
