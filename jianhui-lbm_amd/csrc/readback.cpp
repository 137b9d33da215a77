// readback.cpp -- host side of the state reads (readback.h).
#include "readback.h"

#include <omp.h>

#include <cstring>
#include <mutex>

namespace lbm {

namespace {
std::mutex mu;
int users = 0;                // handles
int sets = 0;                 // page-locked sets there are, idle or in a read
PinnedSet idle[PIN_SETS];     // the first n_idle
int n_idle = 0;

void free_set(PinnedSet &s)
{
    for (int k = 0; k < PIN_SLOTS; ++k) {
        if (s.slot[k]) (void)hipHostFree(s.slot[k]);
        if (s.done[k]) (void)hipEventDestroy(s.done[k]);
    }
    s = PinnedSet{};
}

// threads for a job of this many bytes: 256 KiB at least for each, eight at most (a copy out of
// the slots gained nothing from 16: 24 GB/s into fresh pages against 21)
int team(size_t bytes) { return (int)std::min<size_t>({size_t(8), (size_t)omp_get_max_threads(), 1 + bytes / (256u << 10)}); }
}  // namespace

PinnedUser::PinnedUser()
{
    std::lock_guard<std::mutex> lk(mu);
    ++users;
}

PinnedUser::~PinnedUser()
{
    std::lock_guard<std::mutex> lk(mu);
    --users;
    // a handle reads with one set at a time
    for (; sets > users && n_idle > 0; --sets) free_set(idle[--n_idle]);
}

bool pinned_take(int device, int slots, PinnedSet &out)
{
    out = PinnedSet{};
    out.device = device;
    {
        std::lock_guard<std::mutex> lk(mu);
        int pick = -1;   // an idle set of the device, one that has the slots if there is
        for (int k = 0; k < n_idle; ++k)
            if (idle[k].device == device && (pick < 0 || !idle[pick].done[slots - 1])) pick = k;
        if (pick >= 0) {
            out = idle[pick];
            idle[pick] = idle[--n_idle];
        } else {
            if (sets == PIN_SETS) {
                if (n_idle == 0) return false;
                free_set(idle[--n_idle]);   // of another device
                --sets;
            }
            ++sets;
        }
    }
    hipError_t e = hipSuccess;
    for (int k = 0; k < slots && e == hipSuccess; ++k) {
        if (out.done[k]) continue;
        e = hipHostMalloc(&out.slot[k], PIN_BYTES, hipHostMallocDefault);
        if (e == hipSuccess) e = hipEventCreateWithFlags(&out.done[k], hipEventDisableTiming);
    }
    if (e == hipSuccess) return true;
    free_set(out);
    (void)hipGetLastError();   // not for the next call to report
    std::lock_guard<std::mutex> lk(mu);
    --sets;
    return false;
}

void pinned_return(PinnedSet &s)
{
    std::lock_guard<std::mutex> lk(mu);
    idle[n_idle++] = s;
}

void read_scatter(const ReadPart *parts, int np, int64_t i0, int64_t i1, size_t at, size_t bytes, const void *from)
{
    const int nt = team(bytes);
#pragma omp parallel for num_threads(nt) schedule(static) if (nt > 1)
    for (int t = 0; t < nt; ++t) {
        // this thread's share of the piece, part by part
        size_t lo = at + bytes / 64 * (size_t)t / (size_t)nt * 64;
        const size_t hi = t == nt - 1 ? at + bytes : at + bytes / 64 * (size_t)(t + 1) / (size_t)nt * 64;
        size_t base = 0;
        for (int k = 0; k < np && lo < hi; ++k) {
            if (!parts[k].dst) continue;
            const size_t wide = sizeof(double) * (size_t)parts[k].width, end = base + wide * (size_t)(i1 - i0);
            if (lo < end) {
                const size_t len = std::min(hi, end) - lo;
                std::memcpy((char *)parts[k].dst + wide * (size_t)i0 + (lo - base), (const char *)from + (lo - at), len);
                lo += len;
            }
            base = end;
        }
    }
}

void read_touch(const ReadPart *parts, int np, int64_t items)
{
    for (int k = 0; k < np; ++k) {
        if (!parts[k].dst) continue;
        const size_t bytes = sizeof(double) * (size_t)parts[k].width * (size_t)items;
        const int nt = team(bytes / 4);
        if (nt == 1) continue;
        char *p = (char *)parts[k].dst;
#pragma omp parallel for num_threads(nt) schedule(static)
        for (int t = 0; t < nt; ++t)
            for (size_t o = bytes / (size_t)nt * (size_t)t, end = t == nt - 1 ? bytes : bytes / (size_t)nt * (size_t)(t + 1); o < end;
                 o += 4096) {
                char was = 0;   // zero for zero: a write in any case, of what is there
                __atomic_compare_exchange_n(p + o, &was, (char)0, false, __ATOMIC_RELAXED, __ATOMIC_RELAXED);
            }
    }
}

}  // namespace lbm
