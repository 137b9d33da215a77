// readback.cpp -- host side of the state reads (readback.h).
#include "readback.h"

#include <omp.h>

#include <cstring>
#include <mutex>
#include <vector>

namespace lbm {

namespace {
constexpr size_t PIN_IDLE = 2;
std::mutex mu;
int users = 0;
std::vector<PinnedSet> &idle()
{
    static std::vector<PinnedSet> *v = [] {   // alive at process exit
        auto *p = new std::vector<PinnedSet>;
        p->reserve(PIN_IDLE);
        return p;
    }();
    return *v;
}

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
    if (--users > 0) return;
    for (PinnedSet &s : idle()) free_set(s);
    idle().clear();
}

bool pinned_take(int device, PinnedSet &out)
{
    {
        std::lock_guard<std::mutex> lk(mu);
        for (size_t k = 0; k < idle().size(); ++k)
            if (idle()[k].device == device) {
                out = idle()[k];
                idle().erase(idle().begin() + (ptrdiff_t)k);
                return true;
            }
    }
    out = PinnedSet{};
    out.device = device;
    hipError_t e = hipSuccess;
    for (int k = 0; k < PIN_SLOTS && e == hipSuccess; ++k) {
        e = hipHostMalloc(&out.slot[k], PIN_BYTES, hipHostMallocDefault);
        if (e == hipSuccess) e = hipEventCreateWithFlags(&out.done[k], hipEventDisableTiming);
    }
    if (e == hipSuccess) return true;
    free_set(out);
    (void)hipGetLastError();   // not for the next call to report
    return false;
}

void pinned_return(PinnedSet &s)
{
    {
        std::lock_guard<std::mutex> lk(mu);
        if (idle().size() < PIN_IDLE) {
            idle().push_back(s);
            return;
        }
    }
    free_set(s);
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
