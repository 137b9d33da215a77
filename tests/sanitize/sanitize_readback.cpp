// sanitize_readback.cpp -- the state reads (readback.h) under the sanitizers, on a stand-in for the device
// runtime: "device" memory is host memory, copies are made at once, and page-locked allocations and copies
// can be made to fail.  Arguments name the check.
#include <algorithm>
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <string>
#include <thread>
#include <vector>

#include "readback.h"

namespace {
std::atomic<int> live{0}, made{0};        // page-locked slots: alive, ever made
std::atomic<int> made_at_most{1 << 30};   // allocations that succeed
std::atomic<int> copies_at_most{1 << 30};
std::atomic<int> pending{0};   // as the runtime keeps the last error
hipError_t failed(hipError_t e) { return pending = (int)e, e; }
}  // namespace

extern "C" {
hipError_t hipHostMalloc(void **p, size_t n, unsigned int)
{
    if (made >= made_at_most) return failed(hipErrorOutOfMemory);
    *p = std::malloc(n);
    ++live, ++made;
    return hipSuccess;
}
hipError_t hipHostFree(void *p) { return std::free(p), --live, hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return *e = (hipEvent_t)std::malloc(1), hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { return std::free(e), hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError() { return (hipError_t)pending.exchange(0); }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t)
{
    if (copies_at_most-- <= 0) return failed(hipErrorUnknown);
    return std::memcpy(d, s, n), hipSuccess;
}
}

using namespace lbm;

namespace {
constexpr size_t BUF = size_t(16) << 20;
int failures = 0;
void expect(bool ok, const char *what)
{
    if (!ok) std::fprintf(stderr, "FAIL %s\n", what), ++failures;
}

double value(int part, int64_t at) { return 1.0 + part + 1e-3 * (double)at; }

struct Reader {
    PinnedUser user;
    std::vector<char> buf = std::vector<char>(BUF);
    int64_t n;
    std::vector<double> f, u;
    explicit Reader(int64_t items) : n(items), f((size_t)items * 19, -1.0), u((size_t)items * 3, -2.0) {}
    template <typename G>
    hipError_t read(G &&meanwhile)
    {
        const ReadPart parts[3] = {{f.data(), 19}, {nullptr, 5}, {u.data(), 3}};
        return read_back(0, nullptr, n, parts, 3, buf.data(), BUF, 256, [&](int64_t i0, int64_t i1, double *const *p) {
            meanwhile();
            for (int64_t i = i0 * 19; i < i1 * 19; ++i) p[0][i - i0 * 19] = value(0, i);
            for (int64_t i = i0 * 3; i < i1 * 3; ++i) p[2][i - i0 * 3] = value(2, i);
            return hipGetLastError();   // as the kernels' launches report
        });
    }
    // items whose values are neither those that are read nor those from before
    int64_t wrong(bool read) const
    {
        int64_t bad = 0;
        for (int64_t i = 0; i < n * 19; ++i) bad += f[(size_t)i] != value(0, i) && (read || f[(size_t)i] != -1.0);
        for (int64_t i = 0; i < n * 3; ++i) bad += u[(size_t)i] != value(2, i) && (read || u[(size_t)i] != -2.0);
        return bad;
    }
};

// the slots that a read of n items fills
int slots_of(int64_t n) { return (int)std::min<int64_t>(PIN_SLOTS, (n * 22 * 8 + (int64_t)PIN_BYTES - 1) / (int64_t)PIN_BYTES); }

// one piece, several pieces, several chunks with a remainder
const int64_t SIZES[] = {1, 255, 4224, 40329, 157286};

// no page-locked memory, or not all of a set: the values all the same, and no error left behind
void refused()
{
    for (int slots : {0, 2})
        for (int64_t n : SIZES) {
            made = 0;
            made_at_most = slots;
            Reader r(n);
            expect(r.read([] {}) == hipSuccess && r.wrong(true) == 0, "read without page-locked memory");
            const int used = slots_of(n);
            expect(live == (used <= slots ? used : 0) && pending == 0, "nothing left of a refused set");
        }
    made_at_most = 1 << 30;
    for (int64_t n : SIZES) {
        Reader r(n);
        expect(r.read([] {}) == hipSuccess && r.wrong(true) == 0 && live == slots_of(n), "read through the slots");
    }
    expect(live == 0, "slots given back");
}

// a copy that fails: its error, and of every array what was read so far and else what was there before
void failing()
{
    for (int good : {0, 3, 5, 9})
        for (int64_t n : {int64_t(40329), int64_t(157286)}) {
            const int64_t copies = (n * 22 * 8 + (int64_t)PIN_BYTES - 1) / (int64_t)PIN_BYTES;
            copies_at_most = good;
            Reader r(n);
            const hipError_t e = r.read([] {});
            expect(good >= copies + 1 || e == hipErrorUnknown, "a failed copy is reported");
            expect(r.wrong(false) == 0, "arrays of a failed read");
            pending = 0;
        }
    copies_at_most = 1 << 30;
}

// handles that read at once, all of them in the middle of a read together: their slots are made once, for
// as many as may be at a time, the others read without; given back as the handles go
void at_once()
{
    for (int count : {2, 5, 20}) {
        made = 0;
        std::vector<std::unique_ptr<Reader>> readers;
        for (int k = 0; k < count; ++k) readers.emplace_back(new Reader(4224));
        for (int round = 0; round < 3; ++round) {
            std::atomic<int> here{0};
            std::vector<std::thread> threads;
            std::atomic<int> bad{0};
            for (auto &r : readers)
                threads.emplace_back([&, r = r.get()] {
                    std::fill(r->f.begin(), r->f.end(), -1.0);
                    const hipError_t e = r->read([&] {
                        ++here;
                        while (here < count) std::this_thread::yield();
                    });
                    bad += e != hipSuccess || r->wrong(true) != 0;
                });
            for (auto &t : threads) t.join();
            expect(bad == 0, "reads at once");
        }
        const int each = slots_of(4224), want = std::min(count, PIN_SETS) * each;
        expect(made == want && live == want, "slots made once");
        readers.resize(1);
        expect(live == each, "slots given back as handles go");
        readers.clear();
        expect(live == 0, "slots given back");
    }
    // a set that grows with the reads, and is kept at its largest
    made = 0;
    Reader small(255), large(157286);
    for (int k = 0; k < 3; ++k)
        for (Reader *r : {&small, &large}) {
            std::fill(r->f.begin(), r->f.end(), -1.0);
            expect(r->read([] {}) == hipSuccess && r->wrong(true) == 0, "reads in turn");
        }
    expect(made == PIN_SLOTS && live == PIN_SLOTS, "one set for reads in turn");
}
}  // namespace

int main(int, char **argv)
{
    const std::string what = argv[1];
    if (what == "refused") refused();
    else if (what == "failing") failing();
    else if (what == "at_once") at_once();
    else return 2;
    if (failures) return 1;
    std::printf("sanitized checks passed\n");
    return 0;
}
