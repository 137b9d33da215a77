// tune.h -- the launch autotuner: times a kernel's candidate launch settings on the handle's own
// geometry and keeps the fastest, with a process-wide cache of the choices.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <vector>

#include "lbm_mi355x.h"

namespace lbm {

// boxes with fewer fluid nodes are not tuned: their launches are too short to time
constexpr int64_t TUNE_MIN_NODES = int64_t(1) << 20;
// Their settings go by size.  Where both buffers fit the eight L2s (32 MB), a slab of tiles for
// each XCD serves a step: a tile is read where the launch before wrote it.  Workgroups of 128 nodes
// fill the CUs of such a box better.  Step, default -> 128-node tiles in slabs: single phase 4,224
// nodes FP64 4.71 -> 4.27 us, 28,800 FP32 4.52 -> 4.08, 117,964 FP32 6.27 -> 5.42, FP16 5.51 -> 5.14
// (398,131 FP32 16.2 -> 15.8, FP64 27.0 -> 26.7, above the line: no gain worth a setting); solute
// 26,214 nodes 3.07 -> 2.75, 209,715 4.22 -> 3.90, with the flow 5.36 -> 4.71 and 12.6 -> 11.6 us
// (707,788: 11.7 -> 11.7 and 31.3 -> 32.5).
constexpr int64_t SP_SLAB_NODES = int64_t(1) << 17, SP_KEEP_SLAB_NODES = int64_t(1) << 18;
constexpr int64_t ST_SLAB_NODES = int64_t(1) << 18;
// Colour gradient, both launches in slabs (one gathers what the other has just written), collide
// and colour gathering below the line, staged above it where most blocks read from their runs.
// Step FP32 / FP64, runs of 8 and gathers -> slabs and gathers | slabs and staged: 55,296 nodes 11.2 /
// 16.2 -> 10.5 / 14.3 | 13.9 / 21.7 us, 131,072 16.4 / 26.8 -> 13.7 / 24.9 | 14.0 / 25.9, 184,320 22.3 /
// 38.4 -> 20.1 / 37.8 | 23.4 / 44.9, 240,000 27.4 / 48.5 -> 26.4 / 48.3 | 24.2 / 47.6, 649,605 56.7 /
// 109.2 -> 57.4 / 110.5 | 50.4 / 99.3, 921,600 77.3 / 153.9 -> 79.1 / 157.4 | 66.2 / 135.1.
constexpr int64_t CG_STAGED_NODES = 215000;
constexpr double CG_STAGED_FAST = 0.85;
constexpr int64_t CG_SMALL_NODES = int64_t(1) << 15;   // 128-node collide tiles: 16,384 nodes 9.8 -> 9.3 us, 55,296 10.5 -> 10.9
// Steps whose arrays fit the 256 MB memory-side cache together store without the nontemporal hint, so
// that the next step finds them there, and from 2^18 nodes on run in slabs, 256 nodes a tile.  Step on
// device, hint -> none -> none and slabs: single phase FP64 256,000 nodes 17.6 -> 15.4 -> 13.4 us,
// 702,464 (227 MB) 41.7 -> 39.7 -> 34.4, 1,048,576 (339 MB) 59.4 -> 63.7; FP32 442,368 16.8 -> 15.2 -> 13.0,
// 1,492,992 (255 MB) 45.7 -> 37.9, 2,048,000 (350 MB) 61.4 -> 69.2; FP16 702,464 18.6 -> 16.9 -> 16.0;
// 815,257 nodes FP32 with faces and power law 30.3 -> 25.0; colour gradient FP32 864,000 (185 MB) 67.4 -> 56.5,
// 1,492,992 (321 MB) 104.2 -> 105.4, FP64 562,432 91.4 -> 80.7; solute FP32 530,841 9.0 -> 8.3 -> 7.3, with the
// flow 25.6 -> 23.7 -> 20.0; sixteen served samples of edges 32 to 88 58.5 -> 49.3 ms a batch.  A solute's
// slabs go by the bytes of the step with its flow, also on its own: FP64 boxes of 588,505 to 1.05 M nodes
// with a frozen velocity store without the hint but keep the hardware's order (788,456 nodes 18.5 us, in
// slabs 17.2).
// The rule counts the step of one handle.  Where several step at once and do not fit together, the hint
// would be the better choice: FP64 501,992 nodes (162 MB) in two threads 25.9 us a step, with the hint
// 29.0, in four 28.7 and 28.7, in eight 30.3 and 28.5; FP32 1,102,614 nodes (189 MB) 30.7 and 31.7, 33.0 and
// 30.7, 34.8 and 31.2.
constexpr int64_t CACHE_BYTES = 256000000;
inline bool fits_cache(int64_t step_bytes) { return step_bytes <= CACHE_BYTES; }
// Values of 2 and 4 bytes keep the hint where a buffer has 4.5 to 12 MB, in most of which the flow step
// was slower without it: FP32 131,072 nodes 6.73 -> 7.04 us, 186,624 (14 MB) 8.99 -> 8.19; FP16 131,072 5.6 ->
// 5.9, 256,000 8.0 -> 8.4, 340,736 (13 MB) 10.6 -> 10.3; but FP64 70,304 (11 MB) 5.9 -> 5.65.  Not in all of it: in
// 128-node tiles, FP32 72,565 nodes 4.47 -> 4.22 and 122,507 5.58 -> 5.16, FP16 122,507 4.70 -> 4.55.  The
// colour gradient, FP32: 72,565 nodes 12.5 -> 12.5, 95,375 12.6 -> 12.7, 122,507 12.8 -> 13.3, 137,837 17.3 -> 16.2.
inline bool keep_stores(int64_t step_bytes, int64_t buffer_bytes, size_t width)
{
    return fits_cache(step_bytes) && (width > 4 || buffer_bytes < 4500000 || buffer_bytes > 12000000);
}
// Where they do not fit, from this size on, launches into one of the two buffers run through the tiles
// from the last to the first, so that a step begins with what the one before has written last, some of
// it still in that cache; a colour launch runs against its collide launch.  Step on device: 171 x 203 x
// 187 FP64 105.4 -> 103.6 us, 256^3 sphere pack FP32 167.1 -> 166.2 us, 192^3 fibres with solute FP32
// 213.0 -> 212.1 us, colour gradient 192^3 FP32 209.8 -> 207.4 us and FP64 443.3 -> 437.3 us (colour launch
// with its collide launch: 209.3 and 441.2 us).
constexpr int64_t BACK_NODES = int64_t(1) << 20;
// an alternative replaces the default only when it is faster by this fraction
constexpr double TUNE_MARGIN = 0.01;

// what a flow step reads and writes: populations (19 rows of st bytes, twice), links, a solute's rows
inline int64_t sp_step_bytes(int64_t P, size_t st, size_t solute) { return P * (int64_t)(2 * 19 * st + solute + 19); }

// What a choice is kept under: the kernel, the precision, the size class (two an octave) and all else
// that decides which form of the kernel a launch runs and in which direction.  Both lines of the cache
// fall inside a size class, and an FP16 and an FP32 flow carry the same FP32 solute.
struct TuneKey {
    int kernel, precision;
    int64_t nodes;
    bool fits;               // the step fits the memory-side cache
    bool narrow = false;     // 8-bit ranks
    size_t flow_width = 0;   // coupled solute: bytes of a stored flow value,
    bool flow_fits = false;  // and whether the flow's own step fits
};
// cached choice; false if none
bool tune_cache_get(const TuneKey &key, lbm_launch &out);
void tune_cache_put(const TuneKey &key, const lbm_launch &ls);

// The fastest of `cands` (cands[0] is the default): each candidate is launched `warm` times,
// then timed as the median of `rounds` rounds of `reps` launches between HIP events on s.
// launch(ls) queues one launch and returns its status.  On an error the default is returned
// with its status.  out.tuned = 1 and out.time_us = the median time of one launch.
template <typename F>
hipError_t tune_launch(hipStream_t s, const std::vector<lbm_launch> &cands, F &&launch, lbm_launch &out, int warm = 2,
                       int reps = 5, int rounds = 3)
{
    hipEvent_t e0 = nullptr, e1 = nullptr;
    hipError_t e = hipEventCreate(&e0);
    if (e == hipSuccess) e = hipEventCreate(&e1);
    std::vector<double> t(cands.size(), 0.0);
    for (size_t c = 0; c < cands.size() && e == hipSuccess; ++c) {
        for (int w = 0; w < warm && e == hipSuccess; ++w) e = launch(cands[c]);
        std::vector<double> r;
        for (int k = 0; k < rounds && e == hipSuccess; ++k) {
            e = hipEventRecord(e0, s);
            for (int i = 0; i < reps && e == hipSuccess; ++i) e = launch(cands[c]);
            if (e == hipSuccess) e = hipEventRecord(e1, s);
            if (e == hipSuccess) e = hipEventSynchronize(e1);
            float ms = 0.f;
            if (e == hipSuccess) e = hipEventElapsedTime(&ms, e0, e1);
            r.push_back(1e3 * (double)ms / reps);
        }
        if (e == hipSuccess) {
            std::sort(r.begin(), r.end());
            t[c] = r[r.size() / 2];
        }
    }
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    out = cands[0];
    if (e != hipSuccess) return e;
    size_t best = 0;
    for (size_t c = 1; c < cands.size(); ++c)
        if (t[c] < t[best] * (best == 0 ? 1.0 - TUNE_MARGIN : 1.0)) best = c;
    out = cands[best];
    out.tuned = 1;
    out.time_us = t[best];
    return hipSuccess;
}

// the candidates of a kernel: block sizes x tile orders (x variants), the default first
std::vector<lbm_launch> tune_candidates(const lbm_launch &def, const std::vector<int> &blocks,
                                        const std::vector<int> &orders, const std::vector<int> &variants);

// argument checks shared by the handles' set_launch
bool launch_valid(const lbm_launch &ls, const std::vector<int> &blocks, const std::vector<int> &variants);

}  // namespace lbm
