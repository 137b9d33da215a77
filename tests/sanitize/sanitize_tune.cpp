// sanitize_tune.cpp -- the autotuner's cache (tune.h) under the sanitizers: a choice is found again by the
// box it was made for and by others of its size class, and by no box whose launches run another form of
// the kernel.
#include <cstdio>

#include "tune.h"

using namespace lbm;

int main()
{
    int failures = 0;
    auto expect = [&](bool ok, const char *what) {
        if (!ok) std::fprintf(stderr, "FAIL %s\n", what), ++failures;
    };
    lbm_launch set{}, got{};
    set.block = 512;
    set.order = LBM_ORDER_SLAB;
    // FP16 boxes of one size class on both sides of the memory-side cache's line
    const int64_t in = 2600000, out = 2800000;
    const bool fits_in = fits_cache(sp_step_bytes(in, 2, 0)), fits_out = fits_cache(sp_step_bytes(out, 2, 0));
    expect(fits_in && !fits_out, "the line lies between the boxes");
    const TuneKey small{LBM_KERNEL_SP_STEP, LBM_FP16, in, fits_in, true}, large{LBM_KERNEL_SP_STEP, LBM_FP16, out, fits_out, true};
    tune_cache_put(small, set);
    expect(tune_cache_get(small, got) && got.block == 512 && got.order == LBM_ORDER_SLAB, "found again");
    TuneKey near = small;
    near.nodes = in - 1000;
    expect(tune_cache_get(near, got), "found by the size class");
    expect(!tune_cache_get(large, got), "not found by a box that does not fit the cache");
    TuneKey wide = small;
    wide.narrow = false;
    expect(!tune_cache_get(wide, got), "not found by a box of 16-bit ranks");
    // an FP32 solute in an FP16 and in an FP32 flow
    const TuneKey half{-LBM_KERNEL_ST_STEP, LBM_FP32, in, false, true, 2, true};
    TuneKey whole = half;
    whole.flow_width = 4;
    tune_cache_put(half, set);
    expect(tune_cache_get(half, got) && !tune_cache_get(whole, got), "flows of another storage type kept apart");
    if (failures) return 1;
    std::printf("sanitized checks passed\n");
    return 0;
}
