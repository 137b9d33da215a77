// sanitize_links.cpp -- the packed link tables (pack_neighbours) in both widths under the sanitizers.
//
//   sanitize_links pack                 random boxes: every table is decoded back by the packing itself, and
//                                       the width is what the share of waves in full words says
//   sanitize_links width nx ny nz FILE  the bits of a rank in the flow solver's table of the box in FILE (int32)
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <fstream>
#include <random>
#include <string>
#include <vector>

#include "handle.h"
#include "lattice.h"

using namespace lbm;

namespace {
int failures = 0, narrow = 0, narrow_with_full = 0, broad = 0;

void check(int nx, int ny, int nz, double porosity, std::mt19937 &rng)
{
    std::uniform_real_distribution<double> u(0.0, 1.0);
    std::vector<int32_t> solid((size_t)nx * ny * nz);
    for (auto &v : solid) v = u(rng) < porosity ? 0 : 1;
    solid[solid.size() / 2] = 0;
    SparseGeometry g;
    std::string err;
    bool ok = build_sparse_geometry(nx, ny, nz, solid.data(), g, err) == LBM_OK;
    const int64_t W = g.P / 64;
    PackedNbr a, b;
    ok = ok && pack_neighbours(g, a, err) == LBM_OK && pack_neighbours(g, b, err, true) == LBM_OK;
    ok = ok && !a.narrow && a.res.size() == (size_t)(NCOL * g.P) && a.res8.empty();
    // a rank less the node's id spreads over less than 256 in all but the waves in full words
    for (int64_t w = 0; ok && w < W; ++w) {
        const int64_t n0 = w * 64, n1 = std::min(n0 + 64, g.N);
        bool spread = false;
        for (int q = 1; q < Q; ++q) {
            if (EZ[q] != 0) continue;   // of a column, its link at the node's height: a spread that is there
            int64_t lo = INT64_MAX, hi = INT64_MIN;
            for (int64_t n = n0; n < n1; ++n) {
                const uint32_t v = g.nbr[(size_t)((q - 1) * g.P + n)];
                if (v & BB_FLAG) continue;
                lo = std::min(lo, (int64_t)v - n);
                hi = std::max(hi, (int64_t)v - n);
            }
            spread |= hi >= lo && hi - lo > 255;
        }
        const bool full = b.hdr[(size_t)(w * HDR_WORDS + HDR_WIDE)] != HDR_COMPACT;
        if (b.narrow && spread && !full) ok = false;
    }
    if (b.narrow) ok = ok && b.res8.size() == (size_t)(NCOL * g.P) && b.res.empty() && b.wide.size() / (18 * 64) <= (size_t)(W / NARROW_WIDE);
    else ok = ok && b.res == a.res && b.hdr == a.hdr && b.edge == a.edge && b.wide == a.wide;
    broad += !b.narrow;
    narrow += b.narrow;
    narrow_with_full += b.narrow && !b.wide.empty();
    if (!ok) {
        std::fprintf(stderr, "FAIL links of %dx%dx%d, porosity %g %s\n", nx, ny, nz, porosity, err.c_str());
        ++failures;
    }
}
}  // namespace

int main(int argc, char **argv)
{
    if (argc == 6 && !std::strcmp(argv[1], "width")) {
        const int nx = std::atoi(argv[2]), ny = std::atoi(argv[3]), nz = std::atoi(argv[4]);
        std::vector<int32_t> solid((size_t)nx * ny * nz);
        std::ifstream(argv[5], std::ios::binary).read((char *)solid.data(), (std::streamsize)(solid.size() * 4));
        SparseGeometry g;
        PackedNbr p;
        std::string err;
        if (build_sparse_geometry(nx, ny, nz, solid.data(), g, err) != LBM_OK ||
            pack_neighbours(g, p, err, g.N >= NARROW_NODES) != LBM_OK)
            return 1;
        std::printf("%d bits\n", p.narrow ? 8 : 16);
        return 0;
    }
    std::mt19937 rng(20261205u);
    const int sizes[][3] = {{1, 1, 1}, {1, 1, 300}, {1, 300, 1}, {300, 1, 1}, {2, 2, 2}, {5, 4, 3}, {17, 13, 11}, {3, 40, 2}, {70, 3, 3},
                            {40, 30, 40}, {12, 60, 70}, {60, 6, 90}, {4, 200, 150}};
    for (const auto &s : sizes)
        for (double por : {0.02, 0.4, 0.9, 1.0}) check(s[0], s[1], s[2], por, rng);
    std::printf("%d boxes in 16 bits, %d in 8, %d of them with waves in full words\n", broad, narrow, narrow_with_full);
    if (failures || !broad || !narrow || !narrow_with_full) return 1;
    std::printf("sanitized checks passed\n");
    return 0;
}
