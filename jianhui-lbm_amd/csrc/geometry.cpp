// geometry.cpp -- fluid-node numbering and pull neighbour lists (host).
//
// Follows the reference's sparse structure: pore voxels are numbered in i-major order, x
// slowest and z fastest (SP:1172-1193), and SupInv holds each node's linear voxel index
// (SP:1261-1277).  Where the reference pushes post-collision populations to the downstream
// node and bounces back in place when that node is solid (SP:1874-1926), the device kernels
// pull: population q of node x comes from x - e_q, or from the opposite population of x
// itself when x - e_q is solid.  Both give the same post-streaming state.
#include <algorithm>
#include <cstring>

#include "connectivity.h"
#include "handle.h"
#include "lattice.h"

namespace lbm {

int build_sparse_geometry(int nx, int ny, int nz, const int32_t *solid, SparseGeometry &g, std::string &err)
{
    if (nx <= 0 || ny <= 0 || nz <= 0 || !solid) {
        err = "invalid box size or null geometry";
        return LBM_ERR_ARG;
    }
    const int64_t nvox = (int64_t)nx * ny * nz;
    if (nvox >= ((int64_t)1 << 31)) {
        err = "box has 2^31 or more voxels";
        return LBM_ERR_ARG;
    }
    std::vector<int32_t> idx((size_t)nvox, -1);
    int64_t N = 0;
    for (int64_t v = 0; v < nvox; ++v)
        if (solid[v] == 0) idx[(size_t)v] = (int32_t)N++;
    if (N == 0) {
        err = "geometry has no pore voxels";
        return LBM_ERR_ARG;
    }
    // node indices fit in 31 bits (bit 31 is the bounce-back flag) because nvox < 2^31;
    // element offsets q*P + node are formed in 64-bit arithmetic on the device
    const int64_t P = padded_stride(N);
    g.nx = nx;
    g.ny = ny;
    g.nz = nz;
    g.N = N;
    g.P = P;
    g.supinv.assign((size_t)N, 0);
    g.nbr.assign((size_t)(18 * P), 0u);
    for (int64_t v = 0; v < nvox; ++v)
        if (idx[(size_t)v] >= 0) g.supinv[(size_t)idx[(size_t)v]] = (int32_t)v;

    const int64_t nyz = (int64_t)ny * nz;
#pragma omp parallel for schedule(static)
    for (int64_t n = 0; n < N; ++n) {
        const int64_t s = g.supinv[(size_t)n];
        const int i = (int)(s / nyz), j = (int)((s % nyz) / nz), k = (int)(s % nz);
        for (int q = 1; q < Q; ++q) {
            int iu = i - EX[q], ju = j - EY[q], ku = k - EZ[q];
            iu = iu < 0 ? iu + nx : (iu >= nx ? iu - nx : iu);
            ju = ju < 0 ? ju + ny : (ju >= ny ? ju - ny : ju);
            ku = ku < 0 ? ku + nz : (ku >= nz ? ku - nz : ku);
            const int32_t up = idx[(size_t)(((int64_t)iu * ny + ju) * nz + ku)];
            g.nbr[(size_t)((q - 1) * P + n)] = up >= 0 ? (uint32_t)up : ((uint32_t)n | BB_FLAG);
        }
    }
    return LBM_OK;
}

void reference_rank_ends(const SparseGeometry &g, int nranks, std::vector<int64_t> &ends)
{
    // pore count of each x-plane, and the node id where each plane starts
    const int64_t nyz = (int64_t)g.ny * g.nz;
    std::vector<int64_t> loc_por((size_t)g.nx, 0), first((size_t)g.nx + 1, 0);
    for (int64_t n = 0; n < g.N; ++n) ++loc_por[(size_t)(g.supinv[(size_t)n] / nyz)];
    for (int i = 0; i < g.nx; ++i) first[(size_t)i + 1] = first[(size_t)i] + loc_por[(size_t)i];
    // cut r + 1 where the running plane sum first reaches ave * (r + 1): before or after the plane
    // that crosses it, whichever sum is closer (SP:1089-1102); the last rank keeps the rest
    const double ave = (double)g.N / nranks;
    ends.assign((size_t)nranks, g.N);
    for (int r = 0; r < nranks - 1; ++r) {
        int64_t pre = 0, aft = 0;
        int n_i = 0;
        while (aft < ave * (r + 1) && n_i < g.nx) {
            pre = aft;
            aft += loc_por[(size_t)n_i];
            ++n_i;
        }
        const int disp = ((double)(aft - ave * (r + 1)) > (double)(ave * (r + 1) - pre)) ? n_i - 1 : n_i;
        ends[(size_t)r] = first[(size_t)disp];
    }
}

bool pores_wrap_along(const SparseGeometry &g, int axis)
{
    const int64_t P = g.P;
    return lattice_loop_wraps(g.N, axis, [&g, P](int64_t n, int q) -> int64_t {
        const uint32_t v = g.nbr[(size_t)((q - 1) * P + n)];
        return (v & BB_FLAG) ? -1 : (int64_t)v;
    });
}

namespace {

// link_column, column_link and edge_slot (lattice.h) as tables
struct ColumnTables {
    int column[Q] = {}, slot[Q] = {}, at[NCOL + 1] = {}, below[NCOL + 1] = {}, above[NCOL + 1] = {};
    constexpr ColumnTables()
    {
        for (int q = 1; q < Q; ++q) {
            column[q] = link_column(q);
            slot[q] = edge_slot(q);
        }
        for (int c = 0; c <= NCOL; ++c) {
            at[c] = column_link(c, 0);
            below[c] = column_link(c, 1);
            above[c] = column_link(c, -1);
        }
    }
};
constexpr ColumnTables COL;

// Whether the packed form of node n's links, as load_links decodes it, is not what link(q) gives.
template <typename F>
bool unpacks_wrong(const PackedNbr &p, int64_t P, int64_t n, F &&link)
{
    const uint32_t *h = &p.hdr[(size_t)((n >> 6) * HDR_WORDS)];
    const int lane = (int)(n & 63);
    auto lane_in = [h, lane](int at) { return (h[at + (lane >> 5)] >> (lane & 31) & 1u) != 0; };
    const bool wide = h[HDR_WIDE] != HDR_COMPACT, is_edge = !wide && lane_in(HDR_EDGE);
    const uint64_t edge = (uint64_t)h[HDR_EDGE] | (uint64_t)h[HDR_EDGE + 1] << 32;
    const int64_t rec = is_edge ? (int64_t)h[HDR_EDGE_BASE] + __builtin_popcountll(edge & ((1ull << lane) - 1)) : 0;
    uint32_t rank[NCOL];
    for (int c = 0; c < NCOL && !wide; ++c) {
        const size_t at = (size_t)(((c / 4) * P + n) * 4 + c % 4);
        rank[c] = p.narrow ? h[c] + (uint32_t)n + p.res8[at] : h[c] + p.res[at];
    }
    bool wrong = false;
    for (int q = 1; q < Q; ++q) {
        const int c = COL.column[q];
        const bool solid = lane_in(HDR_MASK + 2 * (q - 1));
        uint32_t up;
        if (wide) up = p.wide[(size_t)(((int64_t)h[HDR_WIDE] * 18 + q - 1) * 64 + lane)];
        else if (EZ[q] != 0 && is_edge) up = p.edge[(size_t)(rec * EDGE_WORDS + COL.slot[q])];
        else if (c == NCOL) up = (uint32_t)(n - EZ[q]);
        else if (EZ[q] == 0) up = rank[c];
        else up = EZ[q] > 0 ? rank[c] - 1 : rank[c] + !lane_in(HDR_MASK + 2 * (COL.at[c] - 1));
        wrong |= (solid ? (uint32_t)n | BB_FLAG : up) != link(q);   // selected last: no branch on what is close to random
    }
    return wrong;
}

}  // namespace

int pack_neighbours(const SparseGeometry &g, PackedNbr &out, std::string &err, bool narrow_ok)
{
    const int64_t P = g.P, N = g.N, W = P / 64;
    // the 8-bit form, worked out only where the caller may take it
    std::vector<uint32_t> base8((size_t)(narrow_ok ? W * NCOL : 0), 0u);
    std::vector<uint8_t> wide8((size_t)(narrow_ok ? W : 0), 0u);
    out.hdr.assign((size_t)(W * HDR_WORDS), 0u);
    auto link = [&g, P](int64_t n, int q) { return g.nbr[(size_t)((q - 1) * P + n)]; };
    auto none = [](uint32_t v) { return (v & BB_FLAG) != 0; };
    // the upstream sites of column c around the node: at its height, one below, one above (an xy
    // diagonal has the first only, the node's own column the other two)
    auto column = [&](int64_t n, int c, uint32_t &at, uint32_t &below, uint32_t &above) {
        at = COL.at[c] ? link(n, COL.at[c]) : (uint32_t)n;
        below = COL.below[c] ? link(n, COL.below[c]) : BB_FLAG;
        above = COL.above[c] ? link(n, COL.above[c]) : BB_FLAG;
    };
    // per node and column the rank (the number of pore voxels before the site at the node's
    // height), from which the three sites' ids follow unless the column wraps round in z there
    auto rank = [&](uint32_t at, uint32_t below, uint32_t above) {
        return !none(at) ? at : !none(below) ? below + 1 : above;
    };
#pragma omp parallel for schedule(static)
    for (int64_t w = 0; w < W; ++w) {
        const int64_t n0 = w * 64, n1 = std::min(n0 + 64, N);
        uint32_t *h = &out.hdr[(size_t)(w * HDR_WORDS)];
        auto set = [h](int at, uint64_t lanes) {
            h[at] |= (uint32_t)lanes;
            h[at + 1] |= (uint32_t)(lanes >> 32);
        };
        bool wide = false;
        for (int c = 0; c <= NCOL; ++c) {
            uint32_t lo = 0xFFFFFFFFu, hi = 0, at, below, above;
            int64_t lo8 = INT64_MAX, hi8 = INT64_MIN;   // of the rank less the node's own id
            uint64_t no_at = 0, no_below = 0, no_above = 0, edge = 0;
            // without branches: which sites are solid is close to random
            for (int64_t n = n0; n < n1; ++n) {
                column(n, c, at, below, above);
                const uint64_t na = none(at), nb = none(below), nv = none(above);
                const int lane = (int)(n - n0);
                no_at |= na << lane;
                no_below |= nb << lane;
                no_above |= nv << lane;
                const uint32_t r = rank(at, below, above);
                const bool any = !(na & nb & nv);
                const bool jumps = (!nb & (below != r - 1)) | (!nv & (above != r + !na));
                edge |= (uint64_t)(any & jumps) << lane;
                lo = std::min(lo, any ? r : lo);
                hi = std::max(hi, any ? r : hi);
                if (narrow_ok) {
                    lo8 = std::min(lo8, any ? (int64_t)r - n : lo8);
                    hi8 = std::max(hi8, any ? (int64_t)r - n : hi8);
                }
            }
            if (COL.at[c]) set(HDR_MASK + 2 * (COL.at[c] - 1), no_at);
            if (COL.below[c]) set(HDR_MASK + 2 * (COL.below[c] - 1), no_below);
            if (COL.above[c]) set(HDR_MASK + 2 * (COL.above[c] - 1), no_above);
            set(HDR_EDGE, edge);
            if (c == NCOL || lo == 0xFFFFFFFFu) continue;   // the own column needs no ranks
            h[c] = lo;
            wide |= hi - lo > 0xFFFFu;
            if (!narrow_ok) continue;
            base8[(size_t)(w * NCOL + c)] = (uint32_t)lo8;
            wide8[(size_t)w] |= hi8 - lo8 > 0xFF;
        }
        h[HDR_WIDE] = wide ? 0u : HDR_COMPACT;
        // lanes past the last node: solid all round, so that following their links stays in place
        for (int64_t n = std::max(n0, n1); n < n0 + 64; ++n)
            for (int q = 1; q < Q; ++q) set(HDR_MASK + 2 * (q - 1), 1ull << (n - n0));
    }
    int64_t n_wide8 = 0;
    for (uint8_t v : wide8) n_wide8 += v;
    out.narrow = narrow_ok && n_wide8 <= W / NARROW_WIDE;
    out.res.assign(out.narrow ? 0 : (size_t)(NCOL * P), 0u);
    out.res8.assign(out.narrow ? (size_t)(NCOL * P) : 0, 0u);
    int64_t nw = 0, ne = 0;
    for (int64_t w = 0; w < W; ++w) {
        uint32_t *h = &out.hdr[(size_t)(w * HDR_WORDS)];
        if (out.narrow) {
            std::copy_n(&base8[(size_t)(w * NCOL)], NCOL, h);
            h[HDR_WIDE] = wide8[(size_t)w] ? 0u : HDR_COMPACT;
        }
        if (h[HDR_WIDE] != HDR_COMPACT) {
            h[HDR_WIDE] = (uint32_t)nw++;
            continue;
        }
        h[HDR_EDGE_BASE] = (uint32_t)ne;
        ne += __builtin_popcount(h[HDR_EDGE]) + __builtin_popcount(h[HDR_EDGE + 1]);
    }
    out.wide.assign((size_t)(nw * 18 * 64), 0u);
    out.edge.assign((size_t)(ne * EDGE_WORDS), 0u);
#pragma omp parallel for schedule(static)
    for (int64_t w = 0; w < W; ++w) {
        const int64_t n0 = w * 64, n1 = std::min(n0 + 64, N);
        const uint32_t *h = &out.hdr[(size_t)(w * HDR_WORDS)];
        if (h[HDR_WIDE] != HDR_COMPACT) {
            for (int q = 1; q < Q; ++q)
                for (int64_t n = n0; n < n1; ++n)
                    out.wide[(size_t)(((int64_t)h[HDR_WIDE] * 18 + q - 1) * 64 + (n - n0))] = link(n, q) & ~BB_FLAG;
            continue;
        }
        uint32_t rec = h[HDR_EDGE_BASE];
        for (int64_t n = n0; n < n1; ++n) {
            for (int c = 0; c < NCOL; ++c) {
                uint32_t at, below, above;
                column(n, c, at, below, above);
                if (none(at) && none(below) && none(above)) continue;
                const size_t i = (size_t)(((c / 4) * P + n) * 4 + c % 4);
                const uint32_t r = rank(at, below, above) - h[c];
                if (out.narrow) out.res8[i] = (uint8_t)(r - (uint32_t)n);
                else out.res[i] = (uint16_t)r;
            }
            if (h[HDR_EDGE + ((n - n0) >> 5)] >> ((n - n0) & 31) & 1) {
                for (int q = 1; q < Q; ++q)
                    if (EZ[q] != 0) out.edge[(size_t)((int64_t)rec * EDGE_WORDS + COL.slot[q])] = link(n, q) & ~BB_FLAG;
                ++rec;
            }
        }
    }
    // decode everything as the device does and compare
    int64_t bad = 0;
#pragma omp parallel for schedule(static) reduction(+ : bad)
    for (int64_t n = 0; n < N; ++n) bad += unpacks_wrong(out, P, n, [&](int q) { return link(n, q); });
    if (bad) {
        err = "neighbour table packing failed its decode check (" + std::to_string(bad) + " nodes)";
        return LBM_ERR_STATE;
    }
    return LBM_OK;
}

hipError_t DeviceNbr::upload(const PackedNbr &p, hipStream_t s)
{
    release();
    const void *from[4] = {p.narrow ? (const void *)p.res8.data() : (const void *)p.res.data(), p.hdr.data(), p.edge.data(),
                           p.wide.data()};
    const size_t bytes[4] = {p.narrow ? p.res8.size() : p.res.size() * sizeof(uint16_t), p.hdr.size() * sizeof(uint32_t),
                             p.edge.size() * sizeof(uint32_t), p.wide.size() * sizeof(uint32_t)};
    size_t at[5] = {0};
    for (int k = 0; k < 4; ++k) at[k + 1] = at[k] + (bytes[k] + 255) / 256 * 256;
    hipError_t e;
    if ((e = hipMalloc(&res, at[4])) != hipSuccess) return e;
    char *d = (char *)res;
    hdr = (uint32_t *)(d + at[1]);
    edge = (uint4 *)(d + at[2]);
    wide = (uint32_t *)(d + at[3]);
    narrow = p.narrow;
    for (int k = 0; k < 4; ++k)
        if (bytes[k] && (e = hipMemcpyAsync(d + at[k], from[k], bytes[k], hipMemcpyHostToDevice, s)) != hipSuccess) return e;
    return hipSuccess;
}

void DeviceNbr::release()
{
    if (res) (void)hipFree(res), res = nullptr;
    hdr = wide = nullptr;
    edge = nullptr;
}

}  // namespace lbm
