// nbrpack.h -- the device form of the pull neighbour lists: 16-bit or 8-bit ranks per neighbour
// column and per-wave solid masks.
//
// The host builds the full table (18 x P uint32 upstream indices, BB_FLAG for bounce-back),
// which would be 72 of the 224 bytes an FP32 node update moves.  Nodes are numbered along z
// first, so of one column of voxels a node needs a single number, its rank there: the count of
// pore voxels before the site at the node's height.  The site at the height is that node if it
// is a pore, the one below is rank - 1, the one above rank + 1 (rank, if the site between is
// solid).  The 18 upstream sites lie in the node's own column and eight others.  Per wavefront
// (64 consecutive node ids):
//
//   hdr[w][0..7]   uint32  base of each column: the smallest rank of the wave (16-bit), or the
//                          smallest rank less the node's own id (8-bit)
//   hdr[w][8..43]  uint64  per direction, the lanes whose upstream site is solid
//   hdr[w][44..]   uint64  the edge lanes, and the index of their first record
//   res[c / 4][n]  4 x uint16 or 4 x uint8  rank (less the node's id) - base of columns 0-3 (axis)
//                          and 4-7 (xy diagonals)
//   edge[]         the ten upstream nodes with e_z != 0 of an edge lane: one whose column wraps
//                  round in z, where the neighbours in height are not neighbours in rank
//
// and only a wave whose numbers spread over more than their bits in some column keeps its 18 x 64
// full words in a side table, named by hdr[w][47].  With 16 bits these straddle the periodic wrap of
// a large box; with 8 bits also those that cross from one plane of nodes to the next, where the y
// neighbours' ids jump by a plane (0.6 to 1.8 % of the waves of 192^3 to 384^3 boxes).  Elsewhere
// ranks and ids advance together.  A node update reads 16 or 8 bytes of ranks, 3 of header and
// 48 / (nz / 2) of edge records, in three to six loads.  The step is bound by memory, so the bytes
// are its time.  Step on device with 37.25 bytes in 18 loads (a 16-bit residual per direction) ->
// 16-bit ranks: 256^3 sphere pack (5.87 M nodes) FP32 207.7 -> 188.1 us; 171 x 203 x 187 field
// (1.95 M) FP64 122.6 -> 116.9 us; 192^3 fibres with solute (5.66 M) FP32 254.7 -> 242.4 us; colour
// gradient 192^3 (3.19 M) FP32 233.5 -> 225.2 us.  16-bit -> 8-bit: 174.5 -> 171.2, 109.3 -> 107.6,
// 221.0 -> 215.9 us and 208 x 224 x 240 FP16 73.6 -> 72.6 us.
//
// The flow solver's tables are narrow from NARROW_NODES nodes on where at most one wave in
// NARROW_WIDE needs full words: those cost 72 bytes a node in the place of 8, and a round trip.
// Below 2^20 nodes a step is bound by the caches and by latency, and the gain is lost (815,257 nodes
// 30.7 -> 30.6 us).  Colour-gradient tables keep 16 bits: its kernels wait for other loads (192^3
// 208.5 -> 207.8 us, 649,605 nodes FP64 97.6 -> 99.4).  So do a solute's own (20.3 -> 20.6 us).
// The header is the same for all lanes of a wave: scalar loads bring it into scalar registers,
// where the masks serve as the condition of a select without a compare.
#pragma once
#include <cstdint>

#include "handle.h"
#include "lattice.h"

namespace lbm {

constexpr int64_t WAVE_NODES = 64;

// The first node of n's 64-node group: launches over a node range that does not start on a
// group boundary start their threads here (and idle the lanes before the range).
__host__ __device__ __forceinline__ int64_t group_floor(int64_t n) { return n & ~int64_t(63); }

// The row a lane reads: its own node's, also past the last node (the arrays have P rows, and the
// links of a row past the last node stay in place), or past the last row the one of the same lane in
// the last wave.  A lane always reads the row of its own place in a wave: the header's masks go by
// lane.
__device__ __forceinline__ int64_t lane_row(int64_t n, int64_t P) { return n < P ? n : P - WAVE_NODES + (n & (WAVE_NODES - 1)); }

// How a kernel follows links.  LINK_16 and LINK_8: ranks of that width, and in the flow step also
// 32-bit offsets, into buffers of less than 4 GiB (pull_value).  LINK_FAR: any table and any buffer.
// The width is a template parameter as a branch on it in the kernel cost short steps 3 to 4 %
// (4,224 nodes FP64 3.63 -> 3.77 us, colour gradient of 49,577 nodes FP32 9.67 -> 10.0 us).
enum LinkForm : int { LINK_FAR = 0, LINK_16 = 1, LINK_8 = 2 };
inline int link_form(const NbrDev &d, uint64_t buffer_bytes)
{
    return buffer_bytes >> 32 ? LINK_FAR : d.narrow ? LINK_8 : LINK_16;
}

// Where a node's K first populations come from (K = 6: the axis directions, all a D3Q7 pull
// needs): population q from node up[q - 1], or from the node itself where solid(q).
template <int K>
struct Links {
    uint32_t up[K];
    uint64_t bb[K];   // the wave's lanes with a solid upstream site
    uint64_t edge;    // the wave's lanes whose columns wrap round in z
    uint32_t first;   // the index of their first record
    __device__ __forceinline__ bool solid(int q) const { return __builtin_amdgcn_inverse_ballot_w64(bb[q - 1]); }
};

// The links of row n < P, but for those of an edge lane with e_z != 0, which wrap_links adds.
// Lane k of the calling wave must hold row k of one group of 64 (n & 63 == k for every active lane,
// n >> 6 the same for all), which holds for launches whose workgroups are whole wavefronts over
// consecutive, 64-aligned row ranges.
template <int LF, int K>
__device__ __forceinline__ void level_links(const NbrDev &d, int64_t P, int64_t n, Links<K> &l)
{
    static_assert(K == 18 || K == 6, "all links, or those along the axes");
    const uint32_t w = __builtin_amdgcn_readfirstlane((uint32_t)(n >> 6));
    const uint32_t *__restrict__ h = d.hdr + (int64_t)w * HDR_WORDS;
    const bool narrow = LF == LINK_FAR ? d.narrow != 0 : LF == LINK_8;
    uint2 ra{}, rb{};
    if (narrow) {
        ra.x = reinterpret_cast<const uint32_t *>(d.res)[n];
        if (K > 6) rb.x = reinterpret_cast<const uint32_t *>(d.res)[P + n];
    } else {
        ra = reinterpret_cast<const uint2 *>(d.res)[n];
        if (K > 6) rb = reinterpret_cast<const uint2 *>(d.res)[P + n];
    }
#pragma unroll
    for (int q = 1; q <= K; ++q) l.bb[q - 1] = reinterpret_cast<const uint64_t *>(h + HDR_MASK)[q - 1];
    l.edge = reinterpret_cast<const uint64_t *>(h + HDR_EDGE)[0];
    l.first = h[HDR_EDGE_BASE];
    const uint32_t slot = h[HDR_WIDE];
    uint32_t r[NCOL];
    if (narrow) {
#pragma unroll
        for (int c = 0; c < NCOL; ++c) r[c] = (uint32_t)n + ((c < 4 ? ra.x : rb.x) >> (8 * (c % 4)) & 0xFFu);
    } else {
#pragma unroll
        for (int c = 0; c < NCOL; ++c) {
            const uint32_t v = c < 4 ? (c < 2 ? ra.x : ra.y) : (c < 6 ? rb.x : rb.y);
            r[c] = c % 2 ? v >> 16 : v & 0xFFFFu;
        }
    }
    // decoded whether the wave is compact or not: in an else branch, the rank loads would be
    // issued only when the header has arrived
#pragma unroll
    for (int q = 1; q <= K; ++q) {
        const int c = link_column(q);
        if (c == NCOL) {
            l.up[q - 1] = EZ[q] > 0 ? (uint32_t)n - 1 : (uint32_t)n + 1;
        } else {
            const uint32_t at = h[c] + r[c];
            l.up[q - 1] = EZ[q] == 0 ? at : EZ[q] > 0 ? at - 1 : at + (l.solid(column_link(c)) ? 0u : 1u);
        }
    }
    if (slot != HDR_COMPACT) {
        const uint32_t *__restrict__ wp = d.wide + (int64_t)slot * (18 * 64) + (n & 63);
#pragma unroll
        for (int q = 1; q <= K; ++q) l.up[q - 1] = wp[(q - 1) * 64];
        l.edge = 0;
    }
}

template <int K>
__device__ __forceinline__ void wrap_links(const NbrDev &d, Links<K> &l)
{
    if (l.edge == 0) return;
    const uint32_t before = __builtin_amdgcn_mbcnt_hi((uint32_t)(l.edge >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)l.edge, 0u));
    if (!__builtin_amdgcn_inverse_ballot_w64(l.edge)) return;
    const uint4 *__restrict__ e = d.edge + ((int64_t)l.first + before) * (EDGE_WORDS / 4);
    const uint4 e0 = e[0];
    l.up[4] = e0.x;
    l.up[5] = e0.y;
    if (K > 6) {
        const uint4 e1 = e[1], e2 = e[2];
        const uint32_t v[EDGE_WORDS] = {e0.x, e0.y, e0.z, e0.w, e1.x, e1.y, e1.z, e1.w, e2.x, e2.y, e2.z, e2.w};
#pragma unroll
        for (int q = 11; q <= K; ++q) l.up[q - 1] = v[edge_slot(q)];
    }
}

template <int LF = LINK_FAR, int K>
__device__ __forceinline__ void load_links(const NbrDev &d, int64_t P, int64_t n, Links<K> &l)
{
    level_links<LF>(d, P, n, l);
    wrap_links(d, l);
}

}  // namespace lbm
