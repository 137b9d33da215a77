// pull.h -- the pull-stream gather shared by the single-phase and colour-gradient kernels.
//
// Population q of node n after streaming is the post-collision population q of the upstream
// node n - e_q, or -- when that site is solid -- the post-collision population opp(q) of n
// itself (halfway bounce-back).  The links of a node (load_links) give, per moving direction
// q = 1..18, the upstream node and whether its site is solid, so each load is one select and
// one gather; the rest population needs no link.
#pragma once
#include "collide.h"
#include "lattice.h"
#include "nbrpack.h"
#include "storage.h"

namespace lbm {

enum KMode { K_INIT = 0, K_DIRECT = 1, K_PULL = 2 };

// Element offset of population q of node n after streaming, in a buffer of NQ a node: the node and
// the row are selected, not the offsets, which the compiler would compute in divergent branches.
template <int NQ, int K>
__device__ __forceinline__ int64_t pull_offset(const Links<K> &l, int64_t n, int q)
{
    const uint32_t at = l.solid(q) ? (uint32_t)n : l.up[q - 1];
    const uint32_t row = l.solid(q) ? uint32_t(opp(q) * POP_BLOCK) : uint32_t(q * POP_BLOCK);
    return (int64_t)((uint64_t)(at / POP_BLOCK) * uint32_t((NQ - 1) * POP_BLOCK) + (at + row));
}

// Population q of node n after streaming.  Where the form allows it, the offset is worked out in 32
// bits from a base that is the same for all lanes: five full-rate instructions in the place of a
// 64-bit multiply-add (quarter rate) and six others, in FP16 a sixth of the step's vector issue.
// With 8-bit ranks, 64-bit -> 32-bit offsets: 208 x 224 x 240 FP16 72.6 -> 68.5 us, 256^3 sphere pack
// FP32 171.2 -> 167.1 us, 171 x 203 x 187 FP64 107.6 -> 105.6 us, 192^3 fibres with solute FP32 215.9 ->
// 213.0 us; with 16-bit ranks 4,224 nodes FP64 3.63 -> 3.54 us, 157,286 nodes 12.8 -> 12.6 us.  Not in
// the colour-gradient and solute kernels, where it lost 1 to 3 %.
template <int NQ, int LF, int K, typename T>
__device__ __forceinline__ T pull_value(const T *__restrict__ src, const Links<K> &l, int64_t n, int q)
{
    if (LF == LINK_FAR) return src[pull_offset<NQ>(l, n, q)];
    constexpr uint32_t SKIP = (NQ - 1) * POP_BLOCK;
    const int row = q < opp(q) ? q : opp(q);
    const uint32_t up = l.up[q - 1], own = (uint32_t)n;
    const uint32_t there = up + (up / POP_BLOCK) * SKIP + (q - row) * POP_BLOCK;
    const uint32_t here = own + (own / POP_BLOCK) * SKIP + (opp(q) - row) * POP_BLOCK;
    const uint32_t at = (l.solid(q) ? here : there) * (uint32_t)sizeof(T);
    return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(src + row * POP_BLOCK) + at);
}

// load(q) for the links of node n, the ones at the node's height first: an edge lane's others wait
// for its record.  The records are asked for before those loads, not after: loads return in order,
// and behind them the wait for a record was a wait for all of them, in every wave, as the compiler
// counts the loads of both sides of a branch.  Step on device: 4,224 nodes FP64 4.05 -> 3.63 us, colour
// gradient of 49,577 nodes FP32 10.06 -> 9.76 us, of 649,605 nodes FP64 99.4 -> 97.6 us, 256^3 sphere
// pack FP32 176.0 -> 174.7 us; without the barrier, which keeps the order, 157,286 nodes FP64 12.8 -> 13.2.
template <int LF, int K, typename F>
__device__ __forceinline__ void gather_links(const NbrDev &nbr, int64_t P, int64_t n, Links<K> &l, F &&load)
{
    load_links<LF>(nbr, P, n, l);
#pragma unroll
    for (int q = 1; q <= K; ++q)
        if (EZ[q] == 0) load(q);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 1; q <= K; ++q)
        if (EZ[q] != 0) load(q);
}

// Gather the 19 pre-collision deviations of node n.  In K_DIRECT mode the buffer holds a
// post-streaming state (a loaded checkpoint) and is read in place.  The node's links are
// returned in l (K_PULL only) for callers that also need the neighbour sites.
template <typename ST, int MODE, int LF = LINK_FAR>
__device__ __forceinline__ void gather_pops(const ST *__restrict__ src, const NbrDev &nbr, int64_t P, int64_t n,
                                            float inv_scale, typename Store<ST>::C (&h)[Q], Links<Q - 1> &l)
{
    h[0] = Store<ST>::load(src[pop_at<Q>(0, n)], inv_scale);
    if (MODE == K_DIRECT) {
#pragma unroll
        for (int q = 1; q < Q; ++q) h[q] = Store<ST>::load(src[pop_at<Q>(q, n)], inv_scale);
        return;
    }
    gather_links<LF>(nbr, P, n, l, [&](int q) { h[q] = Store<ST>::load(pull_value<Q, LF>(src, l, n, q), inv_scale); });
}

}  // namespace lbm
