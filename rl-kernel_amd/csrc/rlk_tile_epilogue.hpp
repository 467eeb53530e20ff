// Pieces shared by the 16-bit MFMA kernels and the fp32 MFMA kernels of the fused linear-logprob
// path: both work on the same 256 x 256 workgroup tile with the same wavefront grid, and their
// accumulator layouts (16 x 16 and 32 x 32 MFMA tiles) differ only in the constants of AccTile, so
// the code that consumes a finished tile is written once.
#pragma once
#include "rlk_gemm.hpp"

namespace rlk {

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

// Online-softmax update of one wavefront slab (128 vocab rows x 64 tokens) held in `acc`, for
// either accumulator geometry AT (see AccTile).  `a` supplies V (vocab rows of the shard) and scale2
// (log2(e) / temperature).
// GENERAL = false: no bias and no masked vocab rows (every tile full), the common case.
// The target logit is picked up in the same pass that feeds the sum, so the captured value is
// the very fp32 number that entered the softmax.  `vw` is the slab's first vocab row; targets below
// `v_own` belong to another tile (a last tile that is shifted back overlaps its neighbour).
template <bool GENERAL, class AT, class Args>
__device__ inline void fwd_epilogue(const typename AT::vec (&acc)[AT::TM][AT::TN], const Args& a,
                                    const float* bias, int vw, int v_own, int lane, const int (&tgt)[AT::TN],
                                    float (&m)[AT::TN], float (&s)[AT::TN], float (&zt)[AT::TN])
{
    constexpr int TM = AT::TM, TN = AT::TN, R = AT::kRegs;
    auto logit = [&](int i, int j, int r) -> float {
        float z = acc[i][j][r];
        if (GENERAL) {
            const int v = vw + AT::quad_row(i, r >> 2, lane) + (r & 3);
            if (bias != nullptr) z += bias[v < a.V ? v : a.V - 1];
            if (v >= a.V) z = -INFINITY;
        }
        return z;
    };
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        float tmax = -INFINITY;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int r = 0; r < R; ++r) tmax = fmaxf(tmax, logit(i, j, r));
        __builtin_amdgcn_sched_barrier(0);
        tmax *= a.scale2;
        const float mnew = fmaxf(m[j], tmax);
        const float mref = mnew == -INFINITY ? 0.f : mnew;
        // register index (i * R + r) of the target row in this lane, or -1
        const int etgt = AT::reg_of_row(tgt[j] >= v_own ? tgt[j] - vw : -1, lane);
        // four partial sums (fixed association) keep the exp results off a single add chain; the
        // target capture runs only when some lane of the wavefront owns a target row in this slab
        float ps[4] = {0.f, 0.f, 0.f, 0.f};
        float zraw = 0.f;
        if (__builtin_amdgcn_ballot_w64(etgt >= 0) != 0) {  // uniform
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const float z = logit(i, j, r);
                    ps[r & 3] += __builtin_amdgcn_exp2f(fmaf(z, a.scale2, -mref));
                    zraw = (etgt == i * R + r) ? z : zraw;
                }
        } else {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int r = 0; r < R; ++r)
                    ps[r & 3] += __builtin_amdgcn_exp2f(fmaf(logit(i, j, r), a.scale2, -mref));
        }
        const float sum = (ps[0] + ps[1]) + (ps[2] + ps[3]);
        __builtin_amdgcn_sched_barrier(0);
        s[j] = s[j] * __builtin_amdgcn_exp2f(m[j] - mref) + sum;
        m[j] = mnew;
        if (etgt >= 0) zt[j] = zraw * a.scale2;
    }
}

// acc += bias of a full tile: `vw` is the first vocab row of this wavefront's slab, relative to
// bias[0].  A lane holds quads of four consecutive vocab rows, so the bias arrives in 16-byte
// loads that are the same for every lane of a lane group (one broadcast request each).
template <class AT>
__device__ inline void add_bias(typename AT::vec (&acc)[AT::TM][AT::TN], const float* bias, int vw, int lane)
{
#pragma unroll
    for (int i = 0; i < AT::TM; ++i)
#pragma unroll
        for (int q = 0; q < AT::kQuads; ++q) {
            const float* p = bias + vw + AT::quad_row(i, q, lane);
            const float b0 = p[0], b1 = p[1], b2 = p[2], b3 = p[3];
#pragma unroll
            for (int j = 0; j < AT::TN; ++j) {
                acc[i][j][q * 4 + 0] += b0;
                acc[i][j][q * 4 + 1] += b1;
                acc[i][j][q * 4 + 2] += b2;
                acc[i][j][q * 4 + 3] += b3;
            }
        }
}

// Rows below `skip` of a finished 256-row tile (M index) become -inf: they belong to the left neighbour
// of a tile that was shifted back to end at the vocabulary's edge, and exp2 makes them exact zeros, in
// the softmax sum and in dZ alike.  One more product does it: A holds -inf in k = 0 of those rows, B
// holds 1 there, everything else is zero.  (Selecting in the accumulators, on a branch or before the
// first product, cost the forward 28 to 497 spilled registers and 2 % of its time.)
template <class T, int TM, int TN>
__device__ inline void mask_rows(f32x4_t (&acc)[TM][TN], int slab_row0, int skip, int lane)
{
    if (skip <= __builtin_amdgcn_readfirstlane(slab_row0)) return;  // uniform
    const bool k0 = lane < 16;  // lanes 0 .. 15 hold k = 0 .. 7 of an operand fragment, k = 0 in the low half
    const u32x4_t one{k0 ? static_cast<uint32_t>(T::from_float(1.f)) : 0u, 0u, 0u, 0u};
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const bool out = k0 && slab_row0 + i * 16 + lane < skip;
        const u32x4_t low{out ? static_cast<uint32_t>(T::from_float(-INFINITY)) : 0u, 0u, 0u, 0u};
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = T::mfma(low, one, acc[i][j]);
    }
}

// 16-byte store of results that no kernel reads soon, past the L2 (agent scope, sc1, and non-temporal cache policy;
// either alone leaves the lines dirty in the L2).  Inline assembly because no builtin gives a global store both
// bits.  The value stays of the type it has: accumulators bit-cast to integers for the operand (or for the buffer
// store builtins) cost the forward 100 spilled registers.
// The compiler sees no hazards of an inline store, so both sides of it are kept here (build.py checks the device
// code for them):
// - behind it two wait states (s_nop 1) before a vector instruction may overwrite its data registers, as the
//   compiler puts them behind its own stores of more than 8 bytes on this target;
// - in front of it twelve between a matrix instruction and the store of its result: a value that no vector
//   instruction has touched since goes through settle_column first.
template <class V>
__device__ inline void stream_store(void* p, uint32_t lane_offset, V v)
{
    static_assert(sizeof(V) == 16, "16 bytes a lane");
    asm volatile("global_store_dwordx4 %0, %1, off sc1 nt\n\ts_nop 1"
                 :
                 : "v"(static_cast<char*>(p) + lane_offset), "v"(v)
                 : "memory");
}

// The matrix instructions that write column j of the accumulators are done: sixteen wait states, tied to the
// registers so that none of them moves behind.
template <int TN>
__device__ inline void settle_column(f32x4_t (&acc)[8][TN], int j)
{
    asm volatile("s_nop 15"
                 : "+v"(acc[0][j]), "+v"(acc[1][j]), "+v"(acc[2][j]), "+v"(acc[3][j]), "+v"(acc[4][j]),
                   "+v"(acc[5][j]), "+v"(acc[6][j]), "+v"(acc[7][j]));
}

// Tiles of a launch are handed out round by round: workgroup b computes the tiles with linear ids
// b, b + gridDim.x, b + 2 gridDim.x, ...  With a grid that is a multiple of 8, a workgroup keeps
// its XCD from round to round, so every round forms the same L2-sharing patches as a launch with
// one workgroup per tile would.
constexpr int kWalkPatch = 8;  // tile rows of the patch the 32 workgroups of one XCD cover per round
struct TileWalk {
    int lin, total, gm, gn;
    __device__ inline TileWalk(int total_, int gm_, int gn_)
        : lin(blockIdx.x), total(total_), gm(gm_), gn(gn_) {}
    __device__ inline bool valid() const { return lin < total; }
    __device__ inline bool has_next() const { return lin + static_cast<int>(gridDim.x) < total; }
    __device__ inline void coords(bool next, int& tm, int& tn) const
    {
        xcd_tile(next ? lin + static_cast<int>(gridDim.x) : lin, total, gm, gn, kWalkPatch, tm, tn);
    }
    __device__ inline void advance() { lin += static_cast<int>(gridDim.x); }
};

// Walk of a tile list whose launch gives the first `busy` workgroups other work in front: the others start with
// `lead` rounds among themselves, then all go through common rounds.  With a grid and a `busy` that are
// multiples of 8 a workgroup keeps its XCD, as above.
struct LeadWalk {
    int k, at, total, gm, gn, lead, rest;
    __device__ inline LeadWalk(int total_, int gm_, int gn_, int busy, int lead_)
        : total(total_), gm(gm_), gn(gn_), lead(lead_), rest(static_cast<int>(gridDim.x) - busy)
    {
        const int b = static_cast<int>(blockIdx.x);
        at = b < busy ? b + rest : b - busy;
        k = b < busy ? lead : 0;
    }
    __device__ inline int lin(int round) const
    {
        return (round < lead ? round * rest : lead * rest + (round - lead) * static_cast<int>(gridDim.x)) + at;
    }
    __device__ inline bool valid() const { return lin(k) < total; }
    __device__ inline bool has_next() const { return lin(k + 1) < total; }
    __device__ inline void coords(bool next, int& tm, int& tn) const
    {
        xcd_tile(lin(next ? k + 1 : k), total, gm, gn, kWalkPatch, tm, tn);
    }
    __device__ inline void advance() { ++k; }
};

template <class V, int TM, int TN>
__device__ inline void zero_acc(V (&acc)[TM][TN])
{
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < static_cast<int>(sizeof(V) / sizeof(float)); ++r) acc[i][j][r] = 0.f;
}

}  // namespace rlk
