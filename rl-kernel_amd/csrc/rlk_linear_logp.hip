// Fused linear -> selected-token log-prob for gfx950: forward (online logsumexp over vocab
// tiles, logits not stored but for a small training step), split combine, and the recompute-based backward (dZ block,
// dH and dW contractions).  All reductions run in a fixed order: same input, same bits.
//
// Orientation used by every kernel here: the MFMA "M" index lives in accumulator registers (the
// 4 registers of a 16 x 16 tile hold rows 4 (l / 16) + 0..3 of column l % 16), the "N" index is
// the lane.  In the forward and in the dZ recompute M = vocab and N = token, so the softmax
// reduction over vocab is an in-register loop per lane; the four lanes that share a token column
// (l, l + 16, l + 32, l + 48) merge their states by two shuffles once per split.
#include "rlk_common.hpp"
#include <algorithm>
#include <mutex>
#include <vector>

#include "rlk_gemm.hpp"
#include "rlk_grpo.hpp"
#include "rlk_tile_epilogue.hpp"

// Load windows (MFMA slots of a K step's second slice over which its 8 loads are spread, see
// TileGemmDtl), measured one kernel at a time at the Llama head (launch time with 16 / 24 / 32
// slots: dZ 791 / 801 / 819 us, dH 822 / 813 / 799 us, dW 866 / 852 / 846 us; forward 23.71 / 23.64 /
// 23.63 ms).
constexpr int kWinFwd = 32;
constexpr int kWinDz = 16;
constexpr int kWinDh = 32;
constexpr int kWinDw = 32;

namespace rlk {


// ------------------------------------------------------------------------------------------- //
// Forward
// ------------------------------------------------------------------------------------------- //
struct FwdArgs {
    const uint16_t* hidden;   // [N][H]
    const uint16_t* weight;   // [V][H]   (local vocab shard)
    const float* bias;        // [V] or null
    const int64_t* targets;   // [N] global ids
    float* part_m;            // [n_split][N] running max (log2 domain)
    float* part_s;            // [n_split][N] running sum of 2^(z - max)
    float* part_z;            // [n_split][N] captured target logit (log2 domain), 0 if not owned
    // optional second head over the same hidden states and targets (a frozen reference model):
    // its tiles follow the first head's in the same pipeline, its partials go to part2_*
    const uint16_t* weight2;  // [V][H] or null
    const float* bias2;       // [V] or null
    float* part2_m;
    float* part2_s;
    float* part2_z;
    int N;
    int H;
    int V;
    int64_t vocab_start;
    int n_split;     // splits handled by this launch
    int split_lo;    // first slot of the partial arrays this launch writes
    int row_blocks;
    int patch_rows;  // token blocks of the patch that the workgroups of one XCD cover per round
    int tile_lo;     // first vocab tile of this launch
    int vtiles;      // vocab tiles of this launch
    float scale2;    // log2(e) / temperature
    float* kept;     // KEEP: logits of every tile, see "Kept logits"
};

// Kept logits: fp32 logits (bias added, masked vocab rows -inf) that a training forward leaves for its backward
// when they are few (rlk_linear_logp_kept_bytes), so that dZ does not have to recompute them.  One block
// of 256 KiB per (token tile, vocab tile), token tile the slow index, made of four slabs of 64 tokens;
// a slab holds the accumulator quads as the wavefronts have them,
// [2 wavefronts along vocab][TM][TN][64 lanes][4], so a wavefront stores a tile in 1 KiB pieces.  The last token tile
// is moved back to end at N as in the backward; columns of 16 tokens past N (fewer than 256 tokens) are not stored,
// and a tile has only the slabs that hold tokens, two at least (dW takes two K steps): kept_slabs.
// They are stored past the L2 (stream_store): forward + backward of 1500 x 4096 x 128256 4067 -> 4020 us, of 64 x
// 4096 x 128256 730 -> 719, of 300 x 2048 x 50257 359 -> 349, of 4096 x 2048 x 50257 2252 -> 2238, of 2000 x 2560 x
// 32000 934 -> 940.  (A forward repeated alone, whose weight stays in the memory-side cache when they bypass it,
// goes from 774 to 655 us at 4096 x 2048 x 50257, 585 without keeping; inside a step keeping costs it 140 us.)
constexpr int kKeptSlab = 64 * 256;       // floats
constexpr int kKeptTile = 4 * kKeptSlab;
// By the width of the token tile in 64 tokens, which follows N up to 192 (launch_fwd_chained, launch_kept).
constexpr int kept_tile_slabs(int tn) { return tn < 2 ? 2 : tn; }
constexpr int kept_slabs(int64_t N) { return kept_tile_slabs(N <= 64 ? 1 : N <= 128 ? 2 : N <= 192 ? 3 : 4); }

// One workgroup = one block of 256 tokens x one contiguous range of vocab tiles.
// GENERAL = false covers vocab tiles [0, vtiles) split n_split ways, every one of 256 valid rows (a
// bias is added to the finished tile before the softmax update); GENERAL = true handles masked rows
// over tiles [tile_lo, tile_lo+vtiles).  When V is not a multiple of 256 the last tile of the chained
// walk is shifted back to rows [V - 256, V) and the rows of its left neighbour are masked, so it runs
// in the same launch and pipeline as all others.  A launch of its own for the ragged tile kept
// row_blocks workgroups busy for a whole tile while the other CUs waited: 70 of 750 us at 4096 x
// 2048 x 50257, 48 of 458 us at 1000 x 1536 x 151936.
// CHAIN (!GENERAL, H a multiple of BK and >= 2 BK, V >= 256): all tiles run through one pipeline.
// KEEP (CHAIN, one head): the logits stay in a.kept.
// AT: Acc16, or with at most 192 tokens the narrower token tile of Acc16Few (CHAIN): the launch is bound by reading
// the weight then and the products of a 256-token tile were the larger part of it.  A token's sums are taken over
// the same rows in the same order, so its bits are those of the full tile.
template <class T, int BK, bool GENERAL, bool CHAIN, bool KEEP = false, class AT = Acc16>
__global__ __launch_bounds__(kThreads) void linear_logp_fwd_kernel(FwdArgs a)
{
    static_assert(!(GENERAL && CHAIN), "the chained variant covers full tiles only");
    static_assert(CHAIN || !KEEP, "logits are kept by the chained variant only");
    static_assert(CHAIN || std::is_same<AT, Acc16>::value, "narrow token tiles are for the chained variant");
    constexpr int TM = AT::TM, TN = AT::TN;
    using Gemm = TileGemm<T, false, false, BK>;
    using Dtl = TileGemmDtl<T, false, false, BK, kWinFwd * TN / 4, false, false, AT>;
    extern __shared__ __attribute__((aligned(16))) char smem[];

    int tb, sp;
    xcd_tile(blockIdx.x, a.row_blocks * a.n_split, a.row_blocks, a.n_split, a.patch_rows, tb, sp);
    // vocab tiles [t0, t1) of this split: the first (vtiles % n_split) splits take one extra.
    const int base = a.vtiles / a.n_split, extra = a.vtiles % a.n_split;
    const int t0 = a.tile_lo + sp * base + (sp < extra ? sp : extra);
    const int t1 = t0 + base + (sp < extra ? 1 : 0);

    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int wm = wave / kWN, wn = wave % kWN;
    const int tok0 = KEEP ? max(0, min(tb * 256, a.N - 256)) : tb * 256;
    const int tok_valid = min(256, a.N - tok0);
    const int tok_own = KEEP ? tb * 256 - tok0 : 0;  // rows below belong to the token block in front

    float m[TN], s[TN], zt[TN];
    int tgt[TN];  // target id relative to the shard, -1 when not in [0, V)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int t = wn * (TN * 16) + AT::col(j, lane);
        int64_t g = a.targets[tok0 + (t < tok_valid ? t : tok_valid - 1)] - a.vocab_start;
        tgt[j] = (g >= 0 && g < a.V) ? static_cast<int>(g) : -1;
    }
    auto reset_state = [&]() {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            m[j] = -INFINITY;
            s[j] = 0.f;
            zt[j] = 0.f;
        }
    };

    // Merge of one head's state: the four lane groups of a wavefront (same token, different vocab
    // rows; groups 16 apart first, then 32 apart), then the wavefronts along M through LDS, in a
    // fixed order; written to that head's partial arrays.  The LDS patch lies behind the pipeline
    // stages, so the merge of the first head can run while the second head's first K steps are
    // already on their way.
    float* red = reinterpret_cast<float*>(smem + Dtl::kSmemBytes);  // [kWM][256 tokens][3]
    static_assert(Dtl::kSmemBytes + kWM * 256 * 3 * 4 <= Gemm::kSmemBytes, "merge patch must fit the kernel's LDS");
    auto flush_state = [&](float* pm, float* ps, float* pz) {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            float mj = m[j], sj = s[j], zj = zt[j];
#pragma unroll
            for (int off = 16; off <= 32; off <<= 1) {
                const float m2 = __shfl_xor(mj, off);
                const float s2 = __shfl_xor(sj, off);
                const float z2 = __shfl_xor(zj, off);
                const float mm = fmaxf(mj, m2);
                const float mref = mm == -INFINITY ? 0.f : mm;
                // both partners evaluate the same expression: the lower group's term first
                const bool low = (lane & off) == 0;
                const float lo_m = low ? mj : m2, hi_m = low ? m2 : mj;
                const float lo_s = low ? sj : s2, hi_s = low ? s2 : sj;
                sj = lo_s * __builtin_amdgcn_exp2f(lo_m - mref) + hi_s * __builtin_amdgcn_exp2f(hi_m - mref);
                mj = mm;
                zj = (low ? zj : z2) + (low ? z2 : zj);
            }
            if (lane < 16) {
                float* dst = red + ((wm * 256) + wn * (TN * 16) + j * 16 + lane) * 3;
                dst[0] = mj;
                dst[1] = sj;
                dst[2] = zj;
            }
        }
        __syncthreads();
        const int t = threadIdx.x;
        if (t >= tok_own && t < tok_valid) {
            float mm = -INFINITY;
#pragma unroll
            for (int w = 0; w < kWM; ++w) mm = fmaxf(mm, red[(w * 256 + t) * 3]);
            const float mref = mm == -INFINITY ? 0.f : mm;
            float ss = 0.f, zz = 0.f;
#pragma unroll
            for (int w = 0; w < kWM; ++w) {
                const float* pw = red + (w * 256 + t) * 3;
                ss += pw[1] * __builtin_amdgcn_exp2f(pw[0] - mref);
                zz += pw[2];
            }
            const int64_t o = static_cast<int64_t>(a.split_lo + sp) * a.N + tok0 + t;
            pm[o] = mm;
            ps[o] = ss;
            pz[o] = zz;
        }
        __syncthreads();  // the patch may be written again
    };

    const int n_heads = a.weight2 != nullptr ? 2 : 1;
    Operand B{a.hidden + static_cast<int64_t>(tok0) * a.H, a.H, tok_valid};
    // first vocab row of a tile; only the chained walk is ever given a tile that has to move back
    auto tile_row = [&](int vt) { return CHAIN ? min(vt * 256, a.V - 256) : vt * 256; };
    auto tile_origin = [&](int head, int vt) {
        return (head == 0 ? a.weight : a.weight2) + static_cast<int64_t>(tile_row(vt)) * a.H;
    };
    if constexpr (CHAIN) {
        // every tile is full (or moved back) and every split has a tile (n_split <= vtiles): one pipeline
        // runs through all tiles of the range (and then through the same range of the second head), the
        // K loop of a tile already fetching the head of the next one while the softmax update runs (the
        // pipeline looks two K steps ahead, which stays within the next tile from two steps up)
        typename Dtl::Stream st;
        Dtl::begin(st, Operand{tile_origin(0, t0), a.H, 256}, B, a.H, smem);
        bool counted = false;
        for (int head = 0; head < n_heads; ++head) {
            reset_state();
            for (int vt = t0; vt < t1; ++vt) {
                const int row0 = tile_row(vt);
                f32x4_t acc[TM][TN];
                zero_acc(acc);
                const void* next = vt + 1 < t1 ? tile_origin(head, vt + 1)
                                               : (head + 1 < n_heads ? tile_origin(head + 1, t0)
                                                                     : tile_origin(head, vt));
                Dtl::template tile<true, KEEP ? TM * TN : 0>(st, next, B.base, acc, smem, counted);
                const float* bias = head == 0 ? a.bias : a.bias2;
                if (bias != nullptr) add_bias<AT>(acc, bias, row0 + wm * (TM * 16), lane);  // uniform
                mask_rows<T>(acc, wm * (TM * 16), vt * 256 - row0, lane);
                if constexpr (KEEP) {
                    const int64_t tile = static_cast<int64_t>(tb) * a.vtiles + vt;
                    float* dst = a.kept + tile * (kept_tile_slabs(TN) * kKeptSlab) + wm * (kKeptSlab / 2);
#pragma unroll
                    for (int j = 0; j < TN; ++j) {
                        const int cols = wn * TN + j;  // 16 tokens; four of them make a slab
                        if (cols * 16 >= tok_valid) break;  // uniform
                        settle_column(acc, j);
                        float* quads = dst + (cols >> 2) * kKeptSlab + (cols & 3) * 256;
#pragma unroll
                        for (int i = 0; i < TM; ++i)
                            stream_store(quads + i * (Acc16::TN * 256), lane * 16, acc[i][j]);
                    }
                    counted = tok_valid == 256;
                }
                fwd_epilogue<GENERAL, AT>(acc, a, nullptr, row0 + wm * (TM * 16), vt * 256, lane, tgt, m, s, zt);
            }
            if (head == 0)
                flush_state(a.part_m, a.part_s, a.part_z);
            else
                flush_state(a.part2_m, a.part2_s, a.part2_z);
        }
        Dtl::end(st);
    } else {
        for (int head = 0; head < n_heads; ++head) {
            reset_state();
            const float* bias = head == 0 ? a.bias : a.bias2;
            for (int vt = t0; vt < t1; ++vt) {
                const int v0 = vt * 256;
                Operand A{tile_origin(head, vt), a.H, min(256, a.V - v0)};
                f32x4_t acc[TM][TN];
                zero_acc(acc);
                Gemm::run(A, B, a.H, acc, smem);
                if (!GENERAL && bias != nullptr) add_bias<AT>(acc, bias, v0 + wm * (TM * 16), lane);  // uniform
                fwd_epilogue<GENERAL, AT>(acc, a, bias, v0 + wm * (TM * 16), v0, lane, tgt, m, s, zt);
            }
            if (head == 0)
                flush_state(a.part_m, a.part_s, a.part_z);
            else
                flush_state(a.part2_m, a.part2_s, a.part2_z);
        }
    }
}

struct CombineArgs {
    const float* part_m;
    const float* part_s;
    const float* part_z;
    const int64_t* targets;
    float* logp;
    float* lse;
    int32_t* err_flag;
    int N;
    int V;
    int n_split;
    int64_t vocab_start;
    int64_t ignore_index;
    int use_ignore;
    int strict;  // 1: a non-ignored target outside [vocab_start, vocab_start+V) raises err_flag
};

// M = max_s m_s ; S = sum_s s_s 2^(m_s - M) ; z_t = sum_s z_t,s ; lse = ln2 (M + log2 S).
// Writes lse and logp of token n and returns the logp.
__device__ inline float combine_token(const CombineArgs& a, int64_t n)
{
    float mm = -INFINITY;
    for (int sp = 0; sp < a.n_split; ++sp) mm = fmaxf(mm, a.part_m[static_cast<int64_t>(sp) * a.N + n]);
    float ss = 0.f, zz = 0.f;
    for (int sp = 0; sp < a.n_split; ++sp) {
        const int64_t o = static_cast<int64_t>(sp) * a.N + n;
        ss += a.part_s[o] * exp2f(a.part_m[o] - mm);
        zz += a.part_z[o];
    }
    const float lse2 = mm + log2f(ss);
    const int64_t t = a.targets[n];
    const bool ignored = a.use_ignore && t == a.ignore_index;
    const int64_t tl = t - a.vocab_start;
    const bool owned = tl >= 0 && tl < a.V;
    if (!ignored && !owned && a.strict) *a.err_flag = 1;
    const float lp = ignored ? 0.f : (zz - lse2) * kLn2;
    a.lse[n] = lse2 * kLn2;
    a.logp[n] = lp;
    return lp;
}

// Many splits (few tokens): 4 tokens x 64 split groups per workgroup fetch the partial states side by
// side, then one thread per token adds the rescaled sums in split order, as combine_token would; the
// merged state replaces the token's slot 0, which the combine kernels read as their only split.  One
// thread walking all splits of a token through memory is a chain of dependent loads: 37 us for 160
// tokens x 62 splits.  LDS: the terms [2][n_split][4] behind the group maxima.  (16 tokens x 16 groups took
// 14 us for 160 tokens x 251 splits.)
constexpr int kMergeTokens = 4, kMergeGroups = 64;
inline size_t merge_smem(int n_split) { return static_cast<size_t>(kMergeGroups + 2 * n_split) * kMergeTokens * 4; }
__global__ __launch_bounds__(256) void linear_logp_merge_kernel(float* part_m, float* part_s, float* part_z, int N,
                                                                int n_split)
{
    extern __shared__ __attribute__((aligned(16))) char smem[];
    float* gmax = reinterpret_cast<float*>(smem);
    float* term_s = gmax + kMergeGroups * kMergeTokens;
    float* term_z = term_s + n_split * kMergeTokens;
    const int tx = threadIdx.x % kMergeTokens, g = threadIdx.x / kMergeTokens;
    const int n = blockIdx.x * kMergeTokens + tx;
    const bool live = n < N;
    float mm = -INFINITY;
    if (live)
        for (int sp = g; sp < n_split; sp += kMergeGroups) mm = fmaxf(mm, part_m[static_cast<int64_t>(sp) * N + n]);
    gmax[g * kMergeTokens + tx] = mm;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kMergeGroups; ++k) mm = fmaxf(mm, gmax[k * kMergeTokens + tx]);
    if (live)
        for (int sp = g; sp < n_split; sp += kMergeGroups) {
            const int64_t o = static_cast<int64_t>(sp) * N + n;
            term_s[sp * kMergeTokens + tx] = part_s[o] * exp2f(part_m[o] - mm);
            term_z[sp * kMergeTokens + tx] = part_z[o];
        }
    __syncthreads();  // also: every read of slot 0 of these tokens is behind us
    if (g == 0 && live) {
        float ss = 0.f, zz = 0.f;
#pragma unroll 8
        for (int sp = 0; sp < n_split; ++sp) {
            ss += term_s[sp * kMergeTokens + tx];
            zz += term_z[sp * kMergeTokens + tx];
        }
        part_m[n] = mm;
        part_s[n] = ss;
        part_z[n] = zz;
    }
}

__global__ void linear_logp_combine_kernel(CombineArgs a)
{
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= a.N) return;
    combine_token(a, n);
}

// Combine with the GRPO loss epilogue folded in: the launch has the block / thread partition of
// the stand-alone epilogue (block b owns a contiguous token range, thread t walks it with stride
// 256), merges the split partials of each of its tokens and feeds the fresh log-prob straight into
// the loss terms, the fixed-order partial sums and d loss / d logp.  The active-token count comes
// from grpo_count_kernel, which ran before the contraction.  The workgroup that finishes last
// (integer ticket) adds up the block partials in block order and writes the three scalars, so no
// further launch is needed.  Same expressions, same partition, same tree as combine +
// rlk_grpo_loss_from_logp: same bits.
__global__ __launch_bounds__(kRedThreads) void linear_logp_combine_grpo_kernel(CombineArgs c, GrpoArgs g)
{
    const int64_t per = (g.n + g.blocks - 1) / g.blocks;
    const int64_t lo = per * blockIdx.x;
    const int64_t hi = lo + per < g.n ? lo + per : g.n;
    const float denom = grpo_denominator(g.words);
    Term t{0.f, 0.f, 0.f};
    for (int64_t i = lo + threadIdx.x; i < hi; i += kRedThreads) {
        const float lp = combine_token(c, i);
        const bool on = g.mask == nullptr || g.mask[i] != 0;
        float r = 0.f, k = 0.f, gr = 0.f, gk = 0.f;
        if (on) {
            float pol;
            token_terms(g, i, lp, r, pol, k);
            t.pol += pol;
            if (g.ref_lp != nullptr) t.kl += k;
            t.act += 1.f;
            if (g.dcur != nullptr) token_grad(g, i, lp, denom, gr, gk);
        }
        if (g.ratio) g.ratio[i] = r;
        if (g.kl_terms) g.kl_terms[i] = k;
        if (g.dcur) g.dcur[i] = gr;
        if (g.dkl) g.dkl[i] = gk;
    }
    const Term s = block_sum(t);
    __shared__ int last_block;
    if (threadIdx.x == 0) {
        g.partial[blockIdx.x * 3 + 0] = s.pol;
        g.partial[blockIdx.x * 3 + 1] = s.kl;
        g.partial[blockIdx.x * 3 + 2] = s.act;
        __threadfence();  // the partials are visible before the ticket is taken
        last_block = atomicAdd(&g.words[0], 1) == g.blocks - 1;
    }
    __syncthreads();
    if (last_block) {  // uniform: every other workgroup has published its partials
        __threadfence();
        grpo_finish<true>(g);
    }
}

// ------------------------------------------------------------------------------------------- //
// Backward step 1: dZ block = g/T * (onehot - softmax) for a (token chunk) x (vocab piece)
// ------------------------------------------------------------------------------------------- //
struct DzArgs {
    const uint16_t* hidden;  // chunk origin [tok][H]
    const uint16_t* weight;  // piece origin [v][H]
    const float* bias;       // piece origin or null
    const int64_t* targets;  // chunk origin (global ids)
    const float* lse;        // chunk origin (natural log)
    const float* grad;       // chunk origin, upstream d/dlogp
    const float* scales;     // [0] = loss_scale / temperature (device resident)
    uint16_t* dz;            // [tok_tiles*256][ldz]
    int64_t ldz;
    int tok_valid;
    int v_valid;
    int H;
    int tok_tiles;
    int v_tiles;        // vocab tiles of this launch
    int v_tile_lo;      // first vocab tile of this launch
    int tok_shift;      // rows / vocab rows by which the last token / vocab tile is moved back so that it
    int v_shift;        // ends at the last row there is (0 in the unchained kernels)
    int64_t v_global0;  // global id of the piece's first vocab row
    int64_t ignore_index;
    int use_ignore;
    float scale2;
};

// LDS each wavefront needs to turn its part of a dZ tile into full rows: 64 tokens x 32 vocab
// columns of 16-bit values, 64 bytes per token row, no padding.
constexpr int kDzStageBytes = 64 * 64;

// dZ epilogue of one 256 x 256 tile.  A wavefront owns 128 vocab rows x 64 tokens of the tile; for
// each of its four 32-row groups (two 16-row MFMA tiles) it writes the rounded values into its
// private LDS patch as [token][vocab] rows and reads them back row-wise, so that the tile leaves
// in runs of 64 contiguous bytes per token.  Only the wavefront itself touches its patch: no
// workgroup barrier.  The 8-byte units of a row are XOR-swizzled with 2 * ((token / 4) & 3), which
// makes both the writes (16 tokens x 2 lane groups per pass) and the reads (4 rows x 8 units)
// conflict-free.
//
// A tile that is shifted back (tok_back rows, v_back vocab rows) is still stored at its own place of
// the block; what its neighbour owns is stored as zeros (token rows here through gs = 0, vocab rows
// by the caller through mask_rows).
template <class T, bool GENERAL>
__device__ inline void dz_epilogue(const f32x4_t (&acc)[Acc16::TM][Acc16::TN], const DzArgs& a, int vt, int tt,
                                   int v_back, int tok_back, char* stage)
{
    using AT = Acc16;
    constexpr int TM = AT::TM, TN = AT::TN;
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int wm = wave / kWN, wn = wave % kWN;
    const int tok0 = tt * 256 - tok_back;
    const int tok_rows = min(256, a.tok_valid - tok0);
    const float gscale = a.scales[0];
    const int vd = vt * 256 + wm * (TM * 16);  // column of the block
    const int vw = vd - v_back;                // vocab row of the piece
    const int grp = lane >> 4;  // this lane holds rows 4 * grp + 0..3 of every 16-row tile

    float gs[TN], nlse2[TN];
    int etgt[TN];  // register index (i*4 + r) of the target row in this lane, or -1
    bool any_target = false;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int tl = wn * (TN * 16) + AT::col(j, lane);
        const int tc = tok0 + (tl < tok_rows ? tl : tok_rows - 1);
        const int64_t tg = a.targets[tc];
        const bool live = tl >= tok_back && tl < tok_rows && !(a.use_ignore && tg == a.ignore_index);
        gs[j] = live ? a.grad[tc] * gscale : 0.f;
        nlse2[j] = -a.lse[tc] * kLog2e;
        const int64_t tv = tg - a.v_global0, trel = tv - vw;
        etgt[j] = (trel >= 0 && trel < TM * 16 && tv >= vt * 256) ? AT::reg_of_row(static_cast<int>(trel), lane) : -1;
        any_target = any_target || etgt[j] >= 0;
    }
    // the one-hot term is added only when some lane of the wavefront owns its target row here
    const bool hot = __builtin_amdgcn_ballot_w64(any_target) != 0;  // uniform

    uint16_t* dtile = a.dz + static_cast<int64_t>(tt * 256 + wn * (TN * 16)) * a.ldz + vd;
    auto stage_rows = [&](auto ipc, auto hot_c) {
        constexpr int ip = decltype(ipc)::value;  // 32-row group = MFMA tiles 2 ip and 2 ip + 1
        constexpr bool HOT = decltype(hot_c)::value;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int t = j * 16 + (lane & 15);  // token row inside the wavefront's patch
            char* srow = stage + t * 64;
            const int sw = ((t >> 2) & 3) << 1;
#pragma unroll
            for (int ii = 0; ii < 2; ++ii) {
                constexpr int i0 = 2 * ip;
                const int i = i0 + ii;
                float d[4];
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    float z = acc[i][j][c];
                    float pr;
                    if (GENERAL) {
                        const int v = vw + i * 16 + 4 * grp + c;
                        if (a.bias != nullptr) z += a.bias[v < a.v_valid ? v : a.v_valid - 1];
                        pr = v < a.v_valid ? __builtin_amdgcn_exp2f(fmaf(z, a.scale2, nlse2[j])) : 0.f;
                    } else {
                        pr = __builtin_amdgcn_exp2f(fmaf(z, a.scale2, nlse2[j]));
                    }
                    if constexpr (HOT) {
                        const float hit = (etgt[j] == i * 4 + c) ? gs[j] : 0.f;
                        d[c] = fmaf(-gs[j], pr, hit);
                    } else {
                        d[c] = -gs[j] * pr;
                    }
                }
                // rows 16 ii + 4 grp + 0..3 of this 32-row group: unit 4 ii + grp of the token's row
                *reinterpret_cast<u32x2_t*>(srow + (((4 * ii + grp) ^ sw) * 8)) =
                    u32x2_t{T::pack2(d[0], d[1]), T::pack2(d[2], d[3])};
            }
        }
    };
    static_for<0, TM / 2>([&](auto ipc) {
        constexpr int ip = decltype(ipc)::value;
        if (hot)
            stage_rows(ipc, std::true_type{});
        else
            stage_rows(ipc, std::false_type{});
        __builtin_amdgcn_wave_barrier();
        // copy-out: 8 lanes move one token row (64 bytes), 8 rows per instruction
#pragma unroll
        for (int it = 0; it < 8; ++it) {
            const int row = it * 8 + (lane >> 3);
            const int u = lane & 7;
            const u32x2_t v =
                *reinterpret_cast<const u32x2_t*>(stage + row * 64 + ((u ^ (((row >> 2) & 3) << 1)) * 8));
            *reinterpret_cast<u32x2_t*>(dtile + static_cast<int64_t>(row) * a.ldz + ip * 32 + u * 4) = v;
        }
        __builtin_amdgcn_wave_barrier();
    });
}

// GENERAL = false: every vocab tile of the launch is full (a bias is added to the finished tile).
// CHAIN (needs !GENERAL, H a multiple of BK and >= 2 BK, and 256 rows to read for every tile: the last
// token tile and the last vocab tile may be shifted back by a.tok_shift / a.v_shift rows): the
// workgroup walks its tiles through one pipeline; while a tile's epilogue runs, the first K steps of
// the next tile are already on their way into LDS.
template <class T, int BK, bool GENERAL, bool CHAIN>
__global__ __launch_bounds__(kThreads) void linear_logp_dz_kernel(DzArgs a)
{
    static_assert(!(GENERAL && CHAIN), "the chained variant covers full tiles only");
    using AT = Acc16;
    using Gemm = TileGemm<T, false, false, BK>;
    using Dtl = TileGemmDtl<T, false, false, BK, kWinDz>;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int wave = threadIdx.x >> 6;
    TileWalk walk(a.tok_tiles * a.v_tiles, a.v_tiles, a.tok_tiles);
    if (!walk.valid()) return;
    int vt, tt;
    walk.coords(false, vt, tt);
    auto v_back = [&](int v) { return CHAIN && v == a.v_tiles - 1 ? a.v_shift : 0; };
    auto tok_back = [&](int t) { return CHAIN && t == a.tok_tiles - 1 ? a.tok_shift : 0; };
    auto w_origin = [&](int v) {
        return a.weight + static_cast<int64_t>((v + a.v_tile_lo) * 256 - v_back(v)) * a.H;
    };
    auto h_origin = [&](int t) { return a.hidden + static_cast<int64_t>(t * 256 - tok_back(t)) * a.H; };
    f32x4_t acc[AT::TM][AT::TN];
    if constexpr (CHAIN) {
        char* stage = smem + Dtl::kSmemBytes + wave * kDzStageBytes;
        typename Dtl::Stream st;
        Dtl::begin(st, Operand{w_origin(vt), a.H, 256}, Operand{h_origin(tt), a.H, 256}, a.H, smem);
        for (;;) {
            const bool more = walk.has_next();
            int nvt = vt, ntt = tt;
            if (more) walk.coords(true, nvt, ntt);
            const int vb = v_back(vt);
            zero_acc(acc);
            Dtl::template tile<true>(st, w_origin(nvt), h_origin(ntt), acc, smem);
            if (a.bias != nullptr)  // uniform
                add_bias<AT>(acc, a.bias, (vt + a.v_tile_lo) * 256 - vb + (wave / kWN) * (AT::TM * 16), threadIdx.x & 63);
            mask_rows<T>(acc, (wave / kWN) * (AT::TM * 16), vb, threadIdx.x & 63);
            dz_epilogue<T, GENERAL>(acc, a, vt + a.v_tile_lo, tt, vb, tok_back(tt), stage);
            if (!more) break;
            walk.advance();
            vt = nvt;
            tt = ntt;
        }
        Dtl::end(st);
    } else {
        static_assert(kDzStageBytes * (kThreads / 64) <= Gemm::kSmemBytes, "staging must fit the GEMM's LDS");
        for (;;) {
            const int tok0 = tt * 256, v0 = (vt + a.v_tile_lo) * 256;
            Operand A{w_origin(vt), a.H, min(256, a.v_valid - v0)};
            Operand B{h_origin(tt), a.H, min(256, a.tok_valid - tok0)};
            zero_acc(acc);
            Gemm::run(A, B, a.H, acc, smem);  // ends with a barrier: LDS is free
            if (!GENERAL && a.bias != nullptr)  // uniform
                add_bias<AT>(acc, a.bias, v0 + (wave / kWN) * (AT::TM * 16), threadIdx.x & 63);
            dz_epilogue<T, GENERAL>(acc, a, vt + a.v_tile_lo, tt, 0, 0, smem + wave * kDzStageBytes);
            if (!walk.has_next()) break;
            walk.advance();
            walk.coords(false, vt, tt);
            __syncthreads();  // every wavefront has left its staging patch
        }
    }
}

// dZ from kept logits, in place: the 64 KiB of a slab (64 tokens x 256 vocab rows, see "Kept logits") become the
// 32 KiB of its dZ rows [64][256] of the 16-bit type at the slab's head.  One workgroup per slab reads all of it
// before the first write.  A thread makes 8 consecutive vocab rows of a token from two quads, so eight
// lanes store a full line; the reads are full lines too (8 tokens of one quad row).  Bound by memory: 6
// bytes per logit against the 2 H / 1500e12 s that computing it again takes.
// Tokens outside the tile's own rows get zeros (as far as dW's K steps read, row `used` of the tile), whatever
// lies in the block there.  DB: column sums of the slab go to db_part[slab][v] for d_bias.
struct KeptDzArgs {
    float* kept;
    const int64_t* targets;
    const float* lse;
    const float* grad;
    const float* scales;
    float* db_part;  // [slabs * tok_tiles][v_tiles * 256]
    int slabs;       // of a tile: kept_slabs
    int N;
    int V;
    int v_tiles;
    int tok_tiles;
    int tok_shift;  // rows / vocab rows by which the last token / vocab tile is moved back
    int v_shift;
    int used;       // rows of a padded tile that dW reads (256 otherwise)
    int64_t vocab_start;
    int64_t ignore_index;
    int use_ignore;
    float scale2;
};

template <class T, bool DB>
__global__ __launch_bounds__(256) void linear_logp_dz_kept_kernel(KeptDzArgs a)
{
    const int slab = blockIdx.x, vt = blockIdx.y, tt = blockIdx.z;
    const int tok_back = tt == a.tok_tiles - 1 ? a.tok_shift : 0;
    const int v_back = vt == a.v_tiles - 1 ? a.v_shift : 0;
    const int u = threadIdx.x & 7;  // 8 vocab rows of every group of 64
    float* src = a.kept + ((static_cast<int64_t>(tt) * a.v_tiles + vt) * a.slabs + slab) * kKeptSlab;
    const float gscale = a.scales[0];
    f32x4_t z[2][4][2];
    float gs[2], nlse2[2];
    int hot[2];  // target's vocab row relative to this thread's first one, or out of reach
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int t = (threadIdx.x >> 3) + 32 * q, tl = slab * 64 + t;
        const int n = tt * 256 - tok_back + tl;
        gs[q] = 0.f;
        nlse2[q] = -INFINITY;
        hot[q] = -1;
#pragma unroll
        for (int g = 0; g < 4; ++g) z[q][g][0] = z[q][g][1] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        if (tl >= tok_back && n < a.N) {
            const int64_t tg = a.targets[n];
            if (!(a.use_ignore && tg == a.ignore_index)) {
                gs[q] = a.grad[n] * gscale;
                nlse2[q] = -a.lse[n] * kLog2e;
                const int64_t tv = tg - a.vocab_start;
                if (tv >= static_cast<int64_t>(vt) * 256 && tv < a.V)
                    hot[q] = static_cast<int>(min(tv - (vt * 256 - v_back), static_cast<int64_t>(256)));
                const float* p = src + (t >> 4) * 256 + (t & 15) * 4;
#pragma unroll
                for (int g = 0; g < 4; ++g)
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        // rows 64 g + 8 u + 4 e: wavefront g / 2, MFMA row tile 4 (g % 2) + u / 2, lane group 2 (u % 2) + e
                        const int i = 4 * (g & 1) + (u >> 1), grp = 2 * (u & 1) + e;
                        z[q][g][e] = __builtin_nontemporal_load(reinterpret_cast<const f32x4_t*>(
                            p + (g >> 1) * (kKeptSlab / 2) + i * (4 * 256) + grp * 64));
                    }
            }
        }
    }
    u32x4_t out[2][4];
    float sum[4][8];
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            float d[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float pr = __builtin_amdgcn_exp2f(fmaf(z[q][g][e >> 2][e & 3], a.scale2, nlse2[q]));
                d[e] = fmaf(-gs[q], pr, hot[q] == 64 * g + 8 * u + e ? gs[q] : 0.f);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                out[q][g][e] = T::pack2(d[2 * e], d[2 * e + 1]);
                if (DB) {  // of the rounded values
                    const float lo = T::to_float(static_cast<uint16_t>(out[q][g][e] & 0xffffu));
                    const float hi = T::to_float(static_cast<uint16_t>(out[q][g][e] >> 16));
                    sum[g][2 * e] = q == 0 ? lo : sum[g][2 * e] + lo;
                    sum[g][2 * e + 1] = q == 0 ? hi : sum[g][2 * e + 1] + hi;
                }
            }
        }
    // every logit of the slab has been used before the first write (the arithmetic must not move behind it)
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int g = 0; g < 4; ++g) asm volatile("" : "+v"(out[q][g]));
    __syncthreads();
    uint16_t* dst = reinterpret_cast<uint16_t*>(src);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int t = (threadIdx.x >> 3) + 32 * q;
        if (slab * 64 + t < a.used)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                *reinterpret_cast<u32x4_t*>(dst + t * 256 + g * 64 + u * 8) = out[q][g];
    }
    if constexpr (DB) {
        __shared__ float red[32][257];
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
            for (int e = 0; e < 8; ++e) red[threadIdx.x >> 3][g * 64 + u * 8 + e] = sum[g][e];
        __syncthreads();
        float acc = red[0][threadIdx.x];
#pragma unroll 8
        for (int r = 1; r < 32; ++r) acc += red[r][threadIdx.x];
        a.db_part[(static_cast<int64_t>(tt) * a.slabs + slab) * (a.v_tiles * 256) + vt * 256 + threadIdx.x] = acc;
    }
}

// ------------------------------------------------------------------------------------------- //
// Backward step 2: dH[tok][h] (+)= sum_v dZ[tok][v] W[v][h]      (M = h, N = token, K = vocab)
// ------------------------------------------------------------------------------------------- //
struct DhArgs {
    const uint16_t* dz;      // [tok_tiles*256][ldz]
    const uint16_t* weight;  // piece origin [v][H]
    const float* scales;     // [1] = 1 / loss_scale
    float* acc;              // fp32 partial dH of the chunk [tok_tiles*256][H] (may be null if single)
    uint16_t* out;           // dH chunk origin [tok][H], written when `last`
    int64_t ldz;
    int H;
    int v_valid;
    int tok_valid;
    int tok_tiles;
    int h_tiles;
    int first;  // 1: do not read acc
    int last;   // 1: write the 16-bit output instead of acc
    int ksplit;           // > 1: the vocab range is cut into ksplit parts computed by separate
    float* part;          //      workgroups, each writing its own fp32 slot [ksplit][rows][H]
    int64_t part_stride;  //      (elements per slot); linear_logp_dh_reduce_kernel adds them up
    int nk;               // K steps (of 64 vocab rows) of the piece, the shifted tile's among them;
    KTail tail;           //      0: the block has no shifted tiles, K runs over [0, v_valid)
    int v_tiles;          // KEPT: vocab tiles of the block
    int unit;             // !KEPT: K steps that a part is a multiple of
    int tok_shift;        // rows by which the last token tile is moved back
};

// Epilogue of one dH tile.  The read-modify-write of the running fp32 partial is latency-bound, so
// it runs in two batches (one per pair of 16-token column groups): the 16 reads of a batch are all
// issued before the first use, then added and stored.  FULL (the tile lies inside the chunk and
// inside H): addresses are a uniform tile origin plus a 32-bit lane offset and no predicates are
// needed; otherwise rows and columns are clamped for the reads and predicated for the stores.
// The tile covers hidden columns [h0, h0 + 256) and owns those from h_min on (h_min > h0 for the
// last tile of a persistent walk when H is not a multiple of 256: it is shifted back to end at H
// and must leave the columns of its left neighbour alone).
template <class T, bool FULL, class AT = Acc16>
__device__ inline void dh_epilogue_impl(const f32x4_t (&acc)[AT::TM][AT::TN], const DhArgs& a, int tt,
                                        int h0, int h_min, float* acc_dst, bool first, bool last)
{
    constexpr int TM = AT::TM, TN = AT::TN;
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int wm = wave / kWN, wn = wave % kWN;
    const int tok_min = tt * 256;  // first token row this tile owns
    const int tok0 = tok_min - (!FULL && tt == a.tok_tiles - 1 ? a.tok_shift : 0);
    const float oscale = a.scales[1];
    const int hbase = h0 + wm * (TM * 16) + 4 * (lane >> 4);  // + i * 16
    const uint32_t ldh = static_cast<uint32_t>(a.H);
    // FULL: byte offsets inside the tile stay below 256 * H * 4 (32 bits)
    const int64_t origin = static_cast<int64_t>(tok0) * a.H + h0;
    char* acc_tile = reinterpret_cast<char*>(acc_dst + origin);
    char* out_tile = reinterpret_cast<char*>(a.out + origin);
    const uint32_t lane_el = static_cast<uint32_t>(wn * (TN * 16) + (lane & 15)) * ldh +
                             static_cast<uint32_t>(wm * (TM * 16) + 4 * (lane >> 4));
    constexpr int JB = TN % 2 == 0 ? 2 : 1;
#pragma unroll
    for (int jb = 0; jb < TN; jb += JB) {
        f32x4_t old[JB][TM];
        bool tok_ok[JB];
        int64_t trow[JB];
#pragma unroll
        for (int jj = 0; jj < JB; ++jj) {
            const int j = jb + jj;
            const int tl = tok0 + wn * (TN * 16) + AT::col(j, lane);
            tok_ok[jj] = FULL || (tl >= tok_min && tl < a.tok_valid);
            trow[jj] = static_cast<int64_t>(tok_ok[jj] ? tl : a.tok_valid - 1) * a.H;
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                old[jj][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
                if (!first) {  // uniform
                    if (FULL) {
                        const char* rowp = acc_tile + (static_cast<size_t>(j * 16) * ldh + i * 16) * 4u;
                        old[jj][i] = *reinterpret_cast<const f32x4_t*>(rowp + lane_el * 4u);
                    } else {
                        const int h = hbase + i * 16;
                        old[jj][i] = *reinterpret_cast<const f32x4_t*>(acc_dst + trow[jj] + (h < a.H ? h : 0));
                    }
                }
            }
        }
#pragma unroll
        for (int jj = 0; jj < JB; ++jj) {
            const int j = jb + jj;
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                const int h = hbase + i * 16;
                const f32x4_t v = acc[i][j] + old[jj][i];
                const size_t uni = static_cast<size_t>(j * 16) * ldh + i * 16;  // uniform
                if (FULL || (tok_ok[jj] && h >= h_min && h < a.H)) {  // H % 8 == 0: a quad is all-in or all-out
                    if (last) {
                        u32x2_t pk{T::pack2(v.x * oscale, v.y * oscale), T::pack2(v.z * oscale, v.w * oscale)};
                        if (FULL)
                            *reinterpret_cast<u32x2_t*>(out_tile + uni * 2u + lane_el * 2u) = pk;
                        else
                            *reinterpret_cast<u32x2_t*>(a.out + trow[jj] + h) = pk;
                    } else {
                        if (FULL)
                            *reinterpret_cast<f32x4_t*>(acc_tile + uni * 4u + lane_el * 4u) = v;
                        else
                            *reinterpret_cast<f32x4_t*>(acc_dst + trow[jj] + h) = v;
                    }
                }
            }
        }
    }
}

// Returns whether the tile was full (then every wavefront issued all its stores unconditionally).
template <class T>
__device__ inline bool dh_epilogue(const f32x4_t (&acc)[Acc16::TM][Acc16::TN], const DhArgs& a, int tt, int h0,
                                   int h_min, float* acc_dst, bool first, bool last)
{
    // (a token tile that is moved back is short of 256 rows of its own)
    const bool full = tt * 256 + 256 <= a.tok_valid && h0 + 256 <= a.H && h_min == h0;  // uniform
    if (full)
        dh_epilogue_impl<T, true>(acc, a, tt, h0, h_min, acc_dst, first, last);
    else
        dh_epilogue_impl<T, false>(acc, a, tt, h0, h_min, acc_dst, first, last);
    return full;
}

// One tile (or one vocab part of a tile) per workgroup, for the sizes that the chained walk of
// linear_logp_grads_kernel does not take (H < 256 or not a multiple of 64).
template <class T, int BK>
__global__ __launch_bounds__(kThreads) void linear_logp_dh_kernel(DhArgs a)
{
    using Gemm = TileGemm<T, true, false, BK>;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    f32x4_t acc[Acc16::TM][Acc16::TN];
    int tt, ht, ks = 0;
    xcd_tile(blockIdx.x, a.tok_tiles * a.h_tiles * a.ksplit, a.tok_tiles, a.h_tiles * a.ksplit, 8,
             tt, ht);
    // K range of this workgroup: whole BK-row steps, the first (steps % ksplit) parts take one more
    int k0 = 0, kn = a.v_valid;
    float* acc_dst = a.acc;
    bool first = a.first != 0, last = a.last != 0, empty_part = false;
    if (a.ksplit > 1) {  // uniform
        ks = ht % a.ksplit;
        ht /= a.ksplit;
        const int steps = (a.v_valid + BK - 1) / BK;
        const int base = steps / a.ksplit, extra = steps % a.ksplit;
        const int s0 = ks * base + (ks < extra ? ks : extra);
        const int s1 = s0 + base + (ks < extra ? 1 : 0);
        k0 = s0 * BK;
        kn = min(a.v_valid, s1 * BK) - k0;
        if (kn <= 0) {  // a short last piece can leave a part without K steps: it computes one
            empty_part = true;  // step of the piece's head and discards it
            k0 = 0;
            kn = min(a.v_valid, BK);
        }
        acc_dst = a.part + static_cast<int64_t>(ks) * a.part_stride;
        first = true;
        last = false;
    }
    const int tok0 = tt * 256, h0 = ht * 256;
    Operand A{a.weight + static_cast<int64_t>(k0) * a.H + h0, a.H, min(256, a.H - h0)};
    Operand B{a.dz + static_cast<int64_t>(tok0) * a.ldz + k0, a.ldz, 256};
    zero_acc(acc);
    Gemm::run(A, B, kn, acc, smem);
    if (empty_part) zero_acc(acc);  // uniform: this part's slot must hold zeros
    dh_epilogue<T>(acc, a, tt, h0, h0, acc_dst, first, last);
}

// Sum of the ksplit partial dH slots of one chunk in slot order (plus the running fp32 partial of
// earlier vocab pieces unless `first`), written back as the running partial or, for the last
// piece, as the 16-bit gradient.  One thread per 4 consecutive elements of a row.
template <class T>
__global__ void linear_logp_dh_reduce_kernel(const float* part, int ksplit, int64_t part_stride,
                                             float* acc, uint16_t* out, const float* scales,
                                             int64_t n4, int first, int last)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n4) return;
    f32x4_t v{0.f, 0.f, 0.f, 0.f};
    if (!first) v = reinterpret_cast<const f32x4_t*>(acc)[i];
    for (int k0 = 0; k0 < ksplit; k0 += 8) {  // eight loads in flight, added in slot order
        f32x4_t p[8];
#pragma unroll
        for (int k = 0; k < 8; ++k)
            p[k] = reinterpret_cast<const f32x4_t*>(part + (k0 + k < ksplit ? k0 + k : k0) * part_stride)[i];
#pragma unroll
        for (int k = 0; k < 8; ++k)
            if (k0 + k < ksplit) v += p[k];
    }
    if (last) {
        const float oscale = scales[1];
        u32x2_t pk{T::pack2(v.x * oscale, v.y * oscale), T::pack2(v.z * oscale, v.w * oscale)};
        reinterpret_cast<u32x2_t*>(out)[i] = pk;
    } else {
        reinterpret_cast<f32x4_t*>(acc)[i] = v;
    }
}

// ------------------------------------------------------------------------------------------- //
// Backward step 3: dW[v][h] (+)= sum_tok dZ[tok][v] hidden[tok][h]   (M = h, N = vocab, K = token)
// ------------------------------------------------------------------------------------------- //
struct DwArgs {
    const uint16_t* dz;      // [tok_tiles*256][ldz]
    const uint16_t* hidden;  // chunk origin [tok][H]
    const float* scales;     // [1] = 1 / loss_scale
    float* dw;               // piece origin [v][H] fp32
    int64_t ldz;
    int H;
    int v_valid;
    int tok_valid;
    int v_tiles;
    int h_tiles;
    int accumulate;  // 1: dw += ..., 0: dw = ...
    uint16_t* out;   // piece origin [v][H]: the finished sum leaves in the weight's type, dw is only
                     // read (accumulate); null: the sum goes to dw
    int nk;          // K steps (of 64 tokens) of the chunk, the shifted tile's among them; 0: the block
    KTail tail;      // has no shifted tiles, K runs over [0, tok_valid)
    int v_shift;     // vocab rows by which the last vocab tile is moved back
    int busy, lead;  // joint launch: workgroups with one dH item more than the others, and the rounds of dW
                     // tiles that those others have ahead of them (see LeadWalk)
};

// 16-bit results of four 16-row MFMA tiles of one column: lane group g (16 lanes) holds rows 4 g .. 4 g + 3
// of every tile, p[i] = its quad of tile i.  Afterwards p[0], p[1] are rows 8 g .. 8 g + 7 of the first 32 and
// p[2], p[3] those of the other 32: two rounds of half-swaps over lane groups and registers.  The four groups
// then store 64 consecutive bytes of a row at a time, where quads leave in pieces of 8 bytes, 32 apart
// (64 x 4096 x 128256 forward + backward 1166 -> 1121 us with 16-byte pieces; backward from kept logits 617 ->
// 590 with 64-byte ones), same bits.
__device__ inline void gather_rows(u32x2_t (&p)[4])
{
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        auto swap32 = [&](int a, int b) {  // upper half-wave of p[a] <-> lower half-wave of p[b]
            const auto r = __builtin_amdgcn_permlane32_swap(p[a][c], p[b][c], false, false);
            p[a][c] = r[0];
            p[b][c] = r[1];
        };
        auto swap16 = [&](int a, int b) {  // odd lane groups of p[a] <-> even lane groups of p[b]
            const auto r = __builtin_amdgcn_permlane16_swap(p[a][c], p[b][c], false, false);
            p[a][c] = r[0];
            p[b][c] = r[1];
        };
        swap32(0, 1);
        swap32(2, 3);
        swap16(0, 1);
        swap16(2, 3);
    }
}

// K steps up to which the tiles of a dW launch are written past the L2: with few tokens the launch is bound by its
// stores (backward from kept logits of 64 x 4096 x 128256 590 -> 558 us, 300 x 2048 x 50257 into fp32 291 ->
// 254), from 1000 tokens on the two are the same.  Also for sums that a later chunk of the call adds to: dW of 9000 x
// 2048 x 32768 in blocks of 8 MiB 7.08 ms from the L2, 6.27 past it.  The unchained kernel never streams (CHAIN =
// false; its `nk` of 0 counts nothing): dW of 300 x 2056 x 50257 678 us past the L2, 437 without, 1000 x 1032 x 50257
// 514 and 477, from 4000 tokens on the same.
constexpr int kDwStreamSteps = 8;

// Stores that the epilogue of a full dW tile issues per wavefront, all of them unconditional, the fewer of its
// two forms: 16 bytes per quad of fp32 (TM * TN = 32), 16 bytes per pair of quads of 16-bit results (16).
// The tile loop counts on them (TileGemmDtl::tile, YOUNGER): with one fewer it would take a load of the
// next tile for a store and read a stage that has not landed, so there is no margin in the 16-bit form.
constexpr int kDwPairsPerGroup = 2;  // 16-byte stores of 16-bit results per four quads, see the loop
constexpr int kDwStores = Acc16::TM / 4 * kDwPairsPerGroup * Acc16::TN;
static_assert(kDwStores <= Acc16::TM * Acc16::TN, "the fp32 form stores a quad at a time");

// Epilogue of one dW tile.  Orientation: M (accumulator registers) = hidden column, N (lane) =
// vocab row, so a lane holds 4 consecutive columns of one dW row and the read-modify-write of the
// fp32 tile moves 16 bytes per lane (the four lane groups of a 16 x 16 tile make 64 contiguous
// bytes per row).  It is latency-bound and therefore runs in two batches (one per pair of 16-row
// groups): the 16 reads of a batch are issued before the first use.  FULL (the tile lies inside the
// piece and inside H): a uniform tile origin plus a 32-bit lane offset, no predicates; otherwise
// clamped reads and predicated stores.
// The tile covers hidden columns [h0, h0 + 256) and owns those from h_min on (see dh_epilogue_impl).
template <class T, bool FULL, bool CHAIN>
__device__ inline void dw_epilogue_impl(const f32x4_t (&acc)[Acc16::TM][Acc16::TN], const DwArgs& a, int vt,
                                        int h0, int h_min)
{
    using AT = Acc16;
    constexpr int TM = AT::TM, TN = AT::TN;
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int wm = wave / kWN, wn = wave % kWN;
    const int v_min = vt * 256;  // first vocab row this tile owns
    const int v0 = v_min - (!FULL && vt == a.v_tiles - 1 ? a.v_shift : 0);
    const float oscale = a.scales[1];
    const int hbase = h0 + wm * (TM * 16) + 4 * (lane >> 4);  // + i * 16
    const uint32_t ldw = static_cast<uint32_t>(a.H);
    // FULL: byte offsets inside the tile stay below 256 * H * 4 (32 bits)
    char* tile = reinterpret_cast<char*>(a.dw + static_cast<int64_t>(v0) * a.H + h0);
    const bool stream = CHAIN && a.nk <= kDwStreamSteps;       // uniform
    const int hgrp = h0 + wm * (TM * 16) + 8 * (lane >> 4);  // see gather_rows
    const uint32_t lane_el = static_cast<uint32_t>(wn * (TN * 16) + (lane & 15)) * ldw +
                             static_cast<uint32_t>(wm * (TM * 16) + 4 * (lane >> 4));
#pragma unroll
    for (int jb = 0; jb < TN; jb += 2) {
        f32x4_t old[2][TM];
        bool v_ok[2];
        int64_t vrow[2];
#pragma unroll
        for (int jj = 0; jj < 2; ++jj) {
            const int j = jb + jj;
            const int v = v0 + wn * (TN * 16) + AT::col(j, lane);
            v_ok[jj] = FULL || (v >= v_min && v < a.v_valid);
            vrow[jj] = static_cast<int64_t>(v_ok[jj] ? v : a.v_valid - 1) * a.H;
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                old[jj][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
                if (a.accumulate) {  // uniform
                    if (FULL) {
                        const char* rowp = tile + (static_cast<size_t>(j * 16) * ldw + i * 16) * 4u;
                        old[jj][i] = *reinterpret_cast<const f32x4_t*>(rowp + lane_el * 4u);
                    } else {
                        const int h = hbase + i * 16;
                        old[jj][i] = *reinterpret_cast<const f32x4_t*>(a.dw + vrow[jj] + (h < a.H ? h : 0));
                    }
                }
            }
        }
#pragma unroll
        for (int jj = 0; jj < 2; ++jj) {
            const int j = jb + jj;
            u32x2_t pk[4];
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                const int h = hbase + i * 16;
                const f32x4_t val = acc[i][j] * oscale + old[jj][i];
                const bool mine = FULL || (v_ok[jj] && h >= h_min && h < a.H);  // H % 8 == 0: a quad is all-in or all-out
                const size_t uni = static_cast<size_t>(j * 16) * ldw + i * 16;  // uniform
                if (a.out != nullptr) {  // uniform
                    pk[i & 3] = u32x2_t{T::pack2(val.x, val.y), T::pack2(val.z, val.w)};
                    if ((i & 3) == 3) {
                        gather_rows(pk);
                        uint16_t* row = a.out + vrow[jj];
#pragma unroll
                        for (int q = 0; q < kDwPairsPerGroup; ++q) {
                            const int hq = hgrp + (i - 3) * 16 + 32 * q;  // H, h0, h_min % 8 == 0: all-in or all-out
                            const u32x4_t out{pk[2 * q].x, pk[2 * q].y, pk[2 * q + 1].x, pk[2 * q + 1].y};
                            if (FULL && stream)
                                stream_store(row + hq, 0, out);
                            else if (FULL || (v_ok[jj] && hq >= h_min && hq < a.H))
                                *reinterpret_cast<u32x4_t*>(row + hq) = out;
                        }
                    }
                } else {
                    if (FULL && stream)
                        stream_store(tile + uni * 4u, lane_el * 4u, val);
                    else if (FULL)
                        *reinterpret_cast<f32x4_t*>(tile + uni * 4u + lane_el * 4u) = val;
                    else if (mine)
                        *reinterpret_cast<f32x4_t*>(a.dw + vrow[jj] + h) = val;
                }
            }
        }
    }
}

// Returns whether the tile was full (then every wavefront issued all its stores unconditionally).
template <class T, bool CHAIN>
__device__ inline bool dw_epilogue(const f32x4_t (&acc)[Acc16::TM][Acc16::TN], const DwArgs& a, int vt, int h0,
                                   int h_min)
{
    const bool full = vt * 256 + 256 <= a.v_valid && h0 + 256 <= a.H && h_min == h0;  // uniform
    if (full)
        dw_epilogue_impl<T, true, CHAIN>(acc, a, vt, h0, h_min);
    else
        dw_epilogue_impl<T, false, CHAIN>(acc, a, vt, h0, h_min);
    return full;
}

// The sizes that the chained walk of linear_logp_grads_kernel does not take.
template <class T, int BK>
__global__ __launch_bounds__(kThreads) void linear_logp_dw_kernel(DwArgs a)
{
    using Gemm = TileGemm<T, true, true, BK>;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    TileWalk walk(a.v_tiles * a.h_tiles, a.v_tiles, a.h_tiles);
    if (!walk.valid()) return;
    int vt, ht;
    walk.coords(false, vt, ht);
    f32x4_t acc[Acc16::TM][Acc16::TN];
    for (;;) {
        Operand A{a.hidden + static_cast<int64_t>(ht) * 256, a.H, min(256, a.H - ht * 256)};
        Operand B{a.dz + static_cast<int64_t>(vt) * 256, a.ldz, 256};
        zero_acc(acc);
        Gemm::run(A, B, a.tok_valid, acc, smem);
        dw_epilogue<T, false>(acc, a, vt, ht * 256, ht * 256);
        if (!walk.has_next()) break;
        walk.advance();
        walk.coords(false, vt, ht);
    }
}

// dH and dW of one dZ block in one launch (needs H >= 256 and nk >= 2 of either): they read the same block
// and do not depend on each other, so a workgroup walks its dH tiles through one pipeline and its dW
// tiles through another right behind, and the CUs that the last round of dH tiles leaves idle are at dW
// tiles meanwhile (grads_split).  Two launches each rounded their tile count up to whole rounds.
// Both argument sets are live over the first walk: 22 - 25 spilled vector registers (5 with the narrowest token
// tile; the separate launches had 0 and 5), about 19 scratch accesses a tile outside the K loop, which only
// tiles of few K steps feel.
// h.ksplit > 1: a dH item is one part of the vocab range of a tile and leaves for that part's fp32
// slot.  The items of one range are neighbours in the list (they share dZ columns), so the part
// is the slow index.
// KEPT: dz is the block of kept logits that linear_logp_dz_kept_kernel has turned into dZ in place.
// HT (KEPT): Acc16, or for at most 192 tokens the narrower token tile of dH (bound by reading the weight, as in
// the forward; the bits stay).
template <class T, int BK, bool KEPT, class HT = Acc16>
__global__ __launch_bounds__(kThreads) void linear_logp_grads_kernel(DhArgs h, DwArgs d)
{
    static_assert(KEPT || std::is_same<HT, Acc16>::value, "narrow token tiles are for kept logits");
    constexpr int kSlabEls = kKeptSlab * 2, kTileEls = kept_tile_slabs(HT::TN) * kSlabEls;  // 16-bit elements
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int dh_items = h.tok_tiles * h.h_tiles * h.ksplit;
    if (static_cast<int>(blockIdx.x) < dh_items) {
        using Dtl = TileGemmDtl<T, true, false, BK, kWinDh * HT::TN / 4, true, KEPT, HT>;
        f32x4_t acc[HT::TM][HT::TN];
        TileWalk walk(dh_items, h.tok_tiles, h.h_tiles * h.ksplit);
        // parts are whole K steps, of a block of kept logits (or of one that takes its place) whole vocab tiles
        // (the last one is cut off at nk)
        const int unit = KEPT ? 4 : h.unit;
        const int units = (h.nk + unit - 1) / unit;
        const int base = units / h.ksplit, extra = units % h.ksplit;
        struct Item {
            int tt, ht, ks, step0, nk;
        };
        auto item = [&](bool next) {
            Item it;
            walk.coords(next, it.tt, it.ht);
            it.ks = 0;
            if (h.ksplit > 1) {  // uniform
                it.ks = it.ht / h.h_tiles;
                it.ht -= it.ks * h.h_tiles;
            }
            // the first `extra` parts take one unit more
            it.step0 = (it.ks * base + min(it.ks, extra)) * unit;
            it.nk = min((base + (it.ks < extra ? 1 : 0)) * unit, h.nk - it.step0);
            return it;
        };
        // first hidden column of h tile `t`: the last tile is shifted back so that it ends at H
        auto h_col = [&](int t) { return min(t * 256, h.H - 256); };
        auto w_origin = [&](const Item& it) { return h.weight + static_cast<int64_t>(it.step0) * BK * h.H + h_col(it.ht); };
        auto z_origin = [&](const Item& it) {
            return KEPT ? h.dz + (static_cast<int64_t>(it.tt) * h.v_tiles + it.step0 / 4) * kTileEls
                        : h.dz + static_cast<int64_t>(it.tt) * 256 * h.ldz + it.step0 * BK;
        };
        // kept: rows of 256 elements, 64 of them at the head of a slab
        auto z_operand = [&](const Item& it) {
            return KEPT ? Operand{z_origin(it), 256, 256, (kSlabEls - 64 * 256) * 2, BK * 2, kTileEls * 2}
                        : Operand{z_origin(it), h.ldz, 256};
        };
        auto tail_from = [&](const Item& it) { return h.tail.from - it.step0; };
        Item cur = item(false);
        typename Dtl::Stream st;
        bool counted = false;
        Dtl::begin(st, Operand{w_origin(cur), h.H, 256}, z_operand(cur), cur.nk * BK, smem,
                   KTail{tail_from(cur), h.tail.a, h.tail.b});
        for (;;) {
            const bool more = walk.has_next();
            const Item nxt = more ? item(true) : cur;
            zero_acc(acc);
            Dtl::next_steps(st, nxt.nk, tail_from(nxt));
            // a full tile's epilogue issues TM * TN unconditional stores per wavefront; half is enough
            Dtl::template tile<true, HT::TM * HT::TN / 2>(st, w_origin(nxt), z_origin(nxt), acc, smem, counted);
            const bool part = h.ksplit > 1;
            float* to = part ? h.part + cur.ks * h.part_stride : h.acc;
            if constexpr (HT::TN == Acc16::TN)
                counted = dh_epilogue<T>(acc, h, cur.tt, h_col(cur.ht), cur.ht * 256, to, part || h.first != 0,
                                         !part && h.last != 0);
            else
                dh_epilogue_impl<T, false, HT>(acc, h, cur.tt, h_col(cur.ht), cur.ht * 256, to, part || h.first != 0,
                                               !part && h.last != 0);
            if (!more) break;
            walk.advance();
            cur = nxt;
        }
        Dtl::end(st);
    }
    LeadWalk walk(d.v_tiles * d.h_tiles, d.v_tiles, d.h_tiles, d.busy, d.lead);
    if (!walk.valid()) return;
    using Dtl = TileGemmDtl<T, true, true, BK, kWinDw, true, KEPT>;
    f32x4_t acc[Acc16::TM][Acc16::TN];
    int vt, ht;
    walk.coords(false, vt, ht);
    auto h_col = [&](int t) { return min(t * 256, d.H - 256); };
    auto h_origin = [&](int t) { return d.hidden + h_col(t); };                                         // M rows
    auto z_origin = [&](int v) { return d.dz + static_cast<int64_t>(v) * (KEPT ? kTileEls : 256); };  // N rows
    // kept: a K step is the head of one slab of 64 tokens
    const Operand z = KEPT ? Operand{z_origin(vt), 256, 256, 0, kSlabEls * 2,
                                     static_cast<int64_t>(d.v_tiles) * kTileEls * 2}
                           : Operand{z_origin(vt), d.ldz, 256};
    typename Dtl::Stream st;
    bool counted = false;
    Dtl::begin(st, Operand{h_origin(ht), d.H, 256}, z, d.nk * BK, smem, d.tail);
    for (;;) {
        const bool more = walk.has_next();
        int nvt = vt, nht = ht;
        if (more) walk.coords(true, nvt, nht);
        zero_acc(acc);
        Dtl::template tile<true, kDwStores>(st, h_origin(nht), z_origin(nvt), acc, smem, counted);
        counted = dw_epilogue<T, true>(acc, d, vt, h_col(ht), ht * 256);
        if (!more) break;
        walk.advance();
        vt = nvt;
        ht = nht;
    }
    Dtl::end(st);
}

// Fewer tokens than a tile: the rows of `hidden`, the last one repeated up to row `used`, rows of zeros up to
// one 256-row tile, so that dZ and dW run on the full-tile pipeline (at most 256 x H x 2 bytes, a few us
// against the register-staged loop that a K tail of the whole dW contraction would need: 12 to 20 % of a
// backward at 160 tokens).
// dZ evaluates a row past the end against the last token's log-sum-exp and a zero upstream gradient.  The K
// steps of dW read such rows up to `used`: they have to hold that token's logits, a probability of at
// most 1 times 0.  (Rows of zeros have logits of 0 or the bias; against a log-sum-exp below -88 their
// probability is inf and dZ NaN.)  From `used` on nobody reads dZ, and zeros draw the least power in the
// products: backward of 64 x 4096 x 128256 890 us with copies up to the tile's end, 884 so, 882 with zeros alone.
// One row per blockIdx.y, 16 bytes per thread.
__global__ void linear_logp_pad_rows_kernel(const uint16_t* src, uint16_t* dst, int n_rows, int used, int row8)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= row8) return;
    const int64_t row = blockIdx.y, from = row < n_rows ? row : n_rows - 1;
    reinterpret_cast<u32x4_t*>(dst)[row * row8 + i] =
        row < used ? reinterpret_cast<const u32x4_t*>(src)[from * row8 + i] : u32x4_t{0u, 0u, 0u, 0u};
}

// db[v] (+)= sum_tok dZ[tok][v] in two fixed-order levels.  Level 1: one workgroup per (256
// columns) x (256-token tile); a thread owns 8 columns (one 16-byte load per row) of every eighth
// row, the eight row groups are added in order through LDS: part[tile][v].  The dZ block is written
// in whole tiles (rows and columns that nobody owns hold zeros), so no column check is needed here;
// `rows` is 256 but for a padded tile, whose rows past the tokens are left out.
template <class T>
__global__ __launch_bounds__(256) void linear_logp_db_partial_kernel(const uint16_t* dz, int64_t ldz, int rows,
                                                                     float* part, int64_t part_ld)
{
    __shared__ float red[8][256];
    const int cg = threadIdx.x & 31, rg = threadIdx.x >> 5;
    const int v0 = blockIdx.x * 256 + cg * 8;
    const uint16_t* p = dz + (static_cast<int64_t>(blockIdx.y) * 256 + rg) * ldz + v0;
    float sum[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    const int steps = (rows - rg + 7) >> 3;
#pragma unroll 4
    for (int k = 0; k < steps; ++k) {
        const u32x4_t w = *reinterpret_cast<const u32x4_t*>(p + static_cast<int64_t>(k) * 8 * ldz);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            sum[2 * e] += T::to_float(static_cast<uint16_t>(w[e] & 0xffffu));
            sum[2 * e + 1] += T::to_float(static_cast<uint16_t>(w[e] >> 16));
        }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) red[rg][cg * 8 + e] = sum[e];
    __syncthreads();
    float acc = red[0][threadIdx.x];
#pragma unroll
    for (int r = 1; r < 8; ++r) acc += red[r][threadIdx.x];
    part[static_cast<int64_t>(blockIdx.y) * part_ld + blockIdx.x * 256 + threadIdx.x] = acc;
}

// Level 1 of a block that takes the place of kept logits: sums per slab of 64 tokens in the order of
// linear_logp_dz_kept_kernel (rows r and r + 32, then r ascending).  One column per thread.
template <class T>
__global__ __launch_bounds__(256) void linear_logp_db_slab_kernel(const uint16_t* dz, int64_t ldz, int rows, float* part,
                                                                  int64_t part_ld)
{
    const int col = blockIdx.x * 256 + threadIdx.x, first = (blockIdx.y & 3) * 64;
    const uint16_t* p = dz + static_cast<int64_t>(blockIdx.y) * 64 * ldz + col;
    float acc = 0.f;
#pragma unroll 8
    for (int r = 0; r < 32; ++r) {
        const float lo = first + r < rows ? T::to_float(p[r * ldz]) : 0.f;
        const float hi = first + r + 32 < rows ? T::to_float(p[(r + 32) * ldz]) : 0.f;
        acc = r == 0 ? lo + hi : acc + (lo + hi);
    }
    part[blockIdx.y * part_ld + col] = acc;
}

// Level 2: the token tiles (slabs) of the block in ascending order, times 1 / loss_scale.
// v_shift: the last vocab tile's columns start that many vocab rows earlier than its place says.
__global__ void linear_logp_db_finish_kernel(const float* part, int64_t part_ld, int tok_tiles, int v_valid,
                                             int v_shift, const float* scales, float* db, int accumulate)
{
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= v_valid) return;
    const int c = v < v_valid / 256 * 256 ? v : v + v_shift;
    float sum = part[c];
#pragma unroll 8
    for (int t = 1; t < tok_tiles; ++t) sum += part[static_cast<int64_t>(t) * part_ld + c];
    sum *= scales[1];
    db[v] = accumulate ? db[v] + sum : sum;
}

// scales[0] = loss_scale / T, scales[1] = 1 / loss_scale.  For f16 the loss scale is the power of
// two that brings max|g|/T to about 2^12 so that tiny probabilities survive the f16 dZ; bf16 uses 1.
__global__ void linear_logp_scales_kernel(const float* grad, int n, float inv_temperature,
                                          int dtype, float* scales)
{
    __shared__ float red[1024];
    float mx = 0.f;
    if (dtype == 1) {
        for (int i = threadIdx.x; i < n; i += blockDim.x) {
            const float g = fabsf(grad[i]);
            if (g == g && g != INFINITY) mx = fmaxf(mx, g);
        }
    }
    red[threadIdx.x] = mx;
    __syncthreads();
    for (unsigned o = blockDim.x / 2; o > 0; o >>= 1) {
        if (threadIdx.x < o) red[threadIdx.x] = fmaxf(red[threadIdx.x], red[threadIdx.x + o]);
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        float ls = 1.f;
        if (dtype == 1) {
            const float top = red[0] * inv_temperature;
            if (top > 0.f) {
                int e;
                frexpf(top, &e);  // top = f * 2^e, f in [0.5, 1)
                int shift = 12 - e;
                shift = shift < -24 ? -24 : (shift > 60 ? 60 : shift);
                ls = ldexpf(1.f, shift);
            }
        }
        scales[0] = ls * inv_temperature;
        scales[1] = 1.f / ls;
    }
}

}  // namespace rlk

// ------------------------------------------------------------------------------------------- //
// C ABI
// ------------------------------------------------------------------------------------------- //
using namespace rlk;

namespace {

constexpr int kBK = RLK_BK;

// Forward launch plan: a pure function of (N, H, V, which kernels run).
//   fast launch   : vocab tiles split n_fast ways: all of them when the chained walk runs (it moves a
//                   ragged last tile back), otherwise the full ones
//   general launch: the ragged last tile of the other sizes (all tiles for the fp32 kernels), n_gen ways
struct FwdPlan {
    int row_blocks;
    int patch_rows;
    int fast_tiles, n_fast;
    int gen_tiles, n_gen;
    int total_splits;
};

// Token blocks per XCD patch.  The 32 workgroups resident on one XCD cover patch_rows token blocks
// x 32 / patch_rows vocab splits; the hidden blocks of all eight patches in flight (8 x patch_rows
// x 256 x H x 2 bytes) are re-read for every vocab tile and should stay inside the 256 MB
// memory-side cache next to the weight tiles: 8 blocks up to H = 4096, 4 up to 8192, 2 beyond
// (measured at H = 8192 with 16384 tokens and more: 8 blocks 1268 TFLOP/s).
int patch_rows_for(int H)
{
    return H <= 4096 ? 8 : (H <= 8192 ? 4 : 2);
}

// Vocab splits of one forward launch.  The launch is row_blocks x splits workgroups, one per CU at
// a time, each walking ceil(tiles / splits) vocab tiles: it takes ceil(workgroups / 256) rounds of
// the 256 CUs, so a count that lands just above a multiple of 256 wastes most of a round (88 token
// blocks x 6 splits = 528 workgroups ran three rounds for the work of two: 976 instead of 1370
// TFLOP/s).  The count with the lowest rounds x (run + half a tile of start-up and state flush)
// wins, a smaller one when it is within 1.5 %, among the counts that leave every workgroup a run of
// at least 8 tiles and keep the split partials (12 bytes per token and split) within the 8 MiB the
// allocation-free entry point has; measured over 4 - 32 splits at 48 - 243 token blocks, this
// choice is within 1.5 % of the best count tried.  From 64 tiles on shorter runs are taken too as long as
// the launch does not fill one round of the chip: one block of 160 tokens x 501 tiles at H = 4096 ran 62
// workgroups of 8 - 9 tiles in 741 us and runs 251 of two in 250 us.  Below 64 tiles the runs of 8 stay, so
// that a batch and its micro-batches sum in one grouping and give the same bits: whatever their sizes up
// to 14 tiles (V <= 3584, one run per token block), up to 8192 tokens above.  (One tile per workgroup in
// launches of up to 32 tiles took 200 x 64 x 3000 log-probs from 88 to 42 us and forward + backward of 160 x
// 4096 x 8192 from 866 to 260, but grouped by the token count.)
int split_count(int row_blocks, int tiles, int patch_rows)
{
    if (tiles <= 0) return 0;
    // At least 32 / patch_rows splits when each still gets a long run of tiles: the 32 workgroups
    // resident on one XCD then form a compact (token blocks x splits) patch that fetches 12 distinct
    // operand streams into its L2 (8 x 4 or 4 x 8) instead of 18 (16 x 2) or 33 (32 x 1); with 243
    // token blocks, 2 or 3 splits ran at 1160 - 1190 TFLOP/s where 4 ran at 1383.
    const int want = 32 / patch_rows;
    const int lo = tiles >= want * 16 ? want : 1;
    const int most = row_blocks < 4 ? 256 / row_blocks : 64;
    int hi = tiles < most ? tiles : most;
    const int64_t fit = static_cast<int64_t>(RLK_STATIC_SCRATCH_BYTES) / (3072LL * row_blocks);
    if (hi > fit) hi = fit > lo ? static_cast<int>(fit) : lo;
    int best = lo;
    int64_t best_cost = -1;
    for (int s = lo; s <= hi; ++s) {
        const int64_t run = (tiles + s - 1) / s;
        if (s > lo && run < 8 && (tiles < 64 || static_cast<int64_t>(row_blocks) * s > 256)) break;
        const int64_t rounds = (static_cast<int64_t>(row_blocks) * s + 255) / 256;
        const int64_t cost = rounds * (2 * run + 1);
        // a larger count has to be 1.5 % better than the best smaller one to replace it
        if (best_cost < 0 || cost * 1000 < best_cost * 985) {
            best = s;
            best_cost = cost;
        }
    }
    return best;
}

// Sizes whose vocab tiles all run through the forward's one pipeline.
bool fwd_chained(int H, int64_t V) { return H % kBK == 0 && H >= 2 * kBK && V >= 256; }

FwdPlan fwd_plan(int64_t N, int H, int64_t V, bool all_general)
{
    FwdPlan p;
    p.row_blocks = static_cast<int>((N + 255) / 256);
    p.patch_rows = patch_rows_for(H);
    const int all = static_cast<int>((V + 255) / 256);
    const int full = static_cast<int>(V / 256);
    p.fast_tiles = all_general ? 0 : (fwd_chained(H, V) ? all : full);
    p.gen_tiles = all - p.fast_tiles;
    p.n_fast = split_count(p.row_blocks, p.fast_tiles, p.patch_rows);
    p.n_gen = split_count(p.row_blocks, p.gen_tiles, p.patch_rows);
    p.total_splits = p.n_fast + p.n_gen;
    return p;
}

inline size_t align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

// One dZ block is at least one 256 x 256 tile and at most RLK_MAX_DZ_BUDGET bytes: the tile
// loaders address rows inside a tile with 32-bit byte offsets (256 rows x leading dimension), so
// the leading dimension of the block must stay below 2^23 elements.
inline size_t clamp_dz_budget(size_t budget)
{
    if (budget == 0) budget = RLK_DEFAULT_DZ_BUDGET;
    if (budget < 131072) budget = 131072;
    if (budget > RLK_MAX_DZ_BUDGET) budget = RLK_MAX_DZ_BUDGET;
    return budget;
}

struct BwdPlan {
    int tok_chunk;   // tokens per chunk (multiple of 256)
    int v_piece;     // vocab rows per piece (multiple of 256)
    int n_chunks;
    int n_pieces;
    int ksplit;      // dH launch of a full block: parts of the piece's vocab range computed side by
                     // side; a shorter last chunk / last piece takes its own count (dh_parts)
    int64_t ldz;     // elements between consecutive token rows of the dZ block
    size_t dz_bytes;
    size_t acc_bytes;
    size_t part_bytes;
    size_t db_bytes;
    size_t pad_bytes;  // rows of one token tile when there are fewer tokens than that
    bool whole;        // kept_plan: dH parts in whole vocab tiles, d_bias by slabs of 64 tokens
    size_t scales_off, dz_off, acc_off, part_off, db_off, pad_off, total;
};

// Cost of the three launches of one dZ block of ct x pt tiles, in K steps of one CU: a launch of
// t tiles occupies ceil(t / 256) rounds of the 256 CUs, a tile costs its K steps plus an epilogue.
// Measured on MI355X with wall-clock stamps inside the kernels, one K step (256 x 256 x 64) takes
// about 1.56 us in all three kernels; the dZ epilogue (exp + 16-bit store) 4.4 us = 3 steps, the
// fp32 read-modify-write of a dH or dW tile 13 - 14 us = 9 steps.
// Few tokens or a narrow hidden dimension: a dH launch of at most 128 tiles over a long vocab range
// is cut into parts that run side by side (fp32 slots, added up in slot order afterwards).
inline int dh_parts(int64_t ct, int64_t pt, int64_t ht)
{
    const int64_t tiles = ct * ht;
    int parts = 1;
    if (tiles <= 128 && pt >= 32) {
        int64_t lim = 256 / tiles;
        if (lim > pt / 16) lim = pt / 16;
        if (lim > 8) lim = 8;
        while (parts * 2 <= lim) parts *= 2;
    }
    return parts;
}

// What a split dH launch really cuts its vocab range into (the plan below prices and reports dh_parts, a
// lower bound): as many parts as give every CU a tile (at
// least 16 K steps each; their slots stay within 256 tiles of fp32).  The powers of two above left the
// launch on 64 to 192 CUs: 64 x 2048 x 32000 318 -> 239, 64 x 4096 x 128256
// 1306 -> 1168, 1000 x 1536 x 151936 1910 -> 1838 us a pass.
inline int dh_cuts(int64_t ct, int64_t pt, int64_t ht)
{
    const int parts = dh_parts(ct, pt, ht);
    if (parts == 1) return 1;
    int64_t cuts = 256 / (ct * ht);
    if (cuts > pt / 4) cuts = pt / 4;
    if (cuts > 32) cuts = 32;
    return cuts > parts ? static_cast<int>(cuts) : parts;
}

// Epilogues of linear_logp_grads_kernel in K steps, from launches whose tiles fill whole rounds (256 vocab tiles
// x 4096 x 8192 tokens: dH 400 us for 256 steps, dW with the fp32 read-modify-write 212 us for 128; 1024
// tokens x 4096: dW written once in 16 bits 34.5 us for 16; a step is 1.45 - 1.5 us).
constexpr int kDhSteps = 10, kDwSteps = 8, kDwAddSteps = 14;

// How linear_logp_grads_kernel hands out n1 dH items of cost c1 and n2 dW tiles of cost c2 (K steps) to `grid`
// workgroups: dH items in rounds, so the first n1 % grid workgroups (`busy`, in whole groups of the eight
// XCDs) have one more than the others; those others take `lead` rounds of dW tiles among themselves before
// the common rounds, as many as make the longest walk (`cost`) shortest.
struct GradsSplit {
    int busy = 0, lead = 0;
    int64_t cost = 0;
};
inline GradsSplit grads_split(int64_t n1, int64_t c1, int64_t n2, int64_t c2, int64_t grid)
{
    GradsSplit best;
    const int64_t full = n1 / grid, over = n1 % grid;
    int64_t busy = over;
    if (grid % 8 == 0) busy = (over + 7) / 8 * 8;
    const int64_t rest = grid - busy;  // 0: all but at most seven workgroups have the extra item
    const int64_t most = rest > 0 && c1 > 0 ? std::min(c1 / c2 + 1, (n2 + rest - 1) / rest) : 0;
    for (int64_t lead = 0; lead <= most; ++lead) {
        const int64_t left = std::max<int64_t>(0, n2 - lead * rest), rounds = (left + grid - 1) / grid;
        const int64_t last = left - (rounds - 1) * grid;  // tiles of the last common round: the others come first
        const int64_t slow = (full + (over > 0)) * c1 + (last > rest ? rounds : std::max<int64_t>(0, rounds - 1)) * c2;
        const int64_t fast = rest > 0 ? full * c1 + (lead + rounds) * c2 : 0;
        const int64_t cost = busy > 0 ? std::max(slow, fast) : fast;
        if (lead == 0 || cost < best.cost) best = GradsSplit{static_cast<int>(busy), static_cast<int>(lead), cost};
    }
    return best;
}

// The dH + dW launch of one block of ct x pt tiles, in K steps (the reduction of split dH tiles included);
// several: dW is read, added to and written by every token chunk.
inline int64_t grads_cost(int64_t ct, int64_t pt, int64_t ht, bool several)
{
    const int cuts = dh_cuts(ct, pt, ht);
    return grads_split(ct * ht * cuts, (4 * pt + cuts - 1) / cuts + kDhSteps, pt * ht,
                       4 * ct + (several ? kDwAddSteps : kDwSteps), 256).cost + (cuts > 1 ? 10 : 0);
}

// Sizes whose backward runs on the chained walks whatever the token count (ragged tiles are moved back).
bool bwd_chained(int H, int64_t V) { return H % kBK == 0 && H >= 256 && V >= 256; }

inline int64_t block_cost(int64_t ct, int64_t pt, int64_t ht, int64_t hk)
{
    const int64_t dz = (ct * pt + 255) / 256 * (hk + 3);
    const int parts = dh_parts(ct, pt, ht);
    // split launch: every part is a workgroup of its own; the slot reduction costs about 10 steps
    const int64_t dh = parts > 1 ? (ct * ht * parts + 255) / 256 * (4 * pt / parts + 9) + 10
                                 : (ct * ht + 255) / 256 * (4 * pt + 9);
    const int64_t dw = (pt * ht + 255) / 256 * (4 * ct + 9);
    return dz + dh + dw;
}

// The same with dH and dW in one launch (chained sizes).
inline int64_t joint_block_cost(int64_t ct, int64_t pt, int64_t ht, int64_t hk, bool several)
{
    const int64_t dz = (ct * pt + 255) / 256 * (hk + 3);
    return dz + grads_cost(ct, pt, ht, several) + 12;  // filling three pipelines, two launches
}

// Token chunks x vocab pieces such that one dZ block stays within `budget` bytes and block plus
// fp32 dH accumulator within 1.5 x budget.  Among the shapes that fit, the one with the lowest
// modelled time wins: tile counts just above a multiple of 256 waste most of a round, and small
// blocks pay the read-modify-write epilogues more often.  Sizes whose dH and dW share a launch are priced both
// ways, and the blocks that three launches would want stay unless the joint price has others at
// least 2.5 % below them: over 30 sizes (896 <= H <= 8192, 1124 - 24960 tokens) the clock gave 1 - 19 % where the model
// promised more than that (two exceptions at 0 and 1 %), and 0.976 - 1.023, 1.001 on average, where it
// promised less, with every sum grouped another way for it.
BwdPlan bwd_plan(int64_t N, int H, int64_t V, size_t budget)
{
    struct Key {
        int64_t N, V;
        int H;
        size_t budget;
        BwdPlan plan;
    };
    static thread_local Key memo{0, 0, 0, 0, {}};
    if (memo.N == N && memo.V == V && memo.H == H && memo.budget == budget) return memo.plan;

    const int64_t n_t = (N + 255) / 256, v_t = (V + 255) / 256;
    const int64_t ht = (H + 255) / 256, hk = (H + kBK - 1) / kBK;
    const bool chained = bwd_chained(H, V);
    const int64_t tile_bytes = 131072;                          // 256 x 256 16-bit
    const int64_t max_tiles = static_cast<int64_t>(budget) / tile_bytes;
    const int64_t cap = static_cast<int64_t>(budget) + static_cast<int64_t>(budget) / 2;

    // candidate sizes: balanced splits ceil(x / k) and multiples of 8 tiles
    auto candidates = [](int64_t x, std::vector<int64_t>& out) {
        for (int64_t k = 1; k <= x; ++k) {
            const int64_t c = (x + k - 1) / k;
            if (out.empty() || out.back() != c) out.push_back(c);
        }
        for (int64_t c = 8; c <= x; c += 8) out.push_back(c);
    };
    std::vector<int64_t> cts, pts;
    candidates(n_t, cts);
    candidates(v_t, pts);

    struct Best {
        int64_t ct = 1, pt = 1, cost = -1, bytes = 0, joint = 0;
    };
    Best sep, joint;
    for (int64_t ct : cts) {
        if (ct > max_tiles) continue;
        const int64_t nc = (n_t + ct - 1) / ct, ct_last = n_t - (nc - 1) * ct;
        for (int64_t pt : pts) {
            if (ct * pt > max_tiles) continue;
            const int64_t np = (v_t + pt - 1) / pt, pt_last = v_t - (np - 1) * pt;
            const int64_t bytes = ct * pt * tile_bytes + (np > 1 ? ct * 256 * H * 4 : 0);
            if (bytes > cap && ct * pt > 1) continue;
            auto all = [&](auto price) {
                return (nc - 1) * (np - 1) * price(ct, pt) + (np - 1) * price(ct_last, pt) +
                       (nc - 1) * price(ct, pt_last) + price(ct_last, pt_last);
            };
            const int64_t sep_cost = all([&](int64_t c, int64_t v) { return block_cost(c, v, ht, hk); });
            const int64_t joint_cost =
                chained ? all([&](int64_t c, int64_t v) { return joint_block_cost(c, v, ht, hk, nc > 1); }) : 0;
            auto keep_if_better = [&](Best& best, int64_t cost) {
                if (best.cost < 0 || cost < best.cost || (cost == best.cost && bytes < best.bytes))
                    best = Best{ct, pt, cost, bytes, joint_cost};
            };
            keep_if_better(sep, sep_cost);
            keep_if_better(joint, joint_cost);
        }
    }
    const Best& best = chained && joint.cost * 1025 < sep.joint * 1000 ? joint : sep;
    const int64_t best_ct = best.ct, best_pt = best.pt;

    BwdPlan p{};
    p.tok_chunk = static_cast<int>(best_ct) * 256;
    p.v_piece = static_cast<int>(best_pt) * 256;
    p.n_chunks = static_cast<int>((n_t + best_ct - 1) / best_ct);
    p.n_pieces = static_cast<int>((v_t + best_pt - 1) / best_pt);
    p.ldz = p.v_piece;
    p.dz_bytes = static_cast<size_t>(p.tok_chunk) * p.ldz * 2;
    p.acc_bytes = p.n_pieces > 1 ? static_cast<size_t>(p.tok_chunk) * H * 4 : 0;
    p.scales_off = 0;
    p.dz_off = 256;
    p.acc_off = p.dz_off + align_up(p.dz_bytes, 256);
    // Few tokens: the dH launch has fewer tiles than the chip has CUs but a long vocab range, so
    // the range is cut into parts that run side by side and are added up in a fixed order.
    p.ksplit = dh_parts(best_ct, best_pt, ht);
    // fp32 slots of the split dH launches: every (chunk, piece) kind picks its own part count, so
    // a short last chunk does not run its few tiles on a quarter of the chip
    const int64_t ct_last = n_t - (p.n_chunks - 1) * best_ct, pt_last = v_t - (p.n_pieces - 1) * best_pt;
    p.part_bytes = 0;
    for (int64_t ct : {best_ct, ct_last})
        for (int64_t pt : {best_pt, pt_last}) {
            const int parts = dh_cuts(ct, pt, ht);
            if (parts > 1)
                p.part_bytes = std::max(p.part_bytes, static_cast<size_t>(parts) * ct * 256 * H * 4);
        }
    p.part_off = p.acc_off + align_up(p.acc_bytes, 256);
    // per-token-tile column sums of the dZ block (d_bias): 1 KiB per dZ tile
    p.db_bytes = static_cast<size_t>(best_ct) * p.v_piece * 4;
    p.db_off = p.part_off + align_up(p.part_bytes, 256);
    p.pad_bytes = N < 256 ? static_cast<size_t>(256) * H * 2 : 0;
    p.pad_off = p.db_off + align_up(p.db_bytes, 256);
    p.total = p.pad_off + align_up(p.pad_bytes, 256);
    memo = Key{N, V, H, budget, p};
    return p;
}

// Bytes of the kept logits, or 0 where a training forward keeps none: sizes off the chained 16-bit kernels, and
// more than RLK_KEPT_LOGITS_BYTES, the bound that keeps the extra memory of a call below 1 GB whatever N is (a choice,
// about three of the dZ blocks that a larger call has in its backward; the ops hold all live calls of a device to it).
// In whole tiles; fewer than 192 tokens need less of it (kept_least).
// Narrow heads keep none either: a tile of logits costs 4 - 10 us of stores in the forward and 17 us of dZ pass
// (proportionally less with fewer than 256 tokens, whose columns past N stay out), computing it again
// about 1.7 us per 64 of H plus 4 (forward + backward, kept against computed again: 1305 x 896 x 32768 400 against
// 457 us, 325 x 896 x 50257 264 against 323, 2856 x 768 x 32768 636 against 625).
size_t kept_bytes(int64_t N, int H, int64_t V, int dtype)
{
    if (dtype == RLK_DTYPE_F32) return wide_kept_bytes(N, H, V);
    if (!bwd_chained(H, V) || H < std::min<int64_t>(896, 4 * N)) return 0;
    const int64_t tiles = ((N + 255) / 256) * ((V + 255) / 256);
    if (tiles > static_cast<int64_t>(RLK_KEPT_LOGITS_BYTES / (kKeptTile * 4))) return 0;
    return static_cast<size_t>(tiles) * kKeptTile * 4;
}

// What a buffer has to have of kept_bytes: 66 of 131 MB at 128 x 128256.
size_t kept_least(int64_t N, int H, int64_t V, int dtype)
{
    const size_t whole = kept_bytes(N, H, V, dtype);
    return dtype == RLK_DTYPE_F32 ? whole : whole / 4 * kept_slabs(N);
}

// Backward from kept logits: one block of the whole problem, dZ in the place of the logits.  again: none were kept
// (or they are used up); dZ is computed into the workspace, 2 bytes a logit, and every sum is grouped as with them.
BwdPlan kept_plan(int64_t N, int H, int64_t V, bool again)
{
    const int64_t n_t = (N + 255) / 256, v_t = (V + 255) / 256, ht = (H + 255) / 256;
    BwdPlan p{};
    p.tok_chunk = static_cast<int>(n_t) * 256;
    p.v_piece = static_cast<int>(v_t) * 256;
    p.n_chunks = p.n_pieces = 1;
    p.whole = true;
    p.ldz = p.v_piece;
    p.ksplit = dh_cuts(n_t, v_t, ht);
    p.dz_off = 256;
    p.dz_bytes = again ? static_cast<size_t>(n_t) * v_t * 131072 : 0;
    p.part_off = p.dz_off + p.dz_bytes;
    p.part_bytes = p.ksplit > 1 ? static_cast<size_t>(p.ksplit) * n_t * 256 * H * 4 : 0;
    p.db_off = p.part_off + align_up(p.part_bytes, 256);
    p.db_bytes = static_cast<size_t>(4) * n_t * p.v_piece * 4;  // column sums per slab of 64 tokens
    p.pad_off = p.db_off + align_up(p.db_bytes, 256);
    p.pad_bytes = N < 256 ? static_cast<size_t>(256) * H * 2 : 0;
    p.total = p.pad_off + align_up(p.pad_bytes, 256);
    return p;
}

// Raises the dynamic-LDS limit of `kernel` to `bytes` on the current device.  The attribute is
// per device and sticks, so each (kernel instance, device) pair pays the runtime call once.
template <auto kernel>
int set_smem(int bytes)
{
    constexpr int kMaxDev = 64;
    static std::mutex mu;
    static int done[kMaxDev] = {};  // one table per template instance = per kernel
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return rlk_fail(RLK_ERR_LAUNCH, hipGetErrorString(e));
    const bool tracked = dev >= 0 && dev < kMaxDev;
    if (tracked) {
        std::lock_guard<std::mutex> lock(mu);
        if (done[dev] >= bytes) return 0;
    }
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                            hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) return rlk_fail(RLK_ERR_LAUNCH, hipGetErrorString(e));
    if (tracked) {
        std::lock_guard<std::mutex> lock(mu);
        if (done[dev] < bytes) done[dev] = bytes;
    }
    return 0;
}

int check_launch(const char* what)
{
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return rlk_fail(RLK_ERR_LAUNCH, what);
    return 0;
}

int check_common(int64_t N, int32_t H, int64_t V, int dtype)
{
    if (dtype != RLK_DTYPE_BF16 && dtype != RLK_DTYPE_F16 && dtype != RLK_DTYPE_F32)
        return rlk_fail(RLK_ERR_UNSUPPORTED, "dtype must be RLK_DTYPE_BF16, RLK_DTYPE_F16 or RLK_DTYPE_F32");
    if (N <= 0 || H <= 0 || V <= 0) return rlk_fail(RLK_ERR_ARG, "N, H and V must be positive");
    if (N > 0x7fff0000LL || V > 0x7fff0000LL) return rlk_fail(RLK_ERR_ARG, "N or V too large");
    if (H > (1 << 20)) return rlk_fail(RLK_ERR_UNSUPPORTED, "hidden size above 2^20");
    return 0;
}

// The 16-bit MFMA tiles take bf16 / f16 inputs whose rows start on 16-byte boundaries; everything
// else runs on the fp32 matrix-core kernels (rlk_wide.hip).
bool use_mfma(const void* hidden, const void* weight, int32_t H, int dtype)
{
    return (dtype == RLK_DTYPE_BF16 || dtype == RLK_DTYPE_F16) && H % 8 == 0 &&
           (reinterpret_cast<uintptr_t>(hidden) & 15) == 0 && (reinterpret_cast<uintptr_t>(weight) & 15) == 0;
}

// A buffer for kept logits as the forward or the backward is given it (null: the backward computes them again).
int check_kept(const void* kept, size_t bytes, bool mfma, int64_t N, int32_t H, int64_t V, int dtype)
{
    const size_t need = kept_least(N, H, V, dtype);
    if ((!mfma && dtype != RLK_DTYPE_F32) || need == 0)
        return rlk_fail(RLK_ERR_UNSUPPORTED, "no logits are kept for these sizes (rlk_linear_logp_kept_bytes)");
    if (kept != nullptr && (bytes < need || (reinterpret_cast<uintptr_t>(kept) & 15) != 0))
        return rlk_fail(RLK_ERR_ARG, "kept logits: buffer too small or not 16-byte aligned");
    return 0;
}

// Compute units of the current device (looked up once per device): the chained kernels launch
// one workgroup per compute unit.  Which workgroup computes a tile never changes the tile's bits.
int compute_units(int* out)
{
    constexpr int kMaxDev = 64;
    static std::mutex mu;
    static int cached[kMaxDev] = {};
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return rlk_fail(RLK_ERR_LAUNCH, hipGetErrorString(e));
    if (dev < 0 || dev >= kMaxDev) return rlk_fail(RLK_ERR_UNSUPPORTED, "device index too large");
    std::lock_guard<std::mutex> lock(mu);
    if (cached[dev] == 0) {
        int n = 0;
        e = hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev);
        if (e != hipSuccess || n <= 0) return rlk_fail(RLK_ERR_LAUNCH, "cannot read the compute-unit count");
        cached[dev] = n;
    }
    *out = cached[dev];
    return 0;
}

struct BwdCall {
    const float* grad_logp;
    const void* hidden;
    const void* weight;
    const float* bias;
    const int64_t* targets;
    const float* lse;
    void* d_hidden;
    float* d_weight;
    float* d_bias;
    void* workspace;
    int64_t N;
    int32_t H;
    int64_t V;
    int64_t vocab_start;
    int32_t dtype;
    float temperature;
    int64_t ignore_index;
    int32_t use_ignore;
    hipStream_t stream;
    int accumulate;  // 1: d_weight / d_bias already hold the sums of earlier tokens, add to them
    void* d_weight_cast;  // [V][H] of the weight's type or null: the finished d_weight sum goes here and
                          // d_weight only holds the running sums of earlier chunks
    float* kept;          // logits that the forward left (the plan is then kept_plan), or null: computed again
};

// Grid of a chained launch: one workgroup per compute unit, rounded down to a multiple of 8 so
// that a workgroup stays on one XCD from round to round; never more workgroups than tiles.
inline int chain_grid(int tiles, int n_cu)
{
    int g = n_cu >= 8 ? n_cu / 8 * 8 : n_cu;
    return tiles < g ? tiles : g;
}

// Enqueues the backward schedule: for every (token chunk, vocab piece) block
//   dZ recompute -> dH (+)= dZ W -> dW (+)= dZ^T hidden (-> db).
template <class T>
int bwd_enqueue(const BwdCall& c, const BwdPlan& p, int n_cu)
{
    using GZ = TileGemm<T, false, false, kBK>;
    using GH = TileGemm<T, true, false, kBK>;
    using GW = TileGemm<T, true, true, kBK>;
    constexpr int kChainSmem = TileGemmDtl<T, false, false, kBK, 32>::kSmemBytes;
    constexpr int kDzChainSmem = kChainSmem + kDzStageBytes * (kThreads / 64);
    const int H = c.H;
    const int64_t N = c.N, V = c.V;
    hipStream_t stream = c.stream;

    char* ws = static_cast<char*>(c.workspace);
    float* scales = reinterpret_cast<float*>(ws + p.scales_off);
    uint16_t* dz = reinterpret_cast<uint16_t*>(c.kept ? reinterpret_cast<char*>(c.kept) : ws + p.dz_off);
    float* hacc = p.acc_bytes ? reinterpret_cast<float*>(ws + p.acc_off) : nullptr;
    const uint16_t* hid = static_cast<const uint16_t*>(c.hidden);
    const uint16_t* w = static_cast<const uint16_t*>(c.weight);
    uint16_t* dh = static_cast<uint16_t*>(c.d_hidden);
    const int h_tiles = (H + 255) / 256;
    // Ragged token counts and vocabularies on the full-tile pipelines: the last token tile and the last
    // vocab tile are moved back so that they end at N and V (rows that exist whenever there are 256 of
    // them) and what their neighbours own is zero in the dZ block; fewer than 256 tokens are padded.
    // Device time against a launch for the ragged vocab tile, register-staged loops for K tails and
    // unchained dZ / dW launches for ragged token counts (the dW figures with the typed gradient):
    // 1000 x 1536 x 151936 dZ 599 -> 498 us, dW and its cast 1197 -> 515 us; 4096 x 2048 x 50257 dZ
    // 789 -> 732 us, dH 732 -> 658 us.
    const bool shifted = bwd_chained(H, V);
    const bool padded = shifted && N < 256;
    if (padded) {
        uint16_t* pad = reinterpret_cast<uint16_t*>(ws + p.pad_off);
        const int row8 = static_cast<int>(H / 8), n = static_cast<int>(N);
        const int used = std::max(2, (n + kBK - 1) / kBK) * kBK;  // the rows of dW's K steps, see k_steps below
        hipLaunchKernelGGL(linear_logp_pad_rows_kernel, dim3((row8 + 255) / 256, 256), dim3(256), 0, stream, hid, pad,
                           n, used, row8);
        hid = pad;
    }

    hipLaunchKernelGGL(linear_logp_scales_kernel, dim3(1), dim3(1024), 0, stream, c.grad_logp,
                       static_cast<int>(N), 1.f / c.temperature, c.dtype, scales);
    if (int rc = check_launch("scales kernel launch failed")) return rc;

    if (int rc = set_smem<linear_logp_dz_kernel<T, kBK, false, true>>(kDzChainSmem)) return rc;
    if (int rc = set_smem<linear_logp_dz_kernel<T, kBK, false, false>>(GZ::kSmemBytes)) return rc;
    if (int rc = set_smem<linear_logp_dz_kernel<T, kBK, true, false>>(GZ::kSmemBytes)) return rc;
    if (int rc = set_smem<linear_logp_grads_kernel<T, kBK, false>>(kChainSmem)) return rc;
    if (int rc = set_smem<linear_logp_dh_kernel<T, kBK>>(GH::kSmemBytes)) return rc;
    if (int rc = set_smem<linear_logp_dw_kernel<T, kBK>>(GW::kSmemBytes)) return rc;

    for (int ci = 0; ci < p.n_chunks; ++ci) {
        const int64_t tok_lo = static_cast<int64_t>(ci) * p.tok_chunk;
        const int tok_valid = static_cast<int>((N - tok_lo) < p.tok_chunk ? (N - tok_lo) : p.tok_chunk);
        if (tok_valid <= 0) break;
        const int tok_tiles = (tok_valid + 255) / 256;
        for (int pi = 0; pi < p.n_pieces; ++pi) {
            const int64_t v_lo = static_cast<int64_t>(pi) * p.v_piece;
            const int v_valid = static_cast<int>((V - v_lo) < p.v_piece ? (V - v_lo) : p.v_piece);
            if (v_valid <= 0) break;
            const int v_tiles = (v_valid + 255) / 256;
            const bool last_piece = (v_lo + p.v_piece >= V);
            const int tok_rag = tok_valid % 256, v_rag = v_valid % 256;
            const int tok_shift = shifted && !padded && tok_rag != 0 ? 256 - tok_rag : 0;
            const int v_shift = shifted && v_rag != 0 ? 256 - v_rag : 0;
            // K steps of dW (tokens) and dH (vocab rows): four per full tile, and of a shifted tile those
            // that hold rows of its own (two at least where it is the only one: the pipeline's minimum)
            auto k_steps = [](int valid, int shift) {
                const int full = valid / 256, rag = valid % 256;
                if (shift == 0) return full > 0 ? 4 * full : std::max(2, (rag + kBK - 1) / kBK);
                const int own = (rag + kBK - 1) / kBK;
                return 4 * full + (full == 0 ? std::max(2, own) : own);
            };
            // byte offset of those steps: past the tile's leading steps, and for the operand that is read
            // from the tensor itself `shift` rows back (the dZ block has the tile in its place)
            auto k_skip = [&](int valid, int shift) { return 4 * (valid / 256) + 4 - k_steps(valid, shift); };

            DzArgs z;
            z.hidden = hid + tok_lo * H;
            z.weight = w + v_lo * H;
            z.bias = c.bias ? c.bias + v_lo : nullptr;
            z.targets = c.targets + tok_lo;
            z.lse = c.lse + tok_lo;
            z.grad = c.grad_logp + tok_lo;
            z.scales = scales;
            z.dz = dz;
            z.ldz = p.ldz;
            z.tok_valid = tok_valid;
            z.v_valid = v_valid;
            z.H = H;
            z.tok_tiles = tok_tiles;
            z.tok_shift = tok_shift;
            z.v_shift = v_shift;
            z.v_global0 = c.vocab_start + v_lo;
            z.ignore_index = c.ignore_index;
            z.use_ignore = c.use_ignore;
            z.scale2 = kLog2e / c.temperature;

            DhArgs h;
            h.dz = dz;
            h.weight = w + v_lo * H;
            h.scales = scales;
            h.acc = hacc;
            h.out = dh ? dh + tok_lo * H : nullptr;
            h.ldz = p.ldz;
            h.H = H;
            h.v_valid = v_valid;
            h.tok_valid = tok_valid;
            h.tok_tiles = tok_tiles;
            h.h_tiles = h_tiles;
            h.first = pi == 0;
            h.last = last_piece;
            // per (chunk, piece) kind
            const int ksplit = dh_cuts(tok_tiles, v_tiles, h_tiles);
            h.ksplit = ksplit;
            h.part = ksplit > 1 ? reinterpret_cast<float*>(ws + p.part_off) : nullptr;
            h.part_stride = static_cast<int64_t>(tok_tiles) * 256 * H;
            const bool dh_chain = shifted || (ksplit == 1 && H >= 256 && v_valid % kBK == 0 && v_valid >= 2 * kBK);
            h.nk = shifted ? k_steps(v_valid, v_shift) : (dh_chain ? v_valid / kBK : 0);
            h.unit = p.whole ? 4 : 1;
            h.tok_shift = tok_shift;
            h.v_tiles = v_tiles;
            h.tail = KTail();
            if (v_shift != 0) {
                const int64_t skip = static_cast<int64_t>(k_skip(v_valid, v_shift)) * kBK;
                h.tail = KTail{v_valid / 256 * 4, (skip - v_shift) * H * 2, skip * 2};
            }

            DwArgs d;
            d.dz = dz;
            d.hidden = hid + tok_lo * H;
            d.scales = scales;
            d.dw = c.d_weight ? c.d_weight + v_lo * H : nullptr;
            d.out = c.d_weight_cast && ci == p.n_chunks - 1
                        ? static_cast<uint16_t*>(c.d_weight_cast) + v_lo * H : nullptr;
            d.ldz = p.ldz;
            d.H = H;
            d.v_valid = v_valid;
            d.tok_valid = tok_valid;
            d.v_tiles = v_tiles;
            d.h_tiles = h_tiles;
            d.accumulate = ci > 0 || c.accumulate != 0;
            const bool dw_chain = H >= 256 && (shifted || (tok_valid % kBK == 0 && tok_valid >= 2 * kBK));
            d.nk = shifted ? k_steps(tok_valid, tok_shift) : (dw_chain ? tok_valid / kBK : 0);
            d.v_shift = v_shift;
            d.tail = KTail();
            if (tok_shift != 0) {
                const int64_t skip = static_cast<int64_t>(k_skip(tok_valid, tok_shift)) * kBK;
                d.tail = KTail{tok_valid / 256 * 4, (skip - tok_shift) * H * 2,
                               c.kept ? skip / kBK * kKeptSlab * 4 : skip * p.ldz * 2};
            }
            float* db_part = c.d_bias ? reinterpret_cast<float*>(ws + p.db_off) : nullptr;

            // dZ block: chained through one pipeline when every tile can read 256 rows; otherwise the
            // full vocab tiles through the fast variant and the ragged last one through the general one
            // (all through the general one when the launch is tiny)
            const bool tiny = v_rag != 0 && tok_tiles * v_tiles <= 32;
            if (c.kept) {
                KeptDzArgs k;
                k.kept = c.kept;
                k.targets = z.targets;
                k.lse = z.lse;
                k.grad = z.grad;
                k.scales = scales;
                k.db_part = db_part;
                k.N = tok_valid;
                k.V = v_valid;
                k.v_tiles = v_tiles;
                k.tok_tiles = tok_tiles;
                k.tok_shift = tok_shift;
                k.v_shift = v_shift;
                k.used = padded ? d.nk * kBK : 256;
                k.vocab_start = z.v_global0;
                k.ignore_index = z.ignore_index;
                k.use_ignore = z.use_ignore;
                k.scale2 = z.scale2;
                k.slabs = kept_slabs(N);
                const dim3 slabs(k.slabs, v_tiles, tok_tiles);  // at most 3200 tiles in all
                if (db_part)
                    hipLaunchKernelGGL((linear_logp_dz_kept_kernel<T, true>), slabs, dim3(256), 0, stream, k);
                else
                    hipLaunchKernelGGL((linear_logp_dz_kept_kernel<T, false>), slabs, dim3(256), 0, stream, k);
            }
            const int fast_tiles = c.kept ? 0 : shifted ? v_tiles : (tiny ? 0 : v_valid / 256);
            const int gen_tiles = c.kept ? 0 : v_tiles - fast_tiles;
            const bool k_ok = H % kBK == 0 && H >= 2 * kBK;
            if (fast_tiles > 0) {
                z.v_tiles = fast_tiles;
                z.v_tile_lo = 0;
                const int tiles = tok_tiles * fast_tiles;
                if (shifted || (k_ok && tok_valid % 256 == 0))
                    hipLaunchKernelGGL((linear_logp_dz_kernel<T, kBK, false, true>),
                                       dim3(chain_grid(tiles, n_cu)), dim3(kThreads), kDzChainSmem,
                                       stream, z);
                else
                    hipLaunchKernelGGL((linear_logp_dz_kernel<T, kBK, false, false>), dim3(tiles),
                                       dim3(kThreads), GZ::kSmemBytes, stream, z);
            }
            if (gen_tiles > 0) {
                z.v_tiles = gen_tiles;
                z.v_tile_lo = fast_tiles;
                hipLaunchKernelGGL((linear_logp_dz_kernel<T, kBK, true, false>),
                                   dim3(tok_tiles * gen_tiles), dim3(kThreads), GZ::kSmemBytes,
                                   stream, z);
            }
            const bool want_dw = c.d_weight || c.d_weight_cast;
            // chained walks share a launch; a side that is not wanted or not chained has no tiles in it
            const bool dh_in = dh && dh_chain, dw_in = want_dw && dw_chain;
            if (dh && !dh_in)
                hipLaunchKernelGGL((linear_logp_dh_kernel<T, kBK>), dim3(tok_tiles * h_tiles * ksplit),
                                   dim3(kThreads), GH::kSmemBytes, stream, h);
            if (dh_in || dw_in) {
                DhArgs hj = h;
                DwArgs dj = d;
                if (!dh_in) hj.h_tiles = 0;
                if (!dw_in) dj.h_tiles = 0;
                const int items = tok_tiles * hj.h_tiles * ksplit + v_tiles * dj.h_tiles;
                const int grid = chain_grid(items, n_cu);
                const GradsSplit split = grads_split(tok_tiles * hj.h_tiles * ksplit, h.nk / ksplit + kDhSteps,
                                                     v_tiles * dj.h_tiles, d.nk + (d.accumulate ? kDwAddSteps : kDwSteps),
                                                     grid);
                dj.busy = split.busy;
                dj.lead = split.lead;
                auto launch_kept = [&](auto ht) -> int {
                    constexpr auto kernel = linear_logp_grads_kernel<T, kBK, true, decltype(ht)>;
                    if (int rc = set_smem<kernel>(kChainSmem)) return rc;
                    hipLaunchKernelGGL(kernel, dim3(grid), dim3(kThreads), kChainSmem, stream, hj, dj);
                    return 0;
                };
                if (c.kept) {
                    if (int rc = N <= 64 ? launch_kept(Acc16Few<1>{}) : N <= 128 ? launch_kept(Acc16Few<2>{})
                                 : N <= 192 ? launch_kept(Acc16Few<3>{}) : launch_kept(Acc16{}))
                        return rc;
                } else
                    hipLaunchKernelGGL((linear_logp_grads_kernel<T, kBK, false>), dim3(grid), dim3(kThreads),
                                       kChainSmem, stream, hj, dj);
            }
            if (dh && ksplit > 1) {
                const int64_t n4 = static_cast<int64_t>(tok_valid) * H / 4;
                hipLaunchKernelGGL((linear_logp_dh_reduce_kernel<T>),
                                   dim3(static_cast<unsigned>((n4 + 255) / 256)), dim3(256), 0, stream, h.part,
                                   ksplit, h.part_stride, h.acc, h.out, scales, n4, h.first, h.last);
            }
            if (want_dw && !dw_in)
                hipLaunchKernelGGL((linear_logp_dw_kernel<T, kBK>), dim3(v_tiles * h_tiles), dim3(kThreads),
                                   GW::kSmemBytes, stream, d);
            if (c.d_bias != nullptr) {
                const int rows = padded ? static_cast<int>(N) : 256;
                if (p.whole && !c.kept)
                    hipLaunchKernelGGL(linear_logp_db_slab_kernel<T>, dim3(v_tiles, 4 * tok_tiles), dim3(256), 0,
                                       stream, dz, p.ldz, rows, db_part, static_cast<int64_t>(p.v_piece));
                else if (!c.kept)
                    hipLaunchKernelGGL(linear_logp_db_partial_kernel<T>, dim3(v_tiles, tok_tiles), dim3(256), 0,
                                       stream, dz, p.ldz, rows, db_part, static_cast<int64_t>(p.v_piece));
                hipLaunchKernelGGL(linear_logp_db_finish_kernel, dim3((v_valid + 255) / 256), dim3(256), 0,
                                   stream, db_part, static_cast<int64_t>(p.v_piece),
                                   c.kept ? kept_slabs(N) * tok_tiles : p.whole ? 4 * tok_tiles : tok_tiles, v_valid, v_shift, scales, c.d_bias + v_lo,
                                   (ci > 0 || c.accumulate != 0) ? 1 : 0);
            }
            if (int rc = check_launch("linear_logp backward launch failed")) return rc;
        }
    }
    return 0;
}

// One forward contraction launch: a.row_blocks x a.n_split workgroups of the given variant.
template <class T, bool GENERAL>
int launch_fwd_as(const FwdArgs& a, hipStream_t stream)
{
    using G = TileGemm<T, false, false, kBK>;
    if (int rc = set_smem<linear_logp_fwd_kernel<T, kBK, GENERAL, false>>(G::kSmemBytes)) return rc;
    hipLaunchKernelGGL((linear_logp_fwd_kernel<T, kBK, GENERAL, false>), dim3(a.row_blocks * a.n_split),
                       dim3(kThreads), G::kSmemBytes, stream, a);
    return 0;
}

// The chained variants: by the width of the token tile (tokens below a full tile only) and whether logits are kept.
template <class T, bool KEEP, class AT>
int launch_fwd_chained_as(const FwdArgs& a, hipStream_t stream)
{
    using G = TileGemm<T, false, false, kBK>;
    if (int rc = set_smem<linear_logp_fwd_kernel<T, kBK, false, true, KEEP, AT>>(G::kSmemBytes)) return rc;
    hipLaunchKernelGGL((linear_logp_fwd_kernel<T, kBK, false, true, KEEP, AT>), dim3(a.row_blocks * a.n_split),
                       dim3(kThreads), G::kSmemBytes, stream, a);
    return 0;
}

template <class T, bool KEEP>
int launch_fwd_chained(const FwdArgs& a, hipStream_t stream)
{
    if (a.N <= 64) return launch_fwd_chained_as<T, KEEP, Acc16Few<1>>(a, stream);
    if (a.N <= 128) return launch_fwd_chained_as<T, KEEP, Acc16Few<2>>(a, stream);
    if (a.N <= 192) return launch_fwd_chained_as<T, KEEP, Acc16Few<3>>(a, stream);
    return launch_fwd_chained_as<T, KEEP, Acc16>(a, stream);
}

template <bool GENERAL>
int launch_fwd(const FwdArgs& a, int32_t dtype, hipStream_t stream)
{
    return dtype == RLK_DTYPE_BF16 ? launch_fwd_as<Bf16, GENERAL>(a, stream)
                                   : launch_fwd_as<F16, GENERAL>(a, stream);
}

// A second head over the same hidden states and targets (a frozen reference model).
struct SecondHead {
    const void* weight;
    const float* bias;
    float* logp;
    float* lse;
};

int fwd_enqueue(const void* hidden, const void* weight, const float* bias, const int64_t* targets,
                float* logp, float* lse, void* workspace, size_t workspace_bytes, int64_t N,
                int32_t H, int64_t V, int64_t vocab_start, int32_t dtype, float temperature,
                int64_t ignore_index, int32_t use_ignore, int32_t strict_targets,
                int32_t* err_flag, hipStream_t stream, const GrpoArgs* epilogue = nullptr,
                const SecondHead* second = nullptr, float* kept = nullptr, size_t kept_size = 0);

}  // namespace

// Scratch of rlk_linear_logp_fwd_static: the forward's per-split partial softmax states live in
// this file-scope device array instead of a caller workspace, so that entry point allocates
// nothing.  Every GPU the library runs on holds its own copy until the process ends.  In host code
// the array's name is only a handle; the device address is looked up once per device below and
// that pointer is what the kernels receive.
static __device__ __align__(256) unsigned char scratch[RLK_STATIC_SCRATCH_BYTES];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[kMaxDevices] = {};

// Device address of `scratch` on the current device (resolved on the first call per device).
int static_scratch_ptr(void** out)
{
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return rlk_fail(RLK_ERR_LAUNCH, hipGetErrorString(e));
    if (dev < 0 || dev >= kMaxDevices) return rlk_fail(RLK_ERR_UNSUPPORTED, "device index too large");
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (g_scratch_ptr[dev] == nullptr) {
        void* ptr = nullptr;
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || ptr == nullptr)
            return rlk_fail(RLK_ERR_LAUNCH, e != hipSuccess ? hipGetErrorString(e)
                                                            : "static scratch has no device address");
        g_scratch_ptr[dev] = ptr;
    }
    *out = g_scratch_ptr[dev];
    return 0;
}

}  // namespace

extern "C" {

int rlk_linear_logp_fwd_workspace_bytes(int64_t N, int32_t H, int64_t V, int32_t dtype,
                                        size_t* bytes)
{
    (void)dtype;
    if (!bytes || N <= 0 || V <= 0 || H <= 0) return rlk_fail(RLK_ERR_ARG, "bad workspace query");
    // sized for the larger of the two plans so that one query serves both kinds of kernels
    const int a = fwd_plan(N, H, V, false).total_splits, b = fwd_plan(N, H, V, true).total_splits;
    *bytes = static_cast<size_t>(3) * (a > b ? a : b) * N * sizeof(float);
    return 0;
}

int rlk_linear_logp_fwd(const void* hidden, const void* weight, const float* bias,
                        const int64_t* targets, float* logp, float* lse, void* workspace,
                        size_t workspace_bytes, int64_t N, int32_t H, int64_t V,
                        int64_t vocab_start, int32_t dtype, float temperature,
                        int64_t ignore_index, int32_t use_ignore, int32_t strict_targets,
                        int32_t* err_flag, hipStream_t stream)
{
    return fwd_enqueue(hidden, weight, bias, targets, logp, lse, workspace, workspace_bytes, N, H, V,
                       vocab_start, dtype, temperature, ignore_index, use_ignore, strict_targets,
                       err_flag, stream);
}

int rlk_linear_logp_fwd_static(const void* hidden, const void* weight, const float* bias,
                               const int64_t* targets, float* logp, float* lse, int64_t N,
                               int32_t H, int64_t V, int64_t vocab_start, int32_t dtype,
                               float temperature, int64_t ignore_index, int32_t use_ignore,
                               int32_t strict_targets, int32_t* err_flag, hipStream_t stream)
{
    if (int rc = check_common(N, H, V, dtype)) return rc;
    size_t need = 0;
    if (int rc = rlk_linear_logp_fwd_workspace_bytes(N, H, V, dtype, &need)) return rc;
    if (need > static_cast<size_t>(RLK_STATIC_SCRATCH_BYTES))
        return rlk_fail(RLK_ERR_ARG,
                        "rlk_linear_logp_fwd_static: the split partials of this N exceed the "
                        "library's static scratch (RLK_STATIC_SCRATCH_BYTES); use "
                        "rlk_linear_logp_fwd with a caller workspace");
    void* ws = nullptr;
    if (int rc = static_scratch_ptr(&ws)) return rc;
    return fwd_enqueue(hidden, weight, bias, targets, logp, lse, ws, RLK_STATIC_SCRATCH_BYTES, N, H,
                       V, vocab_start, dtype, temperature, ignore_index, use_ignore,
                       strict_targets, err_flag, stream);
}

int rlk_linear_logp_fwd_pair_workspace_bytes(int64_t N, int32_t H, int64_t V, int32_t dtype,
                                             size_t* bytes)
{
    if (int rc = rlk_linear_logp_fwd_workspace_bytes(N, H, V, dtype, bytes)) return rc;
    *bytes *= 2;
    return 0;
}

int rlk_linear_logp_fwd_pair(const void* hidden, const void* weight, const void* ref_weight,
                             const float* bias, const float* ref_bias, const int64_t* targets,
                             float* logp, float* lse, float* ref_logp, float* ref_lse,
                             void* workspace, size_t workspace_bytes, int64_t N, int32_t H,
                             int64_t V, int64_t vocab_start, int32_t dtype, float temperature,
                             int64_t ignore_index, int32_t use_ignore, int32_t strict_targets,
                             int32_t* err_flag, hipStream_t stream)
{
    if (!ref_weight || !ref_logp || !ref_lse) return rlk_fail(RLK_ERR_ARG, "null pointer");
    if ((bias == nullptr) != (ref_bias == nullptr))
        return rlk_fail(RLK_ERR_UNSUPPORTED, "both heads must have a bias or neither");
    const SecondHead second{ref_weight, ref_bias, ref_logp, ref_lse};
    return fwd_enqueue(hidden, weight, bias, targets, logp, lse, workspace, workspace_bytes, N, H, V,
                       vocab_start, dtype, temperature, ignore_index, use_ignore, strict_targets,
                       err_flag, stream, nullptr, &second);
}

int rlk_linear_logp_fwd_grpo_workspace_bytes(int64_t N, int32_t H, int64_t V, int32_t dtype,
                                             size_t* bytes)
{
    size_t fwd = 0, epi = 0;
    if (int rc = rlk_linear_logp_fwd_workspace_bytes(N, H, V, dtype, &fwd)) return rc;
    if (int rc = rlk_grpo_loss_workspace_bytes(N, &epi)) return rc;
    *bytes = (fwd + 255) / 256 * 256 + epi;
    return 0;
}

int rlk_linear_logp_fwd_grpo(const void* hidden, const void* weight, const float* bias,
                             const int64_t* targets, float* logp, float* lse, void* workspace,
                             size_t workspace_bytes, int64_t N, int32_t H, int64_t V,
                             int64_t vocab_start, int32_t dtype, float temperature,
                             int64_t ignore_index, int32_t use_ignore, int32_t strict_targets,
                             int32_t* err_flag, const float* old_logp, const float* ref_logp,
                             const float* advantages, int32_t adv_per_token, const uint8_t* mask,
                             int64_t seq_len, float clip_eps, float beta, float* out3, float* ratio,
                             float* kl_terms, float* d_cur, float* d_kl, hipStream_t stream)
{
    return rlk_linear_logp_fwd_grpo_kept(hidden, weight, bias, targets, logp, lse, workspace, workspace_bytes, N, H, V,
                                         vocab_start, dtype, temperature, ignore_index, use_ignore, strict_targets,
                                         err_flag, old_logp, ref_logp, advantages, adv_per_token, mask, seq_len,
                                         clip_eps, beta, out3, ratio, kl_terms, d_cur, d_kl, nullptr, 0, stream);
}

int rlk_linear_logp_kept_bytes(int64_t N, int32_t H, int64_t V, int32_t dtype, size_t* bytes)
{
    if (!bytes || N <= 0 || V <= 0 || H <= 0) return rlk_fail(RLK_ERR_ARG, "bad kept-logits query");
    *bytes = kept_bytes(N, H, V, dtype);
    return 0;
}

int rlk_linear_logp_kept_least_bytes(int64_t N, int32_t H, int64_t V, int32_t dtype, size_t* bytes)
{
    if (!bytes || N <= 0 || V <= 0 || H <= 0) return rlk_fail(RLK_ERR_ARG, "bad kept-logits query");
    *bytes = kept_least(N, H, V, dtype);
    return 0;
}

int rlk_linear_logp_fwd_kept(const void* hidden, const void* weight, const float* bias,
                             const int64_t* targets, float* logp, float* lse, void* workspace,
                             size_t workspace_bytes, int64_t N, int32_t H, int64_t V,
                             int64_t vocab_start, int32_t dtype, float temperature,
                             int64_t ignore_index, int32_t use_ignore, int32_t strict_targets,
                             int32_t* err_flag, void* kept, size_t kept_bytes, hipStream_t stream)
{
    return fwd_enqueue(hidden, weight, bias, targets, logp, lse, workspace, workspace_bytes, N, H, V, vocab_start, dtype,
                       temperature, ignore_index, use_ignore, strict_targets, err_flag, stream, nullptr, nullptr,
                       static_cast<float*>(kept), kept_bytes);
}

int rlk_linear_logp_fwd_grpo_kept(const void* hidden, const void* weight, const float* bias,
                             const int64_t* targets, float* logp, float* lse, void* workspace,
                             size_t workspace_bytes, int64_t N, int32_t H, int64_t V,
                             int64_t vocab_start, int32_t dtype, float temperature,
                             int64_t ignore_index, int32_t use_ignore, int32_t strict_targets,
                             int32_t* err_flag, const float* old_logp, const float* ref_logp,
                             const float* advantages, int32_t adv_per_token, const uint8_t* mask,
                             int64_t seq_len, float clip_eps, float beta, float* out3, float* ratio,
                             float* kl_terms, float* d_cur, float* d_kl, void* kept, size_t kept_bytes,
                             hipStream_t stream)
{
    if (int rc = check_common(N, H, V, dtype)) return rc;
    if (!old_logp || !advantages || !out3 || !logp) return rlk_fail(RLK_ERR_ARG, "null pointer");
    if (seq_len <= 0) return rlk_fail(RLK_ERR_ARG, "bad sizes");
    if (!adv_per_token && N % seq_len != 0)
        return rlk_fail(RLK_ERR_ARG, "N must be a multiple of seq_len for per-sequence advantages");
    if (d_kl != nullptr && d_cur == nullptr) return rlk_fail(RLK_ERR_ARG, "d_kl requires d_cur");
    size_t need = 0, fwd = 0;
    if (int rc = rlk_linear_logp_fwd_grpo_workspace_bytes(N, H, V, dtype, &need)) return rc;
    rlk_linear_logp_fwd_workspace_bytes(N, H, V, dtype, &fwd);
    if (!workspace || workspace_bytes < need) return rlk_fail(RLK_ERR_ARG, "workspace too small");
    if (reinterpret_cast<uintptr_t>(workspace) & 15) return rlk_fail(RLK_ERR_ARG, "workspace must be 16-byte aligned");
    GrpoArgs g;
    g.cur = logp;
    g.old_lp = old_logp;
    g.ref_lp = ref_logp;
    g.adv = advantages;
    g.mask = mask;
    g.ratio = ratio;
    g.kl_terms = kl_terms;
    g.partial = reinterpret_cast<float*>(static_cast<char*>(workspace) + (fwd + 255) / 256 * 256);
    g.denom = g.partial + kMaxBlocks * 3;
    g.words = reinterpret_cast<int*>(g.denom + 4);
    g.out3 = out3;
    g.dcur = d_cur;
    g.dkl = d_kl;
    g.upstream = nullptr;
    g.n = N;
    g.seq_len = seq_len;
    g.adv_per_token = adv_per_token;
    g.clip_lo = 1.f - clip_eps;
    g.clip_hi = 1.f + clip_eps;
    g.beta = beta;
    g.blocks = grpo_blocks(N);
    return fwd_enqueue(hidden, weight, bias, targets, logp, lse, workspace, fwd, N, H, V, vocab_start,
                       dtype, temperature, ignore_index, use_ignore, strict_targets, err_flag, stream,
                       &g, nullptr, static_cast<float*>(kept), kept_bytes);
}

}  // extern "C"

namespace {

// `epilogue` (optional): GRPO loss arguments whose `cur` is the logp this call produces; the
// per-token loss pass then runs inside the combine launch.
int fwd_enqueue(const void* hidden, const void* weight, const float* bias, const int64_t* targets,
                float* logp, float* lse, void* workspace, size_t workspace_bytes, int64_t N,
                int32_t H, int64_t V, int64_t vocab_start, int32_t dtype, float temperature,
                int64_t ignore_index, int32_t use_ignore, int32_t strict_targets,
                int32_t* err_flag, hipStream_t stream, const GrpoArgs* epilogue,
                const SecondHead* second, float* kept, size_t kept_size)
{
    if (int rc = check_common(N, H, V, dtype)) return rc;
    if (!(temperature > 0.f)) return rlk_fail(RLK_ERR_ARG, "temperature must be greater than zero");
    if (!hidden || !weight || !targets || !logp || !lse) return rlk_fail(RLK_ERR_ARG, "null pointer");
    if (strict_targets && !err_flag)
        return rlk_fail(RLK_ERR_ARG, "strict_targets needs an err_flag to report through");
    const bool mfma = use_mfma(hidden, weight, H, dtype);
    if (kept != nullptr)
        if (int rc = check_kept(kept, kept_size, mfma, N, H, V, dtype)) return rc;
    // Both heads of a pair run through one launch, so they must take the same kind of kernel:
    // otherwise the policy head's results would depend on the reference head's alignment and no
    // longer equal the single-head call bit for bit.
    if (second != nullptr && use_mfma(hidden, second->weight, H, dtype) != mfma)
        return rlk_fail(RLK_ERR_UNSUPPORTED,
                        "rlk_linear_logp_fwd_pair: weight and ref_weight must both start on a 16-byte "
                        "boundary or neither (one would run on the 16-bit MFMA tiles, the other on the "
                        "fp32 matrix-core kernels); call rlk_linear_logp_fwd once per head instead");
    size_t need = 0;
    rlk_linear_logp_fwd_workspace_bytes(N, H, V, dtype, &need);
    if (second != nullptr) need *= 2;
    if (!workspace || workspace_bytes < need) return rlk_fail(RLK_ERR_ARG, "workspace too small");
    if (epilogue != nullptr) {
        // the active-token count only needs the mask: it is ready long before the contraction ends
        const int parts = grpo_count_parts(epilogue->n);
        hipLaunchKernelGGL(grpo_count_kernel<0>, dim3(parts), dim3(kRedThreads), 0, stream,
                           epilogue->mask, epilogue->n, parts, epilogue->words);
        if (int rc = check_launch("grpo_count_kernel launch failed")) return rc;
    }

    FwdArgs a;
    a.hidden = static_cast<const uint16_t*>(hidden);
    a.weight = static_cast<const uint16_t*>(weight);
    a.bias = bias;
    a.weight2 = second ? static_cast<const uint16_t*>(second->weight) : nullptr;
    a.bias2 = second ? second->bias : nullptr;
    a.targets = targets;
    a.N = static_cast<int>(N);
    a.H = H;
    a.V = static_cast<int>(V);
    a.vocab_start = vocab_start;
    // the fp32 matrix-core kernels treat every tile as general
    const FwdPlan plan = fwd_plan(N, H, V, !mfma);
    a.row_blocks = plan.row_blocks;
    a.patch_rows = plan.patch_rows;
    a.part_m = static_cast<float*>(workspace);
    a.part_s = a.part_m + static_cast<size_t>(plan.total_splits) * N;
    a.part_z = a.part_s + static_cast<size_t>(plan.total_splits) * N;
    a.part2_m = a.part_z + static_cast<size_t>(plan.total_splits) * N;
    a.part2_s = a.part2_m + static_cast<size_t>(plan.total_splits) * N;
    a.part2_z = a.part2_s + static_cast<size_t>(plan.total_splits) * N;
    a.scale2 = kLog2e / temperature;

    if (!mfma) {
        if (int rc = wide_fwd_partials(hidden, weight, bias, targets, a.part_m, a.part_s, a.part_z,
                                       plan.total_splits, N, H, V, vocab_start, dtype, temperature, stream, kept))
            return rc;
        if (second != nullptr)
            if (int rc = wide_fwd_partials(hidden, second->weight, second->bias, targets, a.part2_m,
                                           a.part2_s, a.part2_z, plan.total_splits, N, H, V, vocab_start,
                                           dtype, temperature, stream))
                return rc;
    }
    if (mfma && plan.n_fast > 0) {
        a.n_split = plan.n_fast;
        a.split_lo = 0;
        a.tile_lo = 0;
        a.vtiles = plan.fast_tiles;
        a.kept = kept;
        const bool bf16 = dtype == RLK_DTYPE_BF16;
        if (int rc = kept != nullptr ? (bf16 ? launch_fwd_chained<Bf16, true>(a, stream)
                                             : launch_fwd_chained<F16, true>(a, stream))
                     : fwd_chained(H, V) ? (bf16 ? launch_fwd_chained<Bf16, false>(a, stream)
                                                 : launch_fwd_chained<F16, false>(a, stream))
                                         : launch_fwd<false>(a, dtype, stream))
            return rc;
    }
    if (mfma && plan.n_gen > 0) {
        a.n_split = plan.n_gen;
        a.split_lo = plan.n_fast;
        a.tile_lo = plan.fast_tiles;
        a.vtiles = plan.gen_tiles;
        if (int rc = launch_fwd<true>(a, dtype, stream)) return rc;
    }
    if (int rc = check_launch("linear_logp_fwd_kernel launch failed")) return rc;

    CombineArgs c;
    c.part_m = a.part_m;
    c.part_s = a.part_s;
    c.part_z = a.part_z;
    c.targets = targets;
    c.logp = logp;
    c.lse = lse;
    c.err_flag = err_flag;
    c.N = a.N;
    c.V = a.V;
    c.n_split = plan.total_splits;
    c.vocab_start = vocab_start;
    c.ignore_index = ignore_index;
    c.use_ignore = use_ignore;
    c.strict = strict_targets;
    // from 16 splits on the partials are merged by a launch of their own (up to there one thread per
    // token takes at most as long as that launch)
    if (plan.total_splits >= 16) {
        const dim3 blocks((a.N + kMergeTokens - 1) / kMergeTokens);
        const size_t lds = merge_smem(plan.total_splits);  // at most 256 splits: 9 KiB
        hipLaunchKernelGGL(linear_logp_merge_kernel, blocks, dim3(256), lds, stream, a.part_m, a.part_s, a.part_z, a.N,
                           plan.total_splits);
        if (second != nullptr)
            hipLaunchKernelGGL(linear_logp_merge_kernel, blocks, dim3(256), lds, stream, a.part2_m, a.part2_s,
                               a.part2_z, a.N, plan.total_splits);
        c.n_split = 1;
    }
    if (second != nullptr) {  // the reference head: same merge, never strict
        CombineArgs c2 = c;
        c2.part_m = a.part2_m;
        c2.part_s = a.part2_s;
        c2.part_z = a.part2_z;
        c2.logp = second->logp;
        c2.lse = second->lse;
        c2.strict = 0;
        hipLaunchKernelGGL(linear_logp_combine_kernel, dim3((a.N + 255) / 256), dim3(256), 0, stream, c2);
    }
    if (epilogue == nullptr) {
        hipLaunchKernelGGL(linear_logp_combine_kernel, dim3((a.N + 255) / 256), dim3(256), 0, stream, c);
        return check_launch("linear_logp_combine_kernel launch failed");
    }
    hipLaunchKernelGGL(linear_logp_combine_grpo_kernel, dim3(epilogue->blocks), dim3(kRedThreads), 0,
                       stream, c, *epilogue);
    return check_launch("combine + GRPO epilogue launch failed");
}

}  // namespace

extern "C" {

int rlk_linear_logp_bwd_workspace_bytes(int64_t N, int32_t H, int64_t V, int32_t dtype,
                                        size_t dz_budget_bytes, size_t* bytes)
{
    (void)dtype;
    if (!bytes || N <= 0 || V <= 0 || H <= 0) return rlk_fail(RLK_ERR_ARG, "bad workspace query");
    dz_budget_bytes = clamp_dz_budget(dz_budget_bytes);
    // large enough for either implementation (the choice also depends on pointer alignment)
    const size_t a = bwd_plan(N, H, V, dz_budget_bytes).total, b = wide_bwd_workspace(N, H, V, dz_budget_bytes);
    *bytes = a > b ? a : b;
    return 0;
}

int rlk_linear_logp_fwd_plan(int64_t N, int32_t H, int64_t V, int32_t dtype, int64_t* out4)
{
    if (!out4 || N <= 0 || V <= 0 || H <= 0) return rlk_fail(RLK_ERR_ARG, "bad plan query");
    const FwdPlan p = fwd_plan(N, H, V, dtype == RLK_DTYPE_F32);
    out4[0] = p.row_blocks;
    out4[1] = p.n_fast;
    out4[2] = p.n_gen;
    out4[3] = p.patch_rows;
    return 0;
}

int rlk_linear_logp_bwd_plan(int64_t N, int32_t H, int64_t V, int32_t dtype, size_t dz_budget_bytes,
                             int64_t* out5)
{
    (void)dtype;
    if (!out5 || N <= 0 || V <= 0 || H <= 0) return rlk_fail(RLK_ERR_ARG, "bad plan query");
    dz_budget_bytes = clamp_dz_budget(dz_budget_bytes);
    const BwdPlan p = bwd_plan(N, H, V, dz_budget_bytes);
    out5[0] = p.tok_chunk;
    out5[1] = p.v_piece;
    out5[2] = p.n_chunks;
    out5[3] = p.n_pieces;
    out5[4] = p.ksplit;
    return 0;
}

int rlk_linear_logp_bwd(const float* grad_logp, const void* hidden, const void* weight,
                        const float* bias, const int64_t* targets, const float* lse,
                        void* d_hidden, float* d_weight, float* d_bias, void* workspace,
                        size_t workspace_bytes, size_t dz_budget_bytes, int64_t N, int32_t H,
                        int64_t V, int64_t vocab_start, int32_t dtype, float temperature,
                        int64_t ignore_index, int32_t use_ignore, hipStream_t stream)
{
    return rlk::linear_logp_bwd_accumulating(grad_logp, hidden, weight, bias, targets, lse, d_hidden,
                                             d_weight, d_bias, workspace, workspace_bytes,
                                             dz_budget_bytes, N, H, V, vocab_start, dtype, temperature,
                                             ignore_index, use_ignore, 0, stream);
}

int rlk_linear_logp_bwd_accum(const float* grad_logp, const void* hidden, const void* weight,
                              const float* bias, const int64_t* targets, const float* lse,
                              void* d_hidden, float* d_weight, float* d_bias, void* workspace,
                              size_t workspace_bytes, size_t dz_budget_bytes, int64_t N, int32_t H,
                              int64_t V, int64_t vocab_start, int32_t dtype, float temperature,
                              int64_t ignore_index, int32_t use_ignore, int32_t accumulate,
                              hipStream_t stream)
{
    return rlk::linear_logp_bwd_accumulating(grad_logp, hidden, weight, bias, targets, lse, d_hidden,
                                             d_weight, d_bias, workspace, workspace_bytes,
                                             dz_budget_bytes, N, H, V, vocab_start, dtype, temperature,
                                             ignore_index, use_ignore, accumulate != 0 ? 1 : 0, stream);
}

int rlk_linear_logp_bwd_kept_workspace_bytes(int64_t N, int32_t H, int64_t V, int32_t dtype, size_t* bytes)
{
    if (!bytes || N <= 0 || V <= 0 || H <= 0) return rlk_fail(RLK_ERR_ARG, "bad workspace query");
    if (kept_bytes(N, H, V, dtype) == 0)
        return rlk_fail(RLK_ERR_UNSUPPORTED, "no logits are kept for these sizes (rlk_linear_logp_kept_bytes)");
    *bytes = dtype == RLK_DTYPE_F32 ? wide_bwd_kept_workspace(N, H, V, false) : kept_plan(N, H, V, false).total;
    return 0;
}

int rlk_linear_logp_bwd_as_kept_workspace_bytes(int64_t N, int32_t H, int64_t V, int32_t dtype, size_t* bytes)
{
    if (int rc = rlk_linear_logp_bwd_kept_workspace_bytes(N, H, V, dtype, bytes)) return rc;
    *bytes = dtype == RLK_DTYPE_F32 ? wide_bwd_kept_workspace(N, H, V, true) : kept_plan(N, H, V, true).total;
    return 0;
}

int rlk_linear_logp_bwd_kept(const float* grad_logp, const void* hidden, const void* weight,
                             const float* bias, const int64_t* targets, const float* lse,
                             void* d_hidden, float* d_weight, void* d_weight_typed, float* d_bias, void* kept,
                             size_t kept_size, void* workspace, size_t workspace_bytes, int64_t N, int32_t H,
                             int64_t V, int64_t vocab_start, int32_t dtype, float temperature,
                             int64_t ignore_index, int32_t use_ignore, int32_t accumulate, hipStream_t stream)
{
    if (int rc = check_common(N, H, V, dtype)) return rc;
    if (!(temperature > 0.f)) return rlk_fail(RLK_ERR_ARG, "temperature must be greater than zero");
    if (!grad_logp || !hidden || !weight || !targets || !lse) return rlk_fail(RLK_ERR_ARG, "null pointer");
    if (kept == nullptr && kept_size != 0) return rlk_fail(RLK_ERR_ARG, "no kept logits and a size of them");
    if (!d_hidden && !d_weight && !d_bias && !d_weight_typed)
        return rlk_fail(RLK_ERR_ARG, "no gradient requested");
    if (bias == nullptr && d_bias != nullptr) return rlk_fail(RLK_ERR_ARG, "d_bias given without bias");
    if (d_weight_typed != nullptr &&
        (d_weight != nullptr || accumulate != 0 || (reinterpret_cast<uintptr_t>(d_weight_typed) & 15) != 0))
        return rlk_fail(RLK_ERR_ARG, "d_weight_typed takes no fp32 d_weight beside it and starts on a 16-byte boundary");
    if (int rc = check_kept(kept, kept_size, use_mfma(hidden, weight, H, dtype), N, H, V, dtype)) return rc;
    size_t need = 0;
    if (int rc = kept ? rlk_linear_logp_bwd_kept_workspace_bytes(N, H, V, dtype, &need)
                      : rlk_linear_logp_bwd_as_kept_workspace_bytes(N, H, V, dtype, &need))
        return rc;
    if (!workspace || workspace_bytes < need) return rlk_fail(RLK_ERR_ARG, "workspace too small");
    if (reinterpret_cast<uintptr_t>(workspace) & 255)
        return rlk_fail(RLK_ERR_ARG, "workspace must be 256-byte aligned");
    if (dtype == RLK_DTYPE_F32)  // the weight's type is fp32
        return wide_bwd_kept(grad_logp, hidden, weight, bias, targets, lse, d_hidden,
                             d_weight_typed ? static_cast<float*>(d_weight_typed) : d_weight, d_bias,
                             static_cast<float*>(kept), workspace, N, H, V, vocab_start, temperature, ignore_index,
                             use_ignore, accumulate != 0 ? 1 : 0, stream);
    const BwdPlan p = kept_plan(N, H, V, kept == nullptr);
    int n_cu = 0;
    if (int rc = compute_units(&n_cu)) return rc;
    BwdCall c{grad_logp, hidden, weight, bias, targets, lse, d_hidden, d_weight, d_bias, workspace, N, H, V, vocab_start,
              dtype, temperature, ignore_index, use_ignore, stream, accumulate != 0 ? 1 : 0, d_weight_typed,
              static_cast<float*>(kept)};
    return dtype == RLK_DTYPE_BF16 ? bwd_enqueue<Bf16>(c, p, n_cu) : bwd_enqueue<F16>(c, p, n_cu);
}

int rlk_linear_logp_bwd_typed_workspace_bytes(int64_t N, int32_t H, int64_t V, int32_t dtype,
                                              size_t dz_budget_bytes, size_t* bytes)
{
    if (dtype != RLK_DTYPE_BF16 && dtype != RLK_DTYPE_F16)
        return rlk_fail(RLK_ERR_UNSUPPORTED, "the typed weight gradient is for bf16 and f16 heads");
    if (int rc = rlk_linear_logp_bwd_workspace_bytes(N, H, V, dtype, dz_budget_bytes, bytes)) return rc;
    const BwdPlan p = bwd_plan(N, H, V, clamp_dz_budget(dz_budget_bytes));
    // the running fp32 sum of all token chunks but the last
    if (p.n_chunks > 1) *bytes = align_up(*bytes, 256) + static_cast<size_t>(V) * H * 4;
    return 0;
}

int rlk_linear_logp_bwd_typed(const float* grad_logp, const void* hidden, const void* weight,
                              const float* bias, const int64_t* targets, const float* lse,
                              void* d_hidden, void* d_weight, float* d_bias, void* workspace,
                              size_t workspace_bytes, size_t dz_budget_bytes, int64_t N, int32_t H,
                              int64_t V, int64_t vocab_start, int32_t dtype, float temperature,
                              int64_t ignore_index, int32_t use_ignore, hipStream_t stream)
{
    if (int rc = check_common(N, H, V, dtype)) return rc;
    if (!grad_logp || !hidden || !weight || !targets || !lse || !d_weight)
        return rlk_fail(RLK_ERR_ARG, "null pointer");
    if (!use_mfma(hidden, weight, H, dtype) || (reinterpret_cast<uintptr_t>(d_weight) & 15) != 0)
        return rlk_fail(RLK_ERR_UNSUPPORTED,
                        "rlk_linear_logp_bwd_typed takes bf16 / f16, H % 8 == 0 and 16-byte aligned matrices");
    size_t need = 0, base = 0;
    if (int rc = rlk_linear_logp_bwd_typed_workspace_bytes(N, H, V, dtype, dz_budget_bytes, &need)) return rc;
    if (int rc = rlk_linear_logp_bwd_workspace_bytes(N, H, V, dtype, dz_budget_bytes, &base)) return rc;
    if (!workspace || workspace_bytes < need) return rlk_fail(RLK_ERR_ARG, "workspace too small");
    float* running = need > base
                         ? reinterpret_cast<float*>(static_cast<char*>(workspace) + align_up(base, 256)) : nullptr;
    return rlk::linear_logp_bwd_accumulating(grad_logp, hidden, weight, bias, targets, lse, d_hidden, running,
                                             d_bias, workspace, base, dz_budget_bytes, N, H, V, vocab_start,
                                             dtype, temperature, ignore_index, use_ignore, 0, stream, d_weight);
}

}  // extern "C"

int rlk::linear_logp_bwd_accumulating(const float* grad_logp, const void* hidden, const void* weight,
                                      const float* bias, const int64_t* targets, const float* lse,
                                      void* d_hidden, float* d_weight, float* d_bias, void* workspace,
                                      size_t workspace_bytes, size_t dz_budget_bytes, int64_t N,
                                      int32_t H, int64_t V, int64_t vocab_start, int32_t dtype,
                                      float temperature, int64_t ignore_index, int32_t use_ignore,
                                      int32_t accumulate, hipStream_t stream, void* d_weight_cast)
{
    if (int rc = check_common(N, H, V, dtype)) return rc;
    if (!(temperature > 0.f)) return rlk_fail(RLK_ERR_ARG, "temperature must be greater than zero");
    if (!grad_logp || !hidden || !weight || !targets || !lse) return rlk_fail(RLK_ERR_ARG, "null pointer");
    if (!d_hidden && !d_weight && !d_bias && !d_weight_cast)
        return rlk_fail(RLK_ERR_ARG, "no gradient requested");
    if (bias == nullptr && d_bias != nullptr) return rlk_fail(RLK_ERR_ARG, "d_bias given without bias");
    dz_budget_bytes = clamp_dz_budget(dz_budget_bytes);
    size_t need = 0;
    rlk_linear_logp_bwd_workspace_bytes(N, H, V, dtype, dz_budget_bytes, &need);
    if (!workspace || workspace_bytes < need) return rlk_fail(RLK_ERR_ARG, "workspace too small");
    if (reinterpret_cast<uintptr_t>(workspace) & 255)
        return rlk_fail(RLK_ERR_ARG, "workspace must be 256-byte aligned");
    if (!use_mfma(hidden, weight, H, dtype) && d_weight_cast != nullptr)
        return rlk_fail(RLK_ERR_UNSUPPORTED, "the fp32 matrix-core kernels write fp32 weight gradients only");
    if (!use_mfma(hidden, weight, H, dtype))
        return wide_bwd(grad_logp, hidden, weight, bias, targets, lse, d_hidden, d_weight, d_bias,
                        workspace, dz_budget_bytes, N, H, V, vocab_start, dtype, temperature,
                        ignore_index, use_ignore, accumulate, stream);
    const BwdPlan p = bwd_plan(N, H, V, dz_budget_bytes);
    if (d_weight_cast != nullptr && d_weight == nullptr && (p.n_chunks > 1 || accumulate))
        return rlk_fail(RLK_ERR_ARG, "several token chunks need a running fp32 weight gradient");
    int n_cu = 0;
    if (int rc = compute_units(&n_cu)) return rc;
    BwdCall c{grad_logp, hidden, weight, bias, targets, lse, d_hidden, d_weight, d_bias, workspace,
              N, H, V, vocab_start, dtype, temperature, ignore_index, use_ignore, stream, accumulate, d_weight_cast,
              nullptr};
    return dtype == RLK_DTYPE_BF16 ? bwd_enqueue<Bf16>(c, p, n_cu) : bwd_enqueue<F16>(c, p, n_cu);
}
