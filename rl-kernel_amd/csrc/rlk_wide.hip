// fp32 matrix-core kernels of the fused linear-logprob path for inputs the 16-bit MFMA tiles do
// not take: fp32 tensors, hidden sizes that are not a multiple of 8, matrices that do not start on
// a 16-byte boundary.  Every operand is widened to fp32 on its way into LDS (exact for bf16 and
// f16) and multiplied as three bf16 pieces (SplitGemm below; v_mfma_f32_32x32x2_f32 where infinities, NaN or
// rows of tiny elements are in the way), with an error at or below that of the fp32 instruction, sums
// are fp32, and the results follow the reference's fp32 arithmetic.  Same workgroup tile (256 x 256, 2 x 4
// wavefronts), same accumulator layout and same split / combine structure as the 16-bit kernels;
// dZ stays fp32.  All loads are clamped or masked element by element, so any N, H, V >= 1 and any
// element alignment is accepted.  All reductions run in a fixed order: same input, same bits.
#include "rlk_common.hpp"

#include "rlk_gemm.hpp"
#include "rlk_tile_epilogue.hpp"

namespace rlk {

namespace {

constexpr int kWBK = 16;  // K elements per LDS stage

// Element access of the three input types, widened to fp32.
template <int DT>
struct WideElem;

template <>
struct WideElem<RLK_DTYPE_F32> {
    static constexpr int kBytes = 4;
    __device__ static inline float get(const void* p, int64_t i) { return static_cast<const float*>(p)[i]; }
    __device__ static inline f32x4_t get4(const void* p, int64_t i)
    {
        return *reinterpret_cast<const f32x4_t*>(static_cast<const float*>(p) + i);
    }
    __device__ static inline void put(void* p, int64_t i, float v) { static_cast<float*>(p)[i] = v; }
    __device__ static inline void put4(void* p, int64_t i, f32x4_t v)
    {
        *reinterpret_cast<f32x4_t*>(static_cast<float*>(p) + i) = v;
    }
};

template <>
struct WideElem<RLK_DTYPE_BF16> {
    static constexpr int kBytes = 2;
    __device__ static inline float get(const void* p, int64_t i)
    {
        return Bf16::to_float(static_cast<const uint16_t*>(p)[i]);
    }
    __device__ static inline f32x4_t get4(const void* p, int64_t i)
    {
        const u32x2_t w = *reinterpret_cast<const u32x2_t*>(static_cast<const uint16_t*>(p) + i);
        return f32x4_t{__builtin_bit_cast(float, w.x << 16), __builtin_bit_cast(float, w.x & 0xffff0000u),
                       __builtin_bit_cast(float, w.y << 16), __builtin_bit_cast(float, w.y & 0xffff0000u)};
    }
    __device__ static inline void put(void* p, int64_t i, float v)
    {
        static_cast<uint16_t*>(p)[i] = Bf16::from_float(v);
    }
    __device__ static inline void put4(void* p, int64_t i, f32x4_t v)
    {
        *reinterpret_cast<u32x2_t*>(static_cast<uint16_t*>(p) + i) =
            u32x2_t{Bf16::pack2(v.x, v.y), Bf16::pack2(v.z, v.w)};
    }
};

template <>
struct WideElem<RLK_DTYPE_F16> {
    static constexpr int kBytes = 2;
    __device__ static inline float get(const void* p, int64_t i)
    {
        return F16::to_float(static_cast<const uint16_t*>(p)[i]);
    }
    __device__ static inline f32x4_t get4(const void* p, int64_t i)
    {
        const u32x2_t w = *reinterpret_cast<const u32x2_t*>(static_cast<const uint16_t*>(p) + i);
        return f32x4_t{F16::to_float(static_cast<uint16_t>(w.x)), F16::to_float(static_cast<uint16_t>(w.x >> 16)),
                       F16::to_float(static_cast<uint16_t>(w.y)), F16::to_float(static_cast<uint16_t>(w.y >> 16))};
    }
    __device__ static inline void put(void* p, int64_t i, float v)
    {
        static_cast<uint16_t*>(p)[i] = F16::from_float(v);
    }
    __device__ static inline void put4(void* p, int64_t i, f32x4_t v)
    {
        *reinterpret_cast<u32x2_t*>(static_cast<uint16_t*>(p) + i) =
            u32x2_t{F16::pack2(v.x, v.y), F16::pack2(v.z, v.w)};
    }
};

// Operand of one workgroup tile.  `vec`: every group of four consecutive elements along the
// contiguous direction that starts at a multiple of four from `base` is 4-element aligned and may
// be fetched with one load (the leading dimension is a multiple of four and so is the origin).
struct WideOperand {
    const void* base;  // element (row 0, k 0) of the tile
    int64_t ld;        // elements between consecutive memory lines
    int rows;          // valid tile rows from the origin (>= 1)
    bool vec;
};

// One operand's way from global memory into an LDS stage and from there into MFMA fragments.
//   K-contiguous (memory [row][k]):  LDS [256 rows][16 k + 4 pad] floats
//   K-major      (memory [k][row]):  LDS [16 k][256 rows + 4 pad] floats
// The pads make the fragment reads below conflict-free.  A thread moves two groups of four
// consecutive elements per K step.  Rows past `rows` repeat the last valid row (finite values
// that no epilogue stores); elements at k >= K are zeros.
template <int DT, bool KMAJOR>
struct WideIO {
    static constexpr int kPitch = KMAJOR ? 260 : 20;  // floats
    static constexpr int kFloats = KMAJOR ? kWBK * 260 : 256 * 20;
    static constexpr int kBytes = kFloats * 4;
    using E = WideElem<DT>;

    const void* base;
    int64_t off[2];  // element offset of this thread's groups at K step 0 (clamped rows)
    int64_t step;    // element advance per K step
    int rows, K;
    bool vec;

    // FAST (see fast_ok): every group is one aligned 4-element load, no per-element checks.
    static __device__ inline bool fast_ok(const WideOperand& op, int K_)
    {
        return op.vec && K_ % kWBK == 0 && (!KMAJOR || (op.rows & 3) == 0);
    }

    __device__ inline void init(const WideOperand& op, int K_, bool fast)
    {
        base = op.base;
        rows = op.rows;
        K = K_;
        vec = op.vec;
        step = KMAJOR ? static_cast<int64_t>(kWBK) * op.ld : kWBK;
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            const int idx = g * kThreads + static_cast<int>(threadIdx.x);
            if (KMAJOR) {
                const int line = idx >> 6, r = (idx & 63) * 4;
                // past the valid rows: the last valid element, or (FAST) the last valid group
                const int last = fast ? rows - 4 : rows - 1;
                off[g] = static_cast<int64_t>(line) * op.ld + (r < rows ? r : last);
            } else {
                const int row = idx >> 2, k = (idx & 3) * 4;
                off[g] = static_cast<int64_t>(row < rows ? row : rows - 1) * op.ld + k;
            }
        }
    }

    template <bool FAST>
    __device__ inline f32x4_t load(int kt, int g) const
    {
        if (FAST) return E::get4(base, off[g] + kt * step);
        const int idx = g * kThreads + static_cast<int>(threadIdx.x);
        f32x4_t v{0.f, 0.f, 0.f, 0.f};
        if (KMAJOR) {
            const int k = kt * kWBK + (idx >> 6);
            const int r = (idx & 63) * 4;
            if (k < K) {
                const int64_t o = off[g] + kt * step;  // points at min(r, rows - 1) of line k
                if (vec && r + 3 < rows) {
                    v = E::get4(base, o);
                } else {
                    const int64_t line0 = o - (r < rows ? r : rows - 1);
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = E::get(base, line0 + (r + e < rows ? r + e : rows - 1));
                }
            }
        } else {
            const int k = kt * kWBK + (idx & 3) * 4;
            const int64_t o = off[g] + kt * step;
            if (vec && k + 3 < K) {
                v = E::get4(base, o);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (k + e < K) v[e] = E::get(base, o + e);
            }
        }
        return v;
    }

    __device__ static inline void store(float* lds, f32x4_t v, int g)
    {
        const int idx = g * kThreads + static_cast<int>(threadIdx.x);
        const int at = KMAJOR ? (idx >> 6) * kPitch + (idx & 63) * 4 : (idx >> 2) * kPitch + (idx & 3) * 4;
        *reinterpret_cast<f32x4_t*>(lds + at) = v;
    }

    // Half fragment (half = 0, 1) of the 32 tile rows from row0 on: lane l gets row (row0 + l % 32),
    // elements k = 8 * (l / 32) + 4 * half + 0..3 of the stage.  MFMA number j of the stage multiplies
    // element j of the A and B fragments: across the two half-waves that is k = j and k = 8 + j, the
    // same pairing on both operands, so the eight MFMAs together cover the 16 k of the stage once.
    __device__ static inline f32x4_t frag(const float* lds, int row0, int half)
    {
        const int l = threadIdx.x & 63;
        if (KMAJOR) {
            const float* p = lds + (8 * (l >> 5) + 4 * half) * kPitch + row0 + (l & 31);
            return f32x4_t{p[0], p[kPitch], p[2 * kPitch], p[3 * kPitch]};
        } else {
            return *reinterpret_cast<const f32x4_t*>(lds + (row0 + (l & 31)) * kPitch + 8 * (l >> 5) + 4 * half);
        }
    }
};

// Workgroup tile contraction on the fp32 matrix instruction: acc[i][j] += A rows x B rows over
// k in [0, K).  Two LDS stages and one barrier per stage, placed in the middle of the stage's
// MFMAs so that every memory latency has matrix work in front of it:
//   stage kt:  LDS stores of stage kt+1 (fetched one stage ago), global loads of stage kt+2,
//              fragment reads of the second half, 32 MFMAs of the first half,
//              barrier (stage kt+1 is now complete, nobody reads stage kt from LDS any more),
//              fragment reads of the first half of stage kt+1, 32 MFMAs of the second half.
// One MFMA of 32 x 32 x 2 takes 16 passes, so a stage is 4096 matrix cycles per wavefront against a
// dozen fragment reads and 4 global loads: the loop is bound by the matrix pipe.
// All 512 threads must call it (it barriers); on return LDS may be reused.
template <int DTA, int DTB, bool A_KMAJOR, bool B_KMAJOR>
struct WideGemm {
    using IOA = WideIO<DTA, A_KMAJOR>;
    using IOB = WideIO<DTB, B_KMAJOR>;
    static constexpr int kStageFloats = IOA::kFloats + IOB::kFloats;
    static constexpr int kSmemBytes = 2 * kStageFloats * 4;

    __device__ static inline void frags(const float* stage, int wm, int wn, int half, f32x4_t (&fa)[kTM],
                                        f32x4_t (&fb)[kTN])
    {
#pragma unroll
        for (int i = 0; i < kTM; ++i) fa[i] = IOA::frag(stage, wm * (kTM * 32) + i * 32, half);
#pragma unroll
        for (int j = 0; j < kTN; ++j) fb[j] = IOB::frag(stage + IOA::kFloats, wn * (kTN * 32) + j * 32, half);
    }

    __device__ static inline void multiply(const f32x4_t (&fa)[kTM], const f32x4_t (&fb)[kTN],
                                           f32x16_t (&acc)[kTM][kTN])
    {
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
#pragma unroll
            for (int i = 0; i < kTM; ++i)
#pragma unroll
                for (int j = 0; j < kTN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[i][kk], fb[j][kk], acc[i][j], 0, 0, 0);
    }

    __device__ static inline void run(const WideOperand& A, const WideOperand& B, int K,
                                      f32x16_t (&acc)[kTM][kTN], char* smem_c)
    {
        if (IOA::fast_ok(A, K) && IOB::fast_ok(B, K))  // uniform
            run_impl<true>(A, B, K, acc, smem_c);
        else
            run_impl<false>(A, B, K, acc, smem_c);
    }

    template <bool FAST>
    __device__ static inline void run_impl(const WideOperand& A, const WideOperand& B, int K,
                                           f32x16_t (&acc)[kTM][kTN], char* smem_c)
    {
        float* smem = reinterpret_cast<float*>(smem_c);
        IOA la;
        IOB lb;
        la.init(A, K, FAST);
        lb.init(B, K, FAST);
        const int wave = threadIdx.x >> 6;
        const int wm = wave / kWN, wn = wave % kWN;
        const int nk = (K + kWBK - 1) / kWBK;
        f32x4_t ra[2], rb[2];
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            ra[g] = la.template load<FAST>(0, g);
            rb[g] = lb.template load<FAST>(0, g);
        }
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            IOA::store(smem, ra[g], g);
            IOB::store(smem + IOA::kFloats, rb[g], g);
        }
        if (nk > 1) {  // uniform
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                ra[g] = la.template load<FAST>(1, g);
                rb[g] = lb.template load<FAST>(1, g);
            }
        }
        __syncthreads();
        f32x4_t fa0[kTM], fb0[kTN], fa1[kTM], fb1[kTN];
        frags(smem, wm, wn, 0, fa0, fb0);
        for (int kt = 0; kt < nk; ++kt) {
            const float* cur = smem + (kt & 1) * kStageFloats;
            float* nxt = smem + ((kt + 1) & 1) * kStageFloats;
            const bool more = kt + 1 < nk;  // uniform
            if (more) {
#pragma unroll
                for (int g = 0; g < 2; ++g) {
                    IOA::store(nxt, ra[g], g);
                    IOB::store(nxt + IOA::kFloats, rb[g], g);
                }
            }
            if (kt + 2 < nk) {
#pragma unroll
                for (int g = 0; g < 2; ++g) {
                    ra[g] = la.template load<FAST>(kt + 2, g);
                    rb[g] = lb.template load<FAST>(kt + 2, g);
                }
            }
            frags(cur, wm, wn, 1, fa1, fb1);
            multiply(fa0, fb0, acc);
            __syncthreads();
            if (more) frags(nxt, wm, wn, 0, fa0, fb0);
            multiply(fa1, fb1, acc);
        }
        __syncthreads();
    }
};

// The same contraction on the 16-bit matrix instruction, at least as accurate as on the fp32 one.  Every
// element is cut into three bf16 pieces on its way into LDS, x = hi + mid + lo exactly (8 bits and a sign
// each, all by rounding to nearest), and a product is the sum of six of the nine piece products, the
// method of Henry, Tang and Heinecke, "Leveraging the bfloat16 Artificial Intelligence Datatype For
// Higher-Precision Computations" (ARITH 2019).  The three left out are below 2^-24 of the product, most of
// them far below and with random sign (by truncation hi and mid would leave 2^-22).
//
// The matrix instruction does not round its running sum to nearest: added straight into a long sum of
// terms of one sign, the pieces fell 60 and 105 x 2^-24 of the sum short at K = 4096 and 16384.  So the six
// products of a stage, smallest first, make a sum of their own from zero, whose last product alone
// rounds at the size of the result, and one ordinary fp32 addition (to nearest) a stage takes it into the
// accumulator, where the fp32 instruction rounds eight times.  Error of a dot product over sum |a b|, rms
// in units of 2^-24, fp32 instruction -> here: random signs K = 16 0.41 -> 0.25, K = 4096 0.48 -> 0.14; one sign
// K = 16 1.1 -> 0.7, K = 4096 14 -> 3.6, K = 16384 29 -> 7.0.
//
// Bound: the matrix pipe under the board's power limit at six 16-bit products (1450 TFLOP/s sustained / 6
// = 240), next to 0.16 of that time in vector instructions for the pieces and as much again for the
// additions, against 157 TFLOP/s peak of the fp32 instruction.  2048 x 2048 x 32768 forward + backward:
// 8.35 ms on the fp32 instruction, 5.00 with the pieces added straight into the accumulator, 5.63 so (the
// additions of a tile put behind the next tile's products, 32 registers instead of 16, spill: 5.60 against
// 5.37 ms of kernel time).
//
// What pieces cannot hold: an infinity or NaN (they make the sum NaN), a sum that passes the largest
// float on the way, and elements so small that mid and lo fall below bf16's smallest number.  The
// workgroup then computes that tile again on the fp32 instruction: when a result is not finite, and
// when all elements of a row that one thread converted, not all of them zero, are below 2^-95 (where a
// row has larger ones too, what the small ones lose, 2^-126 at most, is nothing next to their sum).
//
//   K-contiguous: LDS [256 rows][3 pieces][16 k]; rows 96 bytes apart: eight rows start in eight
//                 different 16-byte chunks of the 256-byte bank line
//   K-major:      LDS [3 pieces][16 k][256 rows], chunks of k-line k moved by 4 (k & 3): the four k-lines
//                 x 64 bytes of a transposing read cover every bank once
struct Pieces {
    u32x2_t hi, mid, lo;  // four elements each
};

__device__ inline Pieces split3(f32x4_t v)
{
    Pieces p;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const float x0 = v[2 * h], x1 = v[2 * h + 1];
        const uint32_t hi = Bf16::pack2(x0, x1);
        const float r0 = x0 - __builtin_bit_cast(float, hi << 16);
        const float r1 = x1 - __builtin_bit_cast(float, hi & 0xffff0000u);
        const uint32_t mid = Bf16::pack2(r0, r1);
        const float q0 = r0 - __builtin_bit_cast(float, mid << 16);
        const float q1 = r1 - __builtin_bit_cast(float, mid & 0xffff0000u);
        p.hi[h] = hi;
        p.mid[h] = mid;
        p.lo[h] = Bf16::pack2(q0, q1);
    }
    return p;
}

// The bits of all elements that this thread converted of a tile row, or-ed together (K-contiguous: one row
// per group of four elements, K-major: the four rows of its groups).  An exponent of 32 or more, a
// magnitude from 2^-95 on, shows in the exponent's upper three bits whatever else is or-ed in.
template <bool KMAJOR>
struct RowBits {
    static constexpr int kRows = KMAJOR ? 4 : 2;
    uint32_t bits[kRows];

    __device__ inline void reset()
    {
#pragma unroll
        for (uint32_t& b : bits) b = 0;
    }
    __device__ inline void note(f32x4_t v, int g)
    {
#pragma unroll
        for (int e = 0; e < 4; ++e) bits[KMAJOR ? e % kRows : g] |= __builtin_bit_cast(uint32_t, v[e]);
    }
    __device__ inline bool too_small() const
    {
        bool small = false;
#pragma unroll
        for (uint32_t b : bits) small = small || ((b & 0x70000000u) == 0 && (b & 0x7fffffffu) != 0);
        return small;
    }
};

template <bool KMAJOR>
struct SplitLds {
    static constexpr int kPiece = KMAJOR ? kWBK * 512 : 32;  // bytes between the pieces of an element
    static constexpr int kBytes = 256 * 3 * kWBK * 2;

    __device__ static inline void store(char* lds, const Pieces& v, int g)
    {
        const int idx = g * kThreads + static_cast<int>(threadIdx.x);
        const int k = idx >> 6, q = idx & 63;  // K-major: k-line, group of four rows
        char* at = lds + (KMAJOR ? k * 512 + ((q >> 1) ^ ((k & 3) << 2)) * 16 + (q & 1) * 8
                                 : (idx >> 2) * 96 + (idx & 3) * 8);
        *reinterpret_cast<u32x2_t*>(at) = v.hi;
        *reinterpret_cast<u32x2_t*>(at + kPiece) = v.mid;
        *reinterpret_cast<u32x2_t*>(at + 2 * kPiece) = v.lo;
    }

    // MFMA 32x32x16 operand fragment: lane l holds row (row0 + l % 32), k = 8 (l / 32) + 0..7
    // (row0 a multiple of 32).
    __device__ static inline bf16x8_t frag(const char* lds, int row0, int piece)
    {
        const int l = threadIdx.x & 63;
        if (KMAJOR) {
            const int a = (l & 15) >> 2, b = l & 3;  // see TileIO::frag
            const int c = (row0 >> 3) + 2 * ((l >> 4) & 1) + (b >> 1);
            const char* p0 = lds + piece * kPiece + (8 * (l >> 5) + a) * 512 + (c ^ (a << 2)) * 16 + (b & 1) * 8;
            const s16x4_t x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((RLK_LDS s16x4_t*)(p0));
            const s16x4_t y = __builtin_amdgcn_ds_read_tr16_b64_v4i16((RLK_LDS s16x4_t*)(p0 + 4 * 512));
            const u32x2_t x2 = __builtin_bit_cast(u32x2_t, x), y2 = __builtin_bit_cast(u32x2_t, y);
            return __builtin_bit_cast(bf16x8_t, u32x4_t{x2.x, x2.y, y2.x, y2.y});
        } else {
            return *reinterpret_cast<const bf16x8_t*>(lds + (row0 + (l & 31)) * 96 + piece * kPiece + 16 * (l >> 5));
        }
    }
};

template <int DTA, int DTB, bool A_KMAJOR, bool B_KMAJOR>
struct SplitGemm {
    using Exact = WideGemm<DTA, DTB, A_KMAJOR, B_KMAJOR>;
    using IOA = typename Exact::IOA;
    using IOB = typename Exact::IOB;
    using LA = SplitLds<A_KMAJOR>;
    using LB = SplitLds<B_KMAJOR>;
    static constexpr int kStageBytes = LA::kBytes + LB::kBytes;
    static constexpr int kStages = 3;
    static constexpr int kSmemBytes = kStages * kStageBytes;
    static_assert(kSmemBytes >= Exact::kSmemBytes, "the fp32 loop runs in the same LDS");
    typedef bf16x8_t Frag[3];  // hi, mid, lo

    __device__ static inline void run(const WideOperand& A, const WideOperand& B, int K,
                                      f32x16_t (&acc)[kTM][kTN], char* smem)
    {
        bool again;
        if (IOA::fast_ok(A, K) && IOB::fast_ok(B, K))  // uniform
            again = run_impl<true>(A, B, K, acc, smem);
        else
            again = run_impl<false>(A, B, K, acc, smem);
        if (__syncthreads_or(again)) {
            zero_acc(acc);
            Exact::template run_impl<false>(A, B, K, acc, smem);
        }
    }

    // One 32 x 32 tile's share of a stage, added to `out` as one number.
    __device__ static inline void product(const Frag& a, const Frag& b, f32x16_t& out)
    {
        auto mul = [](bf16x8_t x, bf16x8_t y, f32x16_t c) {
            return __builtin_amdgcn_mfma_f32_32x32x16_bf16(x, y, c, 0, 0, 0);
        };
        f32x16_t acc = {};
        acc = mul(a[2], b[0], acc);
        acc = mul(a[0], b[2], acc);
        acc = mul(a[1], b[1], acc);
        acc = mul(a[1], b[0], acc);
        acc = mul(a[0], b[1], acc);
        acc = mul(a[0], b[0], acc);
        out += acc;
    }

    // Stage kt multiplies while stage kt + 2 is converted into the LDS stage that kt - 1 has left and
    // the first fragments of stage kt + 1 (published by the last barrier) are read, so that neither
    // conversions nor LDS latency stand in front of the matrix work behind a barrier.
    // Returns whether this thread has a reason to compute the tile again on the fp32 instruction.
    template <bool FAST>
    __device__ static inline bool run_impl(const WideOperand& A, const WideOperand& B, int K,
                                            f32x16_t (&acc)[kTM][kTN], char* smem)
    {
        IOA la;
        IOB lb;
        la.init(A, K, FAST);
        lb.init(B, K, FAST);
        const int wave = threadIdx.x >> 6;
        const int ra0 = (wave / kWN) * (kTM * 32), rb0 = (wave % kWN) * (kTN * 32);
        const int nk = (K + kWBK - 1) / kWBK;
        RowBits<A_KMAJOR> pa;
        RowBits<B_KMAJOR> pb;
        pa.reset();
        pb.reset();
        f32x4_t reg[4];  // groups 0, 1 of A and 0, 1 of B
        auto fetch = [&](int kt, int n) {
            reg[n] = n < 2 ? la.template load<FAST>(kt, n) : lb.template load<FAST>(kt, n - 2);
        };
        auto convert = [&](char* stage, int n) {
            if (n < 2) {
                pa.note(reg[n], n);
                LA::store(stage, split3(reg[n]), n);
            } else {
                pb.note(reg[n], n - 2);
                LB::store(stage + LA::kBytes, split3(reg[n]), n - 2);
            }
        };
        auto stage_at = [&](int st) { return smem + st * kStageBytes; };
        // stages 0 and 1 in LDS, stage 2 on its way (past the last stage: the last one again)
        for (int kt = 0; kt < 2; ++kt) {
#pragma unroll
            for (int n = 0; n < 4; ++n) fetch(min(kt, nk - 1), n);
#pragma unroll
            for (int n = 0; n < 4; ++n) convert(stage_at(kt), n);
        }
#pragma unroll
        for (int n = 0; n < 4; ++n) fetch(min(2, nk - 1), n);
        __syncthreads();
        Frag fa[2], fb[kTN];
        auto read_a = [&](Frag& f, const char* stage, int i) {
#pragma unroll
            for (int p = 0; p < 3; ++p) f[p] = LA::frag(stage, ra0 + i * 32, p);
        };
        auto read_b = [&](Frag& f, const char* stage, int j) {
#pragma unroll
            for (int p = 0; p < 3; ++p) f[p] = LB::frag(stage + LA::kBytes, rb0 + j * 32, p);
        };
#pragma unroll
        for (int j = 0; j < kTN; ++j) read_b(fb[j], stage_at(0), j);
        read_a(fa[0], stage_at(0), 0);
        int cur = 0;
        for (int kt = 0; kt < nk; ++kt) {
            const int nxt = cur + 1 == kStages ? 0 : cur + 1, dst = nxt + 1 == kStages ? 0 : nxt + 1;
            const int ahead = min(kt + 3, nk - 1);
            static_for<0, kTM>([&](auto ic) {
                constexpr int i = decltype(ic)::value;
                if constexpr (i + 1 < kTM)
                    read_a(fa[(i + 1) & 1], stage_at(cur), i + 1);
                else
                    read_a(fa[(i + 1) & 1], stage_at(nxt), 0);
                static_for<0, kTN>([&](auto jc) {
                    constexpr int j = decltype(jc)::value;
                    product(fa[i & 1], fb[j], acc[i][j]);
                    if constexpr (i + 1 == kTM) read_b(fb[j], stage_at(nxt), j);
                    if constexpr (j == 0) {
                        convert(stage_at(dst), i);
                        fetch(ahead, i);
                    }
                    // the addition stays here (sunk below the next products it costs 300 registers)
                    asm volatile("" : "+v"(acc[i][j]));
                });
            });
            __syncthreads();
            cur = nxt;
        }
        float zero = 0.f;  // 0 * finite = 0; NaN once a result is infinite or NaN
#pragma unroll
        for (int i = 0; i < kTM; ++i)
#pragma unroll
            for (int j = 0; j < kTN; ++j)
#pragma unroll
                for (int r = 0; r < Acc32::kRegs; ++r) zero = fmaf(acc[i][j][r], 0.f, zero);
        return zero != 0.f || pa.too_small() || pb.too_small();
    }
};

// ------------------------------------------------------------------------------------------- //
// Forward: partial softmax states of one (256-token block) x (range of vocab tiles)
// ------------------------------------------------------------------------------------------- //
struct WideFwdArgs {
    const void* hidden;  // [N][H]
    const void* weight;  // [V][H]
    const float* bias;   // [V] or null
    const int64_t* targets;
    float* part_m;       // [n_split][N]  running max (log2 domain)
    float* part_s;       // [n_split][N]  running sum of 2^(z - max)
    float* part_z;       // [n_split][N]  captured target logit (log2 domain), 0 if not owned
    int N;
    int H;
    int V;
    int64_t vocab_start;
    int n_split;
    int row_blocks;
    int vtiles;
    float scale2;  // log2(e) / temperature
    bool vec_h, vec_w;
    float* kept;  // KEEP: logits (bias added) for the backward, [N][ldz]
    int64_t ldz;
};

template <int DT, bool KEEP>
__global__ __launch_bounds__(kThreads) void wide_fwd_kernel(WideFwdArgs a)
{
    using Gemm = SplitGemm<DT, DT, false, false>;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    int tb, sp;
    xcd_tile(blockIdx.x, a.row_blocks * a.n_split, a.row_blocks, a.n_split, 8, tb, sp);
    const int base = a.vtiles / a.n_split, extra = a.vtiles % a.n_split;
    const int t0 = sp * base + (sp < extra ? sp : extra);
    const int t1 = t0 + base + (sp < extra ? 1 : 0);

    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int wm = wave / kWN, wn = wave % kWN;
    const int tok0 = tb * 256;
    const int tok_valid = min(256, a.N - tok0);

    float m[kTN], s[kTN], zt[kTN];
    int tgt[kTN];  // target id relative to the shard, -1 when not in [0, V)
#pragma unroll
    for (int j = 0; j < kTN; ++j) {
        const int t = wn * (kTN * 32) + j * 32 + (lane & 31);
        const int64_t g = a.targets[tok0 + (t < tok_valid ? t : tok_valid - 1)] - a.vocab_start;
        tgt[j] = (g >= 0 && g < a.V) ? static_cast<int>(g) : -1;
        m[j] = -INFINITY;
        s[j] = 0.f;
        zt[j] = 0.f;
    }
    const WideOperand B{static_cast<const char*>(a.hidden) +
                            static_cast<int64_t>(tok0) * a.H * WideElem<DT>::kBytes,
                        a.H, tok_valid, a.vec_h};
    for (int vt = t0; vt < t1; ++vt) {
        const int v0 = vt * 256;
        const WideOperand A{static_cast<const char*>(a.weight) +
                                static_cast<int64_t>(v0) * a.H * WideElem<DT>::kBytes,
                            a.H, min(256, a.V - v0), a.vec_w};
        f32x16_t acc[kTM][kTN];
        zero_acc(acc);
        Gemm::run(A, B, a.H, acc, smem);
        if constexpr (KEEP) {
#pragma unroll
            for (int j = 0; j < kTN; ++j) {
                const int tl = wn * (kTN * 32) + j * 32 + (lane & 31);
                float* row = a.kept + static_cast<int64_t>(tok0 + min(tl, tok_valid - 1)) * a.ldz;
#pragma unroll
                for (int i = 0; i < kTM; ++i)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const int v = v0 + wm * (kTM * 32) + Acc32::quad_row(i, q, lane);
                        f32x4_t z;
#pragma unroll
                        for (int c = 0; c < 4; ++c) {
                            z[c] = acc[i][j][q * 4 + c];
                            if (a.bias != nullptr) z[c] += a.bias[v + c < a.V ? v + c : a.V - 1];
                        }
                        // ldz is a multiple of 4 >= V: a quad that starts below V ends below ldz
                        if (tl < tok_valid && v < a.V) *reinterpret_cast<f32x4_t*>(row + v) = z;
                    }
            }
        }
        fwd_epilogue<true, Acc32>(acc, a, a.bias, v0 + wm * (kTM * 32), v0, lane, tgt, m, s, zt);
    }

    // merge: the two half-wave row groups of a token, then the wavefronts along M (fixed order)
    float* red = reinterpret_cast<float*>(smem);  // [kWM][256 tokens][3]; the GEMM has left LDS
#pragma unroll
    for (int j = 0; j < kTN; ++j) {
        const float m2 = __shfl_xor(m[j], 32);
        const float s2 = __shfl_xor(s[j], 32);
        const float z2 = __shfl_xor(zt[j], 32);
        const float mm = fmaxf(m[j], m2);
        const float mref = mm == -INFINITY ? 0.f : mm;
        const float lo_m = lane < 32 ? m[j] : m2, hi_m = lane < 32 ? m2 : m[j];
        const float lo_s = lane < 32 ? s[j] : s2, hi_s = lane < 32 ? s2 : s[j];
        const float ss = lo_s * __builtin_amdgcn_exp2f(lo_m - mref) + hi_s * __builtin_amdgcn_exp2f(hi_m - mref);
        if (lane < 32) {
            float* dst = red + ((wm * 256) + wn * (kTN * 32) + j * 32 + lane) * 3;
            dst[0] = mm;
            dst[1] = ss;
            dst[2] = zt[j] + z2;
        }
    }
    __syncthreads();
    const int t = threadIdx.x;
    if (t < tok_valid) {
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
        const int64_t o = static_cast<int64_t>(sp) * a.N + tok0 + t;
        a.part_m[o] = mm;
        a.part_s[o] = ss;
        a.part_z[o] = zz;
    }
}

// ------------------------------------------------------------------------------------------- //
// Backward step 1: fp32 dZ[tok][v] = g/T * (onehot - softmax) for one token chunk, whole vocab
// ------------------------------------------------------------------------------------------- //
struct WideDzArgs {
    const void* hidden;      // chunk origin [tok][H]
    const void* weight;      // [V][H]
    const float* bias;       // [V] or null
    const int64_t* targets;  // chunk origin (global ids)
    const float* lse;        // chunk origin (natural log)
    const float* grad;       // chunk origin, upstream d/dlogp
    float* dz;               // [tok][ldz], ldz a multiple of 4, 16-byte aligned
    int64_t ldz;
    int tok_valid;
    int V;
    int H;
    int tok_tiles;
    int v_tiles;
    int64_t vocab_start;
    int64_t ignore_index;
    int use_ignore;
    float scale2;  // log2(e) / temperature
    float inv_t;
    bool vec_h, vec_w;
};

template <int DT>
__global__ __launch_bounds__(kThreads) void wide_dz_kernel(WideDzArgs a)
{
    using Gemm = SplitGemm<DT, DT, false, false>;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int wm = wave / kWN, wn = wave % kWN;
    const int hi = lane >> 5;
    for (TileWalk walk(a.tok_tiles * a.v_tiles, a.v_tiles, a.tok_tiles); walk.valid(); walk.advance()) {
        int vt, tt;
        walk.coords(false, vt, tt);
        const int tok0 = tt * 256, v0 = vt * 256;
        const int tok_rows = min(256, a.tok_valid - tok0);
        const WideOperand A{static_cast<const char*>(a.weight) +
                                static_cast<int64_t>(v0) * a.H * WideElem<DT>::kBytes,
                            a.H, min(256, a.V - v0), a.vec_w};
        const WideOperand B{static_cast<const char*>(a.hidden) +
                                static_cast<int64_t>(tok0) * a.H * WideElem<DT>::kBytes,
                            a.H, tok_rows, a.vec_h};
        f32x16_t acc[kTM][kTN];
        zero_acc(acc);
        Gemm::run(A, B, a.H, acc, smem);

        const int vw = v0 + wm * (kTM * 32);
#pragma unroll
        for (int j = 0; j < kTN; ++j) {
            const int tl = wn * (kTN * 32) + j * 32 + (lane & 31);
            const bool in = tl < tok_rows;
            const int tc = tok0 + (in ? tl : tok_rows - 1);
            const int64_t tg = a.targets[tc];
            const bool live = in && !(a.use_ignore && tg == a.ignore_index);
            const float gs = live ? a.grad[tc] * a.inv_t : 0.f;
            const float nlse2 = -a.lse[tc] * kLog2e;
            const int64_t trel = tg - a.vocab_start;  // row of the shard, any value when not owned
            float* row = a.dz + static_cast<int64_t>(tc) * a.ldz;
#pragma unroll
            for (int i = 0; i < kTM; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int v = vw + i * 32 + 8 * q + 4 * hi;  // first of four consecutive rows
                    f32x4_t d;
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        const int vc = v + c;
                        float z = acc[i][j][q * 4 + c];
                        if (a.bias != nullptr) z += a.bias[vc < a.V ? vc : a.V - 1];
                        const float p = vc < a.V ? __builtin_amdgcn_exp2f(fmaf(z, a.scale2, nlse2)) : 0.f;
                        d[c] = gs * ((trel == vc ? 1.f : 0.f) - p);
                    }
                    // ldz is a multiple of 4 >= V: a quad that starts below V ends below ldz
                    if (in && v < a.V) *reinterpret_cast<f32x4_t*>(row + v) = d;
                }
        }
    }
}

// dZ from the logits that the forward kept, in place: the same expressions as above on one pass over memory
// (8 bytes per logit against six products of H terms).  A workgroup takes 256 columns of 64 tokens, a thread
// four of them of every fourth token.  db_part (or null): column sums of the 64 tokens for d_bias,
// [slab][ldz].  MAKE = false: `kept` is dZ already (computed again, nothing was kept) and only its column sums are
// taken, in the same order.
struct WideKeptArgs {
    float* kept;  // [N][ldz]
    const int64_t* targets;
    const float* lse;
    const float* grad;
    float* db_part;
    int64_t ldz;
    int N;
    int V;
    int64_t vocab_start;
    int64_t ignore_index;
    int use_ignore;
    float scale2;
    float inv_t;
};

constexpr int kWideSlab = 64;  // tokens
template <bool MAKE>
__global__ __launch_bounds__(256) void wide_dz_kept_kernel(WideKeptArgs a)
{
    const int v = blockIdx.x * 256 + (threadIdx.x & 63) * 4;
    const int wave = threadIdx.x >> 6, lo = blockIdx.y * kWideSlab;
    f32x4_t sum{0.f, 0.f, 0.f, 0.f};
    if (v < a.V) {
#pragma unroll 4
        for (int t = lo + wave; t < min(lo + kWideSlab, a.N); t += 4) {
            f32x4_t* p = reinterpret_cast<f32x4_t*>(a.kept + static_cast<int64_t>(t) * a.ldz + v);
            if constexpr (!MAKE) {
                const f32x4_t made = *p;
#pragma unroll
                for (int c = 0; c < 4; ++c) sum[c] += v + c < a.V ? made[c] : 0.f;
                continue;
            }
            const int64_t tg = a.targets[t];
            const bool live = !(a.use_ignore && tg == a.ignore_index);
            const float gs = live ? a.grad[t] * a.inv_t : 0.f;
            const float nlse2 = -a.lse[t] * kLog2e;
            const int64_t trel = tg - a.vocab_start;
            const f32x4_t z = *p;
            f32x4_t d;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const float pr = v + c < a.V ? __builtin_amdgcn_exp2f(fmaf(z[c], a.scale2, nlse2)) : 0.f;
                d[c] = gs * ((trel == v + c ? 1.f : 0.f) - pr);
            }
            *p = d;
            // the sums take the rounded values that dW takes: no product may be contracted into them
            asm volatile("" : "+v"(d));
            sum += d;
        }
    }
    if (a.db_part == nullptr) return;  // uniform
    __shared__ f32x4_t red[4][64];
    red[wave][threadIdx.x & 63] = sum;
    __syncthreads();
    if (wave == 0 && v < a.V) {
        for (int w = 1; w < 4; ++w) sum += red[w][threadIdx.x];
        *reinterpret_cast<f32x4_t*>(a.db_part + blockIdx.y * a.ldz + v) = sum;
    }
}

// Slabs in ascending order.
__global__ void wide_db_finish_kernel(const float* part, int64_t ld, int slabs, int V, float* db, int accumulate)
{
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= V) return;
    float sum = part[v];
#pragma unroll 8
    for (int s = 1; s < slabs; ++s) sum += part[s * ld + v];
    db[v] = accumulate ? db[v] + sum : sum;
}

// ------------------------------------------------------------------------------------------- //
// Backward step 2: dH[tok][h] = sum_v dZ[tok][v] W[v][h]   (M = h, N = token, K = vocab)
// The vocab range is cut into `ksplit` parts that run side by side into separate fp32 slots,
// added in slot order by wide_dh_reduce_kernel.
// ------------------------------------------------------------------------------------------- //
struct WideDhArgs {
    const float* dz;     // [tok][ldz]
    int64_t ldz;
    const void* weight;  // [V][H]
    float* part;         // [ksplit][tok_valid][H]
    int64_t slot_stride;
    int H;
    int V;
    int tok_valid;
    int h_tiles;
    int tok_tiles;
    int ksplit;
    int k_per;  // vocab rows per slot (multiple of 16)
    bool vec_w;
};

template <int DT>
__global__ __launch_bounds__(kThreads) void wide_dh_kernel(WideDhArgs a)
{
    using Gemm = SplitGemm<DT, RLK_DTYPE_F32, true, false>;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tiles = a.h_tiles * a.tok_tiles;
    const int slot = blockIdx.x / tiles;
    int ht, tt;
    xcd_tile(blockIdx.x % tiles, tiles, a.h_tiles, a.tok_tiles, 8, ht, tt);
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int wm = wave / kWN, wn = wave % kWN;
    const int h0 = ht * 256, tok0 = tt * 256;
    const int k_lo = slot * a.k_per;
    const int k_n = min(a.k_per, a.V - k_lo);
    const int tok_rows = min(256, a.tok_valid - tok0);
    f32x16_t acc[kTM][kTN];
    zero_acc(acc);
    if (k_n > 0) {  // uniform
        const WideOperand A{static_cast<const char*>(a.weight) +
                                (static_cast<int64_t>(k_lo) * a.H + h0) * WideElem<DT>::kBytes,
                            a.H, min(256, a.H - h0), a.vec_w};
        const WideOperand B{a.dz + static_cast<int64_t>(tok0) * a.ldz + k_lo, a.ldz, tok_rows, true};
        Gemm::run(A, B, k_n, acc, smem);
    }
    float* out = a.part + static_cast<int64_t>(slot) * a.slot_stride;
    const bool vec = (a.H & 3) == 0;
#pragma unroll
    for (int j = 0; j < kTN; ++j) {
        const int tl = wn * (kTN * 32) + j * 32 + (lane & 31);
        if (tl >= tok_rows) continue;
        float* row = out + static_cast<int64_t>(tok0 + tl) * a.H;
#pragma unroll
        for (int i = 0; i < kTM; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int h = h0 + wm * (kTM * 32) + i * 32 + 8 * q + 4 * (lane >> 5);
                const f32x4_t v{acc[i][j][q * 4 + 0], acc[i][j][q * 4 + 1], acc[i][j][q * 4 + 2],
                                acc[i][j][q * 4 + 3]};
                if (vec) {
                    if (h < a.H) *reinterpret_cast<f32x4_t*>(row + h) = v;
                } else {
#pragma unroll
                    for (int c = 0; c < 4; ++c)
                        if (h + c < a.H) row[h + c] = v[c];
                }
            }
    }
}

template <int DT>
__global__ void wide_dh_reduce_kernel(const float* part, int64_t slot_stride, int ksplit, void* out, int64_t n)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float acc = part[i];
    for (int sl = 1; sl < ksplit; ++sl) acc += part[sl * slot_stride + i];
    WideElem<DT>::put(out, i, acc);
}

// ------------------------------------------------------------------------------------------- //
// Backward step 3: dW[v][h] (+)= sum_tok dZ[tok][v] hidden[tok][h]   (M = h, N = vocab, K = token)
// ------------------------------------------------------------------------------------------- //
struct WideDwArgs {
    const float* dz;     // [tok][ldz]
    int64_t ldz;
    const void* hidden;  // chunk origin [tok][H]
    float* dw;           // [V][H] fp32
    int H;
    int V;
    int tok_valid;
    int v_tiles;
    int h_tiles;
    int accumulate;  // 1: dw += ..., 0: dw = ...
    bool vec_h;
};

template <int DT>
__global__ __launch_bounds__(kThreads) void wide_dw_kernel(WideDwArgs a)
{
    using Gemm = SplitGemm<DT, RLK_DTYPE_F32, true, true>;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int wm = wave / kWN, wn = wave % kWN;
    const bool vec = (a.H & 3) == 0 && (reinterpret_cast<uintptr_t>(a.dw) & 15) == 0;
    for (TileWalk walk(a.v_tiles * a.h_tiles, a.v_tiles, a.h_tiles); walk.valid(); walk.advance()) {
        int vt, ht;
        walk.coords(false, vt, ht);
        const int v0 = vt * 256, h0 = ht * 256;
        const WideOperand A{static_cast<const char*>(a.hidden) + static_cast<int64_t>(h0) * WideElem<DT>::kBytes,
                            a.H, min(256, a.H - h0), a.vec_h};
        const WideOperand B{a.dz + v0, a.ldz, min(256, a.V - v0), true};
        f32x16_t acc[kTM][kTN];
        zero_acc(acc);
        Gemm::run(A, B, a.tok_valid, acc, smem);
#pragma unroll
        for (int j = 0; j < kTN; ++j) {
            const int v = v0 + wn * (kTN * 32) + j * 32 + (lane & 31);
            if (v >= a.V) continue;
            float* row = a.dw + static_cast<int64_t>(v) * a.H;
#pragma unroll
            for (int i = 0; i < kTM; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int h = h0 + wm * (kTM * 32) + i * 32 + 8 * q + 4 * (lane >> 5);
                    f32x4_t val{acc[i][j][q * 4 + 0], acc[i][j][q * 4 + 1], acc[i][j][q * 4 + 2],
                                acc[i][j][q * 4 + 3]};
                    if (vec) {
                        if (h < a.H) {
                            if (a.accumulate) val += *reinterpret_cast<const f32x4_t*>(row + h);
                            *reinterpret_cast<f32x4_t*>(row + h) = val;
                        }
                    } else {
#pragma unroll
                        for (int c = 0; c < 4; ++c)
                            if (h + c < a.H) row[h + c] = a.accumulate ? row[h + c] + val[c] : val[c];
                    }
                }
        }
    }
}

// db[v] (+)= sum_tok dZ[tok][v], tokens in ascending order.
__global__ void wide_db_kernel(const float* dz, int64_t ldz, int tok_valid, int V, float* db, int accumulate)
{
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= V) return;
    float acc = 0.f;
    for (int t = 0; t < tok_valid; ++t) acc += dz[static_cast<int64_t>(t) * ldz + v];
    db[v] = accumulate ? db[v] + acc : acc;
}

// ------------------------------------------------------------------------------------------- //
// Host side
// ------------------------------------------------------------------------------------------- //
template <class K>
int wide_smem(K kernel, int bytes)
{
    return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                               hipFuncAttributeMaxDynamicSharedMemorySize, bytes) == hipSuccess
               ? 0
               : rlk_fail(RLK_ERR_LAUNCH, "cannot raise the kernel's LDS limit");
}

int wide_check(const char* what)
{
    return hipGetLastError() == hipSuccess ? 0 : rlk_fail(RLK_ERR_LAUNCH, what);
}

// Four consecutive elements of a row may be fetched with one load when the matrix starts on a
// 4-element boundary and every row does (leading dimension a multiple of four).
bool quad_aligned(const void* p, int64_t ld, int dtype)
{
    const uintptr_t mask = dtype == RLK_DTYPE_F32 ? 15 : 7;
    return (reinterpret_cast<uintptr_t>(p) & mask) == 0 && (ld & 3) == 0;
}

size_t align256(size_t x) { return (x + 255) / 256 * 256; }

struct WidePlan {
    int64_t chunk;  // tokens per dZ block (multiple of 256, or all N)
    int64_t ldz;
    int ksplit;
    int k_per;
    size_t dz_bytes, part_bytes, db_bytes, total;
};

WidePlan wide_plan(int64_t N, int32_t H, int64_t V, size_t budget)
{
    WidePlan p;
    p.ldz = (V + 3) / 4 * 4;
    const int64_t n_up = (N + 255) / 256 * 256;
    int64_t chunk = static_cast<int64_t>(budget / (static_cast<size_t>(p.ldz) * 4)) / 256 * 256;
    // the fp32 dH slots of a chunk (at least one, chunk x H) stay within half the budget
    const int64_t chunk_h = static_cast<int64_t>(budget / 2 / (static_cast<size_t>(H) * 4)) / 256 * 256;
    if (chunk > chunk_h) chunk = chunk_h;
    if (chunk < 256) chunk = 256;
    if (chunk > n_up) chunk = n_up;
    p.chunk = chunk;
    // dH launch: enough vocab parts to give every compute unit a tile, each at least 64 stages long
    const int64_t tiles = ((H + 255) / 256) * (chunk / 256);
    int64_t ks = (256 + tiles - 1) / tiles;
    const int64_t ks_max = (V + 1023) / 1024;
    if (ks > ks_max) ks = ks_max;
    if (ks > 32) ks = 32;
    if (ks < 1) ks = 1;
    int64_t k_per = ((V + ks - 1) / ks + 15) / 16 * 16;
    ks = (V + k_per - 1) / k_per;
    p.ksplit = static_cast<int>(ks);
    p.k_per = static_cast<int>(k_per);
    p.dz_bytes = align256(static_cast<size_t>(chunk) * p.ldz * 4);
    p.part_bytes = align256(static_cast<size_t>(p.ksplit) * chunk * H * 4);
    p.db_bytes = 0;
    p.total = p.dz_bytes + p.part_bytes;
    return p;
}

// Backward from kept logits: the chunks of the default budget, so that the sums are grouped as without; dZ lies in
// the place of the logits.  again: none were kept, dZ is computed into the workspace.
WidePlan wide_kept_plan(int64_t N, int32_t H, int64_t V, bool again)
{
    WidePlan p = wide_plan(N, H, V, RLK_DEFAULT_DZ_BUDGET);
    if (!again) p.dz_bytes = 0;
    p.db_bytes = align256(static_cast<size_t>(p.chunk + kWideSlab - 1) / kWideSlab * p.ldz * 4);
    p.total = p.dz_bytes + p.part_bytes + p.db_bytes;
    return p;
}

template <int DT, bool KEEP = false>
int wide_fwd_launch(const WideFwdArgs& a, hipStream_t stream)
{
    using G = SplitGemm<DT, DT, false, false>;
    if (int rc = wide_smem(wide_fwd_kernel<DT, KEEP>, G::kSmemBytes)) return rc;
    hipLaunchKernelGGL((wide_fwd_kernel<DT, KEEP>), dim3(a.row_blocks * a.n_split), dim3(kThreads), G::kSmemBytes,
                       stream, a);
    return wide_check("wide_fwd_kernel launch failed");
}

template <int DT>
int wide_bwd_launch(const float* grad_logp, const void* hidden, const void* weight, const float* bias,
                    const int64_t* targets, const float* lse, void* d_hidden, float* d_weight,
                    float* d_bias, float* kept, void* workspace, const WidePlan& p, int64_t N, int32_t H, int64_t V,
                    int64_t vocab_start, float temperature, int64_t ignore_index, int32_t use_ignore,
                    int32_t accumulate, hipStream_t stream)
{
    using GZ = SplitGemm<DT, DT, false, false>;
    using GH = SplitGemm<DT, RLK_DTYPE_F32, true, false>;
    using GW = SplitGemm<DT, RLK_DTYPE_F32, true, true>;
    if (int rc = wide_smem(wide_dz_kernel<DT>, GZ::kSmemBytes)) return rc;
    if (int rc = wide_smem(wide_dh_kernel<DT>, GH::kSmemBytes)) return rc;
    if (int rc = wide_smem(wide_dw_kernel<DT>, GW::kSmemBytes)) return rc;
    constexpr int esz = WideElem<DT>::kBytes;
    float* dz = static_cast<float*>(workspace);
    float* part = reinterpret_cast<float*>(static_cast<char*>(workspace) + p.dz_bytes);
    float* db_part = p.db_bytes && d_bias
                         ? reinterpret_cast<float*>(static_cast<char*>(workspace) + p.dz_bytes + p.part_bytes) : nullptr;
    const int v_tiles = static_cast<int>((V + 255) / 256);
    const int h_tiles = (H + 255) / 256;
    const bool vec_h = quad_aligned(hidden, H, DT), vec_w = quad_aligned(weight, H, DT);
    for (int64_t t0 = 0; t0 < N; t0 += p.chunk) {
        const int nt = static_cast<int>(N - t0 < p.chunk ? N - t0 : p.chunk);
        const int tok_tiles = (nt + 255) / 256;
        const void* hid = static_cast<const char*>(hidden) + t0 * H * esz;
        if (kept) dz = kept + t0 * p.ldz;
        const int slabs = (nt + kWideSlab - 1) / kWideSlab;
        WideDzArgs z;
        z.hidden = hid;
        z.weight = weight;
        z.bias = bias;
        z.targets = targets + t0;
        z.lse = lse + t0;
        z.grad = grad_logp + t0;
        z.dz = dz;
        z.ldz = p.ldz;
        z.tok_valid = nt;
        z.V = static_cast<int>(V);
        z.H = H;
        z.tok_tiles = tok_tiles;
        z.v_tiles = v_tiles;
        z.vocab_start = vocab_start;
        z.ignore_index = ignore_index;
        z.use_ignore = use_ignore;
        z.scale2 = kLog2e / temperature;
        z.inv_t = 1.f / temperature;
        z.vec_h = vec_h;
        z.vec_w = vec_w;
        const WideKeptArgs k{dz, z.targets, z.lse, z.grad, db_part, p.ldz, nt, z.V, vocab_start,
                             ignore_index, use_ignore, z.scale2, z.inv_t};
        if (kept) {
            hipLaunchKernelGGL(wide_dz_kept_kernel<true>, dim3(v_tiles, slabs), dim3(256), 0, stream, k);
        } else {
            hipLaunchKernelGGL(wide_dz_kernel<DT>, dim3(tok_tiles * v_tiles), dim3(kThreads), GZ::kSmemBytes, stream, z);
            if (db_part)
                hipLaunchKernelGGL(wide_dz_kept_kernel<false>, dim3(v_tiles, slabs), dim3(256), 0, stream, k);
        }
        if (d_hidden) {
            WideDhArgs h;
            h.dz = dz;
            h.ldz = p.ldz;
            h.weight = weight;
            h.part = part;
            h.slot_stride = static_cast<int64_t>(nt) * H;
            h.H = H;
            h.V = static_cast<int>(V);
            h.tok_valid = nt;
            h.h_tiles = h_tiles;
            h.tok_tiles = tok_tiles;
            h.ksplit = p.ksplit;
            h.k_per = p.k_per;
            h.vec_w = vec_w;
            hipLaunchKernelGGL(wide_dh_kernel<DT>, dim3(h_tiles * tok_tiles * p.ksplit), dim3(kThreads),
                               GH::kSmemBytes, stream, h);
            const int64_t n = static_cast<int64_t>(nt) * H;
            hipLaunchKernelGGL(wide_dh_reduce_kernel<DT>, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256),
                               0, stream, part, h.slot_stride, p.ksplit,
                               static_cast<char*>(d_hidden) + t0 * H * esz, n);
        }
        const int acc = (t0 > 0 || accumulate) ? 1 : 0;
        if (d_weight) {
            WideDwArgs w;
            w.dz = dz;
            w.ldz = p.ldz;
            w.hidden = hid;
            w.dw = d_weight;
            w.H = H;
            w.V = static_cast<int>(V);
            w.tok_valid = nt;
            w.v_tiles = v_tiles;
            w.h_tiles = h_tiles;
            w.accumulate = acc;
            w.vec_h = vec_h;
            hipLaunchKernelGGL(wide_dw_kernel<DT>, dim3(v_tiles * h_tiles), dim3(kThreads), GW::kSmemBytes, stream, w);
        }
        if (db_part)
            hipLaunchKernelGGL(wide_db_finish_kernel, dim3(static_cast<unsigned>((V + 255) / 256)), dim3(256), 0, stream,
                               db_part, p.ldz, slabs, static_cast<int>(V), d_bias, acc);
        else if (d_bias)
            hipLaunchKernelGGL(wide_db_kernel, dim3(static_cast<unsigned>((V + 255) / 256)), dim3(256), 0, stream,
                               dz, p.ldz, nt, static_cast<int>(V), d_bias, acc);
        if (int rc = wide_check("wide backward launch failed")) return rc;
    }
    return 0;
}

}  // namespace

int wide_fwd_partials(const void* hidden, const void* weight, const float* bias, const int64_t* targets,
                      float* part_m, float* part_s, float* part_z, int n_split, int64_t N, int32_t H,
                      int64_t V, int64_t vocab_start, int32_t dtype, float temperature, hipStream_t stream,
                      float* kept)
{
    WideFwdArgs a;
    a.kept = kept;
    a.ldz = (V + 3) / 4 * 4;
    a.hidden = hidden;
    a.weight = weight;
    a.bias = bias;
    a.targets = targets;
    a.part_m = part_m;
    a.part_s = part_s;
    a.part_z = part_z;
    a.N = static_cast<int>(N);
    a.H = H;
    a.V = static_cast<int>(V);
    a.vocab_start = vocab_start;
    a.row_blocks = static_cast<int>((N + 255) / 256);
    a.vtiles = static_cast<int>((V + 255) / 256);
    a.n_split = n_split < a.vtiles ? n_split : a.vtiles;
    if (a.n_split != n_split) return rlk_fail(RLK_ERR_ARG, "more splits than vocab tiles");
    a.scale2 = kLog2e / temperature;
    a.vec_h = quad_aligned(hidden, H, dtype);
    a.vec_w = quad_aligned(weight, H, dtype);
    if (kept != nullptr)
        return dtype == RLK_DTYPE_F32 ? wide_fwd_launch<RLK_DTYPE_F32, true>(a, stream)
                                      : rlk_fail(RLK_ERR_UNSUPPORTED, "the fp32 kernels keep logits of fp32 inputs only");
    if (dtype == RLK_DTYPE_F32) return wide_fwd_launch<RLK_DTYPE_F32>(a, stream);
    if (dtype == RLK_DTYPE_BF16) return wide_fwd_launch<RLK_DTYPE_BF16>(a, stream);
    return wide_fwd_launch<RLK_DTYPE_F16>(a, stream);
}

size_t wide_bwd_workspace(int64_t N, int32_t H, int64_t V, size_t dz_budget_bytes)
{
    return wide_plan(N, H, V, dz_budget_bytes).total;
}

int wide_bwd(const float* grad_logp, const void* hidden, const void* weight, const float* bias,
             const int64_t* targets, const float* lse, void* d_hidden, float* d_weight, float* d_bias,
             void* workspace, size_t dz_budget_bytes, int64_t N, int32_t H, int64_t V,
             int64_t vocab_start, int32_t dtype, float temperature, int64_t ignore_index,
             int32_t use_ignore, int32_t accumulate, hipStream_t stream)
{
    const WidePlan p = wide_plan(N, H, V, dz_budget_bytes);
    if (dtype == RLK_DTYPE_F32)
        return wide_bwd_launch<RLK_DTYPE_F32>(grad_logp, hidden, weight, bias, targets, lse, d_hidden, d_weight,
                                              d_bias, nullptr, workspace, p, N, H, V, vocab_start, temperature,
                                              ignore_index, use_ignore, accumulate, stream);
    if (dtype == RLK_DTYPE_BF16)
        return wide_bwd_launch<RLK_DTYPE_BF16>(grad_logp, hidden, weight, bias, targets, lse, d_hidden, d_weight,
                                               d_bias, nullptr, workspace, p, N, H, V, vocab_start, temperature,
                                               ignore_index, use_ignore, accumulate, stream);
    return wide_bwd_launch<RLK_DTYPE_F16>(grad_logp, hidden, weight, bias, targets, lse, d_hidden, d_weight,
                                          d_bias, nullptr, workspace, p, N, H, V, vocab_start, temperature,
                                          ignore_index, use_ignore, accumulate, stream);
}

// Size of the kept logits of an fp32 head, 0 where none are kept: more than the bound, or a head so narrow that the
// products cost what the trip through memory does.
size_t wide_kept_bytes(int64_t N, int32_t H, int64_t V)
{
    const size_t bytes = static_cast<size_t>(N) * ((V + 3) / 4 * 4) * 4;
    return bytes > RLK_KEPT_LOGITS_BYTES || H < 128 ? 0 : bytes;
}

size_t wide_bwd_kept_workspace(int64_t N, int32_t H, int64_t V, bool again) { return wide_kept_plan(N, H, V, again).total; }

int wide_bwd_kept(const float* grad_logp, const void* hidden, const void* weight, const float* bias,
                  const int64_t* targets, const float* lse, void* d_hidden, float* d_weight, float* d_bias,
                  float* kept, void* workspace, int64_t N, int32_t H, int64_t V, int64_t vocab_start,
                  float temperature, int64_t ignore_index, int32_t use_ignore, int32_t accumulate, hipStream_t stream)
{
    return wide_bwd_launch<RLK_DTYPE_F32>(grad_logp, hidden, weight, bias, targets, lse, d_hidden, d_weight, d_bias, kept,
                                          workspace, wide_kept_plan(N, H, V, kept == nullptr), N, H, V, vocab_start, temperature,
                                          ignore_index, use_ignore, accumulate, stream);
}

}  // namespace rlk
