// Batched GEMV for gfx950: n_tok tokens share every weight read (prefill, speculative or multi-sequence decode; the
// batched path the reference plans in ROADMAP.md:78-96). Token t's output row is the single-token GEMV's bit for
// bit: the same Q8_0 activation quantizer (gemvq_ref.h:236-245, with a per-token RMS norm folded in as the deferred
// norm of gemvqc16.h:52-59), the same exact block terms floor(sumi * fp16(d_w) * d_x * 2^40) summed exactly and
// rounded to FP32 once (gemvqw_engine.h:352-445), the same epilogs. Per 32-weight block and 16 rows x 16 tokens the
// matrix cores do two products:
//   - one v_mfma_i32_16x16x32_i8 for the block sums. A block's 32 quants may be permuted as long as the weight and the
//     activation operands agree, so lane group g (lanes 16g..16g+15) takes quants 4g..4g+3 and 16+4g..16+4g+3: Q4_0
//     and Q4_1 pack exactly those as the low and high nibbles of quant bytes 4g..4g+3, Q8_0 holds them as bytes
//     4g..4g+3 of its two 16-byte halves, and the activation quantizer stores them in that order. Q4_0 enters as
//     16 * (q - 8), the nibble moved to the top of its byte (three instructions a block instead of nine for q - 8);
//   - one v_mfma_f32_16x16x16_f16 for the scale products d_w * d_x of the block: B holds the tokens' scales of 16
//     blocks as they lie in memory, A the row's scale of this block at the block's place and zeros elsewhere, so every
//     product comes out alone, exact in FP32, already where the block sums' rows and tokens are.
// The vector ALUs then do three FP64 instructions a term: both values converted, and one fused multiply-add into an
// accumulator near 1.5 * 2^52 LSB in the round-toward-minus-infinity mode. There the accumulator's last place is the
// LSB 2^-40, so that one rounding is the term's floor, and the sum of the floors is exact while it stays within 2^51
// LSB (checked per 16 blocks; past it the terms go to int64 one by one). The accumulator's bits less those of
// 1.5 * 2^52 LSB are the integer sum.
// Q6_K (super-blocks of 256 weights on Q8_K activations) has one term per super-block, of the sum of its 16 sub-block
// sums times their int8 scales: the sub-block sums come from the same matrix product with half of each operand zeroed (an
// operand's low and high words belong to different sub-blocks), the scales multiply them in the vector ALUs, and the
// super-block's scale product, 11 by 24 bits, is exact in FP64; the fused multiply-add then floors as above.
// Q4_1 adds the term floor(m_w * s_x * 2^40) with the Q8_1 s_x of each activation block (gemvq_ref.h:194-229), its
// product by one more FP16 matrix product of the same form.
#include "gq_gemv_impl.h"

#include <algorithm>
#include <type_traits>

namespace gq {
namespace {

constexpr int GT = 16;             // rows and tokens per MFMA tile
constexpr int GS = 16;             // blocks per step of a wave
constexpr int GNW = 8;             // waves per workgroup; wave w sums steps w, w + GNW, ..
constexpr int GNT = GNW * WAVE;

typedef int v4i __attribute__((ext_vector_type(4)));
typedef unsigned v2u __attribute__((ext_vector_type(2)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));  // native vectors (promoted to registers, unlike uint4)
typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));

// Activation scratch, in the order the waves of gemm_kernel read it (16 consecutive bytes a lane, 1 KiB an
// instruction): per tile of 16 tokens and step of 16 blocks, the pairs of blocks in turn, lane (r, g) = 16 g + r holding
// token r's 8-byte groups g (quants 4g..4g+3 and 16+4g..16+4g+3) of the pair's two blocks.
__device__ __forceinline__ size_t act_group(int tok, int g, int ns, int b) {
    return ((size_t(tok >> 4) * ns + (b >> 4)) * 8 + (b >> 1 & 7)) * 1024 + size_t(g * 16 + (tok & 15)) * 16 + (b & 1) * 8;
}
// Its fp16 scales (and Q8_1 sums): per tile and step, lane (r, g) holds token r's blocks 4g .. 4g + 3.
__device__ __forceinline__ size_t act_scale(int tok, int ns, int b) {
    return (size_t(tok >> 4) * ns + (b >> 4)) * 256 + size_t((b >> 2 & 3) * 16 + (tok & 15)) * 4 + (b & 3);
}
// And each step's part of the term bound, per tile and step one value a token.
__device__ __forceinline__ size_t act_bound(int tok, int ns, int step) {
    return (size_t(tok >> 4) * ns + step) * 16 + (tok & 15);
}

// ---- activation: token rows -> Q8_0 blocks in operand order ----
// Workgroup t quantizes token t exactly as the single-token prologue: thread i holds the 16-float items i, i + NT,
// ... (the two halves of a block in adjacent lanes), the norm scale is the canonical pairwise tree over the row, and
// v = (x * scale) * w. Beside each step of 16 blocks goes its part of the term bound: the sum over the blocks of
// d_x * 2^40 * (sum of |quants|) / (32 * 127), which times a matrix's wbound bounds the step's terms; infinite where a block's
// Q8_1 sum is (its values together past the largest fp16, its scale finite): in the FP16 product the zeros beside such a sum
// would become NaNs, so that these steps go to step_terms_exact, whatever the format.
__global__ __launch_bounds__(NT) void gemm_quant_kernel(GemmQuantArgs a) {
    __shared__ Lds s;
    const int tok = blockIdx.x, nb = a.cols / 32, ns = nb / GS, n16 = a.cols / 16;
    int8_t * q = a.q;
    if (tok >= a.n_tok) {  // padding tokens: zero quants and scales, whose terms are exactly zero
        for (int i = threadIdx.x; i < 2 * nb; i += NT)  // 4 groups of a pair of blocks
            *reinterpret_cast<uint4 *>(q + act_group(tok, i & 3, ns, i >> 2 << 1)) = make_uint4(0u, 0u, 0u, 0u);
        for (int i = threadIdx.x; i < nb; i += NT) a.d[act_scale(tok, ns, i)] = a.s[act_scale(tok, ns, i)] = 0;
        for (int i = threadIdx.x; i < ns; i += NT) a.bound[act_bound(tok, ns, i)] = 0.0f;
        return;
    }
    const float * x = a.x + size_t(tok) * a.x_stride;
    const float sc = a.norm ? block_norm_scale(x, a.cols, a.eps, a.norm_l2, s) : 1.0f;
    for (int i = threadIdx.x; i < n16; i += NT) {  // n16 is a multiple of 32: whole steps of lanes run every round
        float v[16];
        load16(x + size_t(i) * 16, v);
        if (a.norm_w) {
            float w[16];
            load16(a.norm_w + size_t(i) * 16, w);
#pragma unroll
            for (int j = 0; j < 16; ++j) v[j] = (v[j] * sc) * w[j];
        } else {
#pragma unroll
            for (int j = 0; j < 16; ++j) v[j] = v[j] * sc;
        }
        uint32_t packed[4];
        int sum;
        const float d = quantize_half_core(v, packed, sum);
        // half h of block b: its word g (quants 16h + 4g .. 16h + 4g + 3) is word h of group g
        const int b = i >> 1, h = i & 1;
        uint32_t mag = 0;  // sum of |quants| of the half
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            *reinterpret_cast<uint32_t *>(q + act_group(tok, g, ns, b) + 4 * h) = packed[g];
            mag = __builtin_amdgcn_sad_u8(packed[g] ^ 0x80808080u, 0x80808080u, mag);  // |q + 128 - 128| per byte
        }
        const uint32_t dh = f2h(d), sh = f2h(float(sum) * d);
        if (h == 0) {
            a.d[act_scale(tok, ns, b)] = uint16_t(dh);
            a.s[act_scale(tok, ns, b)] = uint16_t(sh);  // ggml quantize_row_q8_1: fp16(sum * d)
        }
        float bs = h2f(dh) * (1099511627776.0f / 4064.0f) * float(mag);
        if ((sh & 0x7c00u) == 0x7c00u) bs = __builtin_inff();
        bs = pair_sum_lanes<32>(bs);  // the 32 halves of the step's 16 blocks
        if ((i & 31) == 0) a.bound[act_bound(tok, ns, i >> 5)] = bs;
    }
}

// The same for K-quant weights: Q8_K super-blocks (gemvq_ref.h:62-81) by the single-token prologue's quantizer, the quants
// in the same order, the FP32 scales (subnormals as zero, as the block terms take them) per tile and step as two rows of 16
// tokens, and the step's sum of |d_x| * (sum of |quants|) * 2^40.
__device__ __forceinline__ float * act_kscale(uint16_t * d, int tok, int ns, int sb) {
    return reinterpret_cast<float *>(d) + (size_t(tok >> 4) * ns + (sb >> 1)) * 32 + (sb & 1) * 16 + (tok & 15);
}

__global__ __launch_bounds__(NT) void gemm_quant_k_kernel(GemmQuantArgs a) {
    __shared__ Lds s;
    const int tok = blockIdx.x, nb = a.cols / 32, ns = nb / GS, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const bool pad = tok >= a.n_tok;  // padding tokens: zero quants and scales
    if (!pad) {
        const float * x = a.x + size_t(tok) * a.x_stride;
        const float sc = a.norm ? block_norm_scale(x, a.cols, a.eps, a.norm_l2, s) : 1.0f;
        quantize_q8_K(x, a.cols, a.norm != 0, a.norm_w, sc, s.xq, s.bs, s.info);
        __syncthreads();
    }
    const uint32_t * q = reinterpret_cast<const uint32_t *>(s.xq);
    for (int i = threadIdx.x; i < nb * 4; i += NT) {  // block b, group g
        const int b = i >> 2, g = i & 3;
        *reinterpret_cast<v2u *>(a.q + act_group(tok, g, ns, b)) = pad ? v2u{0u, 0u} : v2u{q[b * 8 + g], q[b * 8 + 4 + g]};
    }
    for (int step = wave; step < ns; step += NWAVES) {
        const int sb = step * 2 + (lane >> 5);  // lane l: 16 quants of super-block l / 32 of the step
        uint32_t mag = 0, bits = 0;
        if (!pad) {
            bits = s.info[sb];
            if ((bits & 0x7f800000u) == 0) bits = 0;
#pragma unroll
            for (int k = 0; k < 2; ++k) mag = __builtin_amdgcn_sad_u8(q[step * 128 + 2 * lane + k] ^ 0x80808080u, 0x80808080u, mag);
        }
        const float bs = pair_sum_lanes<64>(fabsf(__uint_as_float(bits)) * float(mag));
        if ((lane & 31) == 0) *act_kscale(a.d, tok, ns, sb) = __uint_as_float(bits);
        if (lane == 0) a.bound[act_bound(tok, ns, step)] = bs * 1099511627776.0f;
    }
}

// ---- weights ----
// One step of one 16-row tile as a wave loads it: of its 16 blocks' quants, instruction c reads blocks 8 (c / 2) + l % 8 of
// rows 8 (c % 2) + l / 8, so that eight neighbouring lanes read a whole 128-byte line (Q8_0 twice), and the scales of blocks
// 4 (l % 4) .. + 3 of row l / 4 as they lie in memory. Weight bytes are read once per launch: the non-temporal hint keeps
// them from displacing the activations in L2.
template <int TYPE>
struct WStep {
    v4u q[4];
    v4u q2[TYPE == T_Q8_0 ? 4 : 1];  // the high halves of Q8_0 blocks
    typename std::conditional<TYPE == T_Q4_1, v4u, v2u>::type s;  // Q4_1: four (d, m) pairs; others: four d
};

// Q6_K: of the row's two super-blocks the 16 low-bit pieces as the quants above, the high-bit piece l % 8 (unit l % 4 of
// super-block l % 8 / 4) of row 8 c + l / 8, 8 of the 32 sub-block scales, and both d.
template <>
struct WStep<T_Q6_K> {
    v4u q[4], h[2];
    v2u s;
    uint32_t d;
};

// Where a lane's part of a step starts: the step's first block in rows l / 8, 8 + l / 8 and l / 4.
// (Block indices: a matrix has fewer than 2^32 blocks of 32, checked at launch.)
struct WAt {
    uint32_t lo, hi, sc;
};

// A SwiGLU pair's tile is 8 rows of g over the same 8 rows of u: rows 8 .. 15 (at.hi and the upper half's at.sc) are u's.
template <int TYPE, bool PAIR>
__device__ __forceinline__ void load_wstep(const WeightView & w, const WeightView & w2, const WAt & at, int lane, WStep<TYPE> & o) {
    const int col = lane & 7;
    const auto piece = [&](const uint8_t * lo, const uint8_t * hi, int c) {
        return __builtin_nontemporal_load(reinterpret_cast<const v4u *>(
            (PAIR && (c & 1) ? hi : lo) + size_t((c & 1 ? at.hi : at.lo) + 8 * (c >> 1) + col) * 16));
    };
#pragma unroll
    for (int c = 0; c < 4; ++c) o.q[c] = piece(w.a, w2.a, c);
    if constexpr (TYPE == T_Q8_0) {
#pragma unroll
        for (int c = 0; c < 4; ++c) o.q2[c] = piece(w.b, w2.b, c);
    }
    if constexpr (TYPE == T_Q6_K) {
#pragma unroll
        for (int c = 0; c < 2; ++c)  // the row's 8 high-bit pieces
            o.h[c] = __builtin_nontemporal_load(reinterpret_cast<const v4u *>(w.b + size_t(c & 1 ? at.hi : at.lo) * 8) + col);
        o.s = __builtin_nontemporal_load(reinterpret_cast<const v2u *>(w.c + size_t(at.sc) * 2) + (lane & 3));
        o.d = *reinterpret_cast<const uint32_t *>(w.d + (at.sc >> 2));
    } else {
        const uint8_t * sb = TYPE == T_Q8_0 ? (PAIR && lane >= 32 ? w2.c : w.c) : (PAIR && lane >= 32 ? w2.b : w.b);
        const size_t at4 = at.sc + 4 * (lane & 3);
        if constexpr (TYPE == T_Q4_1) o.s = __builtin_nontemporal_load(reinterpret_cast<const v4u *>(sb + at4 * 4));
        else o.s = __builtin_nontemporal_load(reinterpret_cast<const v2u *>(sb + at4 * 2));
    }
}

// A wave's step in its part of LDS, which turns the load order into the operand order: the 16-byte quants of (row r,
// block 4c + b) at slot 4r + (b + r / 4) % 4 of KiB c (the 16 rows' words of one block then lie in distinct banks), the
// scales of (row r, blocks 4g .. 4g + 3) at lane (r, g).
template <int TYPE>
struct WLds {
    static constexpr int QH = TYPE == T_Q8_0 ? 2 : 1;
    uint32_t q[QH][4][256];
    uint32_t s[WAVE * (TYPE == T_Q4_1 ? 4 : 2)];
};

// The word slot of the piece that lane l loaded with instruction c (row 8 (c % 2) + l / 8, piece l % 4 of its KiB).
__device__ __forceinline__ int stage_slot(int lane, int c) {
    const int row = 8 * (c & 1) + (lane >> 3);
    return 4 * (4 * row + (((lane & 3) + (row >> 2)) & 3));
}

template <int TYPE>
__device__ __forceinline__ void stage(const WStep<TYPE> & w, int lane, WLds<TYPE> & l) {
    const int row = lane >> 2, part = lane & 3;
#pragma unroll
    for (int c = 0; c < 4; ++c) *reinterpret_cast<v4u *>(&l.q[0][2 * (c >> 1) + (lane >> 2 & 1)][stage_slot(lane, c)]) = w.q[c];
    if constexpr (TYPE == T_Q8_0) {
#pragma unroll
        for (int c = 0; c < 4; ++c)
            *reinterpret_cast<v4u *>(&l.q[WLds<TYPE>::QH - 1][2 * (c >> 1) + (lane >> 2 & 1)][stage_slot(lane, c)]) = w.q2[c];
    }
    if constexpr (TYPE == T_Q4_1) *reinterpret_cast<v4u *>(&l.s[4 * (part * 16 + row)]) = w.s;
    else *reinterpret_cast<v2u *>(&l.s[2 * (part * 16 + row)]) = w.s;
}

// The i8 operand of one block from its quant word(s).
template <int TYPE>
__device__ __forceinline__ long a_operand(uint32_t lo, uint32_t hi) {
    uint32_t w0 = lo, w1 = hi;
    if constexpr (TYPE == T_Q4_1) {
        w0 = lo & 0x0F0F0F0Fu;
        w1 = (lo >> 4) & 0x0F0F0F0Fu;
    }
    if constexpr (TYPE == T_Q4_0) {  // 16 (q - 8) as int8: the nibble at the top of the byte, its sign bit flipped
        w0 = ((lo << 4) & 0xF0F0F0F0u) ^ 0x80808080u;
        w1 = (lo & 0xF0F0F0F0u) ^ 0x80808080u;
    }
    return long((uint64_t(w1) << 32) | w0);
}

// Q6_K: the high-bit pieces as the quants; the sub-block scales as integers, those of unit u of super-block c in row r at
// (4c + u) * 16 + r; d as loaded.
template <>
struct WLds<T_Q6_K> {
    uint32_t q[1][4][256], h[2][256];
    int s[8 * 16][4];
    uint32_t d[16];
};

template <>
__device__ __forceinline__ void stage<T_Q6_K>(const WStep<T_Q6_K> & w, int lane, WLds<T_Q6_K> & l) {
    const int row = lane >> 2, part = lane & 3;
#pragma unroll
    for (int c = 0; c < 4; ++c) *reinterpret_cast<v4u *>(&l.q[0][2 * (c >> 1) + (lane >> 2 & 1)][stage_slot(lane, c)]) = w.q[c];
#pragma unroll
    for (int c = 0; c < 2; ++c) *reinterpret_cast<v4u *>(&l.h[lane >> 2 & 1][stage_slot(lane, c)]) = w.h[c];
#pragma unroll
    for (int k = 0; k < 2; ++k) {  // scales 8 part .. + 7 of the row's 32: units 2 part and 2 part + 1 of its eight
        v4i v;
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = int(w.s[k] << (24 - 8 * i)) >> 24;
        *reinterpret_cast<v4i *>(l.s[(2 * part + k) * 16 + row]) = v;
    }
    if (part == 0) l.d[row] = w.d;
}

// The launch as the kernel reads it: the members of a group (one, of a SwiGLU pair) by index, their 16-row tiles after
// one another.
struct GemmMember {
    WeightView w;
    float * y;
    const float * res;
    int rows, y_stride, res_stride, epi, tile0;
    float wbound;
};
struct GemmLaunch {
    const int8_t * q;
    const uint16_t * d, * s;
    const float * bound;
    int cols, n_tok, n_members, n_tiles;
    WeightView w2;  // u of a SwiGLU pair
    GemmMember m[GEMM_MAX_MORE + 1];
};
// The member of tile b: the last whose first tile is <= b.
__device__ __forceinline__ int member_of(const GemmLaunch & a, int b) {
    int mi = 0;
    for (int i = 1; i < a.n_members; ++i) mi = b >= a.m[i].tile0 ? i : mi;
    return mi;
}

// A lane's activation operands of one step (token tiles tile, tile + 1, ..): group g of token r's 16 blocks, and (lane group g) the scales of the
// token's blocks 4g .. 4g + 3; the step's part of the term bound.
template <int TYPE, int T>
struct XStep {
    v4u q[T][GS / 2];
    v2u d[T];
    v2u s[TYPE == T_Q4_1 ? T : 1];
    float bound;  // the largest over the token tiles
};

template <int T>
struct XStep<T_Q6_K, T> {
    v4u q[T][GS / 2];
    float d[T][2];  // token r's scales of the step's super-blocks
    float bound;
};

template <int TYPE, int T>
__device__ __forceinline__ void load_xstep(const GemmLaunch & a, int ns, int lane, int tile, int step, XStep<TYPE, T> & o) {
    float bd[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const size_t at = size_t(tile + t) * ns + step;
        const v4u * p = reinterpret_cast<const v4u *>(a.q + at * 8192) + lane;
#pragma unroll
        for (int k = 0; k < GS / 2; ++k) o.q[t][k] = p[k * WAVE];
        if constexpr (TYPE == T_Q6_K) {
#pragma unroll
            for (int k = 0; k < 2; ++k) o.d[t][k] = reinterpret_cast<const float *>(a.d)[at * 32 + k * 16 + (lane & 15)];
        } else {
            o.d[t] = reinterpret_cast<const v2u *>(a.d + at * 256)[lane];
        }
        if constexpr (TYPE == T_Q4_1) o.s[t] = reinterpret_cast<const v2u *>(a.s + at * 256)[lane];
        bd[t] = a.bound[at * 16 + (lane & 15)];
    }
    o.bound = 0.0f;
#pragma unroll
    for (int t = 0; t < T; ++t) o.bound = bd[t] <= o.bound || o.bound != o.bound ? o.bound : bd[t];  // a NaN stays
}

// The FP16 operand of one block: the row's scale at the block's place c of the lane group that it is mine of, zeros
// elsewhere.
__device__ __forceinline__ v4h one_scale(const v2u & d, int c, bool mine) {
    const uint32_t v = mine ? (c & 1 ? d[c >> 1] & 0xffff0000u : d[c >> 1] & 0xffffu) : 0u;
    const v2u o = c < 2 ? v2u{v, 0u} : v2u{0u, v};
    return __builtin_bit_cast(v4h, o);
}

// 1.5 * 2^52 LSB: the FP64 accumulator's base. Q4_0 block sums carry a factor 16 and Q6_K sums 4, so the LSB is 2^-36 and
// 2^-38 there.
template <int TYPE>
constexpr double acc_base() { return TYPE == T_Q4_0 ? 98304.0 : TYPE == T_Q6_K ? 24576.0 : 6144.0; }

// The sums S = sum over the 16 sub-blocks of scale * (sum of quant products), times 4, of super-block sb of a Q6_K step:
// S[t][i] of row 4g + i, token r. A quant byte is 4 (q - 32): the nibble in bits 2..5, its high bits in 6 and 7, the sign
// bit flipped. Unit j's low nibbles are its quants A and the high nibbles its quants B (gq_runtime.hip's repack), 16 of each
// per 16-byte piece and sub-block: an operand's low word belongs to the first sub-block, its high word to the second.
template <int T>
__device__ __forceinline__ void superblock_sums(const WLds<T_Q6_K> & l, const XStep<T_Q6_K, T> & x, int sb, int lane, int (*S)[4]) {
    const int r = lane & 15, g = lane >> 4;
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) S[t][i] = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int pc = sb * 8 + 4 * (j >> 1) + 2 * (j & 1);  // the unit's first low-bit piece
        const auto slot = [&](int c) { return 4 * (4 * r + ((c + (r >> 2)) & 3)) + g; };
        const uint32_t q0 = l.q[0][pc >> 2][slot(pc & 3)], q1 = l.q[0][pc >> 2][slot((pc & 3) + 1)], hw = l.h[sb][slot(j)];
        constexpr uint32_t LO = 0x3C3C3C3Cu, HI = 0xC0C0C0C0u, SG = 0x80808080u;
        const uint32_t w[4] = {(((q0 << 2) & LO) | ((hw << 6) & HI)) ^ SG, (((q1 << 2) & LO) | ((hw << 4) & HI)) ^ SG,
                               (((q0 >> 2) & LO) | ((hw << 2) & HI)) ^ SG, (((q1 >> 2) & LO) | (hw & HI)) ^ SG};
        v4i sc[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) sc[i] = *reinterpret_cast<const v4i *>(l.s[(sb * 4 + j) * 16 + 4 * g + i]);
#pragma unroll
        for (int t = 0; t < T; ++t) {
#pragma unroll
            for (int k = 0; k < 4; ++k) {  // sub-blocks: A's first and second 16, B's
                const int blk = sb * 8 + 4 * (j >> 1) + 2 * (k >> 1) + (j & 1);
                const v4u qv = x.q[t][blk >> 1];
                const long bx = (blk & 1) ? long((uint64_t(qv[3]) << 32) | qv[2]) : long((uint64_t(qv[1]) << 32) | qv[0]);
                const v4i zi = {0, 0, 0, 0};
                const long aop = (k & 1) ? long(uint64_t(w[k]) << 32) : long(uint64_t(w[k]));
                const v4i p = __builtin_amdgcn_mfma_i32_16x16x32_i8(aop, bx, zi, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; ++i) S[t][i] += __mul24(sc[i][k], p[i]);
            }
        }
    }
}

// One step into the accumulators acc[t][i] (row 4g + i, token r of token tile t).
template <int TYPE, int T>
__device__ __forceinline__ void step_terms(const WLds<TYPE> & l, const XStep<TYPE, T> & x, int lane, double (*acc)[4]) {
    const int r = lane & 15, g = lane >> 4;
    v2u dw, mw;
    if constexpr (TYPE == T_Q4_1) {  // (d, m) words -> the four d and the four m
        const v4u s = *reinterpret_cast<const v4u *>(&l.s[4 * lane]);
        dw = v2u{__builtin_amdgcn_perm(s[1], s[0], 0x05040100u), __builtin_amdgcn_perm(s[3], s[2], 0x05040100u)};
        mw = v2u{__builtin_amdgcn_perm(s[1], s[0], 0x07060302u), __builtin_amdgcn_perm(s[3], s[2], 0x07060302u)};
    } else {
        dw = *reinterpret_cast<const v2u *>(&l.s[2 * lane]);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
#pragma unroll
        for (int gb = 0; gb < 4; ++gb) {
            // block 4c + gb: its scales are lane group c's, at place gb
            const int at = 4 * (4 * r + ((gb + (r >> 2)) & 3)) + g;
            const long aop = a_operand<TYPE>(l.q[0][c][at], TYPE == T_Q8_0 ? l.q[WLds<TYPE>::QH - 1][c][at] : 0u);
            const v4h dw1 = one_scale(dw, gb, g == c), mw1 = one_scale(TYPE == T_Q4_1 ? mw : dw, gb, g == c);
#pragma unroll
            for (int t = 0; t < T; ++t) {
                const v4u qv = x.q[t][2 * c + (gb >> 1)];
                const long bx = (gb & 1) ? long((uint64_t(qv[3]) << 32) | qv[2]) : long((uint64_t(qv[1]) << 32) | qv[0]);
                const v4i zi = {0, 0, 0, 0};
                const v4f zf = {0.0f, 0.0f, 0.0f, 0.0f};
                const v4i sm = __builtin_amdgcn_mfma_i32_16x16x32_i8(aop, bx, zi, 0, 0, 0);
                const v4f sc = __builtin_amdgcn_mfma_f32_16x16x16f16(dw1, __builtin_bit_cast(v4h, x.d[t]), zf, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[t][i] = __builtin_fma(double(sm[i]), double(sc[i]), acc[t][i]);
                if constexpr (TYPE == T_Q4_1) {
                    const v4f ms = __builtin_amdgcn_mfma_f32_16x16x16f16(mw1, __builtin_bit_cast(v4h, x.s[t]), zf, 0, 0, 0);
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[t][i] = acc[t][i] + double(ms[i]);
                }
            }
        }
    }
}

__device__ __forceinline__ void add_total(long long * p, long long v) {
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Q6_K's step: per super-block and output one fused multiply-add, or with `exact` (wave-uniform; as step_terms_exact) the single-token
// kernel's integer term, added to the int64 totals.
template <int T>
__device__ __forceinline__ void step_terms_k(const WLds<T_Q6_K> & l, const XStep<T_Q6_K, T> & x, int lane, bool exact,
                                             double (*acc)[4], long long (*tot)[4][WAVE]) {
    const int g = lane >> 4;
#pragma unroll
    for (int sb = 0; sb < 2; ++sb) {
        int S[T][4];
        superblock_sums<T>(l, x, sb, lane, S);
        if (!exact) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const double dw = h2f(l.d[4 * g + i] >> (16 * sb) & 0xffffu);
#pragma unroll
                for (int t = 0; t < T; ++t) acc[t][i] = __builtin_fma(double(S[t][i]), dw * double(x.d[t][sb]), acc[t][i]);
            }
        } else {
#pragma unroll
            for (int t = 0; t < T; ++t) {
                int m, e;
                float_parts(x.d[t][sb], m, e);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t dw = l.d[4 * g + i] >> (16 * sb) & 0xffffu;
                    int md, ed;
                    half_parts(dw, md, ed);
                    const int v = S[t][i] >> 2;  // exact: a multiple of 4
                    const bool neg = ((dw >> 15) ^ (__float_as_uint(x.d[t][sb]) >> 31)) & 1;
                    add_total(&tot[t][i][lane], fixed_term((long long)(neg ? -v : v) * ((long long)md * (long long)m), ed + e));
                }
            }
        }
    }
}

// One step with every term formed alone and added to the int64 totals: for steps whose terms could pass the
// accumulators' 2^51 LSB (activation outliers in the thousands) or whose scales or Q8_1 sums are not finite. Block by block in a
// rolled loop that reads its activation operands again where they lie, so that it takes no registers from step_terms.
// tot[t][i][lane]: row 4g + i, token r of token tile t.
template <int TYPE, int T>
__device__ __forceinline__ void step_terms_exact(const GemmLaunch & a, const WLds<TYPE> & l, int ns, int lane, int tile, int step,
                                                 long long (*tot)[4][WAVE]) {
    const int r = lane & 15, g = lane >> 4;
    const uint16_t * sc = reinterpret_cast<const uint16_t *>(l.s);
    constexpr int SW = TYPE == T_Q4_1 ? 2 : 1;  // halves per scale
#pragma unroll 1
    for (int j = 0; j < GS; ++j) {
        const int c = j >> 2, gb = j & 3, blk = step * GS + j;
        const int at = 4 * (4 * r + ((gb + (r >> 2)) & 3)) + g;
        const long aop = a_operand<TYPE>(l.q[0][c][at], TYPE == T_Q8_0 ? l.q[WLds<TYPE>::QH - 1][c][at] : 0u);
        float dw[4], mw[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int k = ((c * 16 + 4 * g + i) * 4 + gb) * SW;
            dw[i] = h2f(sc[k]);
            mw[i] = TYPE == T_Q4_1 ? h2f(sc[k + SW - 1]) : 0.0f;
        }
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const int tok = (tile + t) * GT + r;
            const long bx = *reinterpret_cast<const long *>(a.q + act_group(tok, g, ns, blk));
            const v4i zi = {0, 0, 0, 0};
            const v4i sm = __builtin_amdgcn_mfma_i32_16x16x32_i8(aop, bx, zi, 0, 0, 0);
            const float d40 = h2f(a.d[act_scale(tok, ns, blk)]) * 1099511627776.0f;  // * 2^40, exact
            const float s40 = TYPE == T_Q4_1 ? h2f_fixed(a.s[act_scale(tok, ns, blk)]) * 1099511627776.0f : 0.0f;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const double sum = TYPE == T_Q4_0 ? double(sm[i]) * 0.0625 : double(sm[i]);
                long long v = dint_to_i64(floor(sum * double(dw[i] * d40)));
                if constexpr (TYPE == T_Q4_1) v += dint_to_i64(floor(double(mw[i] * s40)));
                add_total(&tot[t][i][lane], v);
            }
        }
    }
}

// A matrix whose bound is not known (a scale that is not finite; the caller's own memory, never scanned): the largest |scale| of the step's
// blocks over the wave, as the host's weight_bound forms it.
template <int TYPE>
__device__ __forceinline__ float step_bound(const WLds<TYPE> & l, int lane) {
    if constexpr (TYPE == T_Q6_K) return __builtin_inff();
    else {
    uint32_t dm = 0, mm = 0;
    constexpr int N = TYPE == T_Q4_1 ? 4 : 2;
#pragma unroll
    for (int k = 0; k < N; ++k) {
        const uint32_t v = l.s[N * lane + k];
        dm = max(dm, TYPE == T_Q4_1 ? v & 0x7fffu : max(v & 0x7fffu, v >> 16 & 0x7fffu));
        mm = max(mm, v >> 16 & 0x7fffu);
    }
#pragma unroll
    for (int s = 1; s < WAVE; s <<= 1) {
        dm = max(dm, uint32_t(__shfl_xor(int(dm), s, WAVE)));
        mm = max(mm, uint32_t(__shfl_xor(int(mm), s, WAVE)));
    }
    constexpr float smax = TYPE == T_Q4_0 ? 32.0f * 8 * 127 : TYPE == T_Q4_1 ? 32.0f * 15 * 127 : 32.0f * 128 * 127;
    return h2f(dm) * smax + (TYPE == T_Q4_1 ? h2f(mm) * (32.0f * 127) : 0.0f);
    }
}

// FP64 round mode (MODE bits 3:2; 0 nearest even, 2 toward minus infinity). FP32 arithmetic keeps its own. As asm: the
// compiler, which takes the default mode for granted, sets it back ahead of FP64 instructions after a builtin's switch.
#define GQ_ROUND_F64(mode) asm volatile("s_setreg_imm32_b32 hwreg(HW_REG_MODE, 2, 2), " #mode "\n\ts_nop 3" ::: "memory")

// Output rows of a tile: of a SwiGLU pair 8, each from a row of both matrices.
template <bool PAIR>
constexpr int tile_rows() { return PAIR ? GT / 2 : GT; }

// The output of row rr of a tile for one token (lane `src` of the totals tt holds the token in lane group 0).
template <bool PAIR>
__device__ __forceinline__ float tile_output(int epi, const long long (*tt)[WAVE], int rr, int src, float res) {
    const float v = fixed_to_float(tt[rr & 3][(rr >> 2) * 16 + src]);
    if (PAIR) return (v / (1.0f + expf_(-v))) * fixed_to_float(tt[rr & 3][((rr >> 2) + 2) * 16 + src]);  // gemvqc_ops.h:88-92
    if (epi == EPI_ADD) return v + res;  // gemvqc16.cpp:282-301
    return epi == EPI_SILU ? silu_(v) : v;
}

// The launch is a stream of weight bytes past activations that stay. The (token group of T tiles, tile of 16 rows) pairs,
// in this order, are dealt to the workgroups in equal contiguous runs (a SwiGLU pair's tile: 8 rows of both matrices), each
// summed in batches of up to 8 tiles whose int64 totals lie in LDS. A batch goes through the columns in chunks of 4096
// (128 blocks): wave w holds the activation operands of the chunk's blocks 16 w .. 16 w + 15 in registers while the
// batch's weights stream past, and adds its part of each tile to the totals (exact in any order). The waves meet at
// barriers only around a batch, so that one wave's staging and waits run beside another's sums. With HOLD chunks of
// operands in registers a launch of up to that many chunks reads its activations once per token group; HOLD = 0 reads a
// chunk's operands once per batch. The weights of the next product, or of the next two where one workgroup per CU leaves
// the registers, are requested before the current one is summed. Every load instruction reads whole 128-byte
// (activation: 1 KiB) runs; the operand order comes from the wave's own part of LDS, without a workgroup barrier.
// Up to 16 tokens the weight bytes bound the launch, past that more and more the vector instructions of the terms (405 a
// wave and product of 16 blocks at one token tile, 662 at two, of which the terms are 192 and 384); past 32 tokens four
// token tiles share every weight operand formed.
// Measured (events, Q4_0, MI355X): gate/up pair 2 x 12288 x 4096 15.4 us at 16 tokens (57 MB: 3.7 TB/s) and 24 at 32, 12352 x
// 4096 group 12.5 and 19, 4096 x 12288 12.5 and 17, 4096 x 4096 6.1 and 8.3. Four waves sharing one staged tile, two rounds of
// 16 blocks in flight and seven vector instructions a term took 17.9 and 29.8 us for the average of these launches (now 11.6
// and 17.0). Loads whose neighbouring lanes lay in different rows (the operand order read straight from memory): 20.5 and
// 30.5; the address unit then works a line per lane. 511 tokens (trace): pair 290 us, group 140 us, a layer's launches 0.66
// ms, where 16 chunks of 32 tokens took 1.1 ms; at 16.4 cycles per 64 terms (the matrix product, two conversions and the
// multiply-add in a loop of their own) the pair's terms alone are 172 us.
template <int T>
constexpr int batch_tiles() { return T == 1 ? 4 : 8; }  // (two workgroups' LDS per CU for one token tile)

// Two workgroups per CU for the variants that 128 registers hold (Q4_0, 16 tokens: the gate/up pair 15.4 us, with one
// workgroup and two products ahead 17.0), else one (Q8_0, where 128 registers spill: a layer's launches 254 us, 322 with two).
template <int TYPE, int T, int HOLD>
constexpr int groups_per_cu() { return T == 1 && HOLD == 1 && (TYPE == T_Q4_0 || TYPE == T_Q4_1) ? 2 : 1; }

template <int TYPE, bool PAIR, int T, int HOLD>
__global__ __launch_bounds__(GNT) __attribute__((amdgpu_waves_per_eu(2 * groups_per_cu<TYPE, T, HOLD>())))
void gemm_kernel(GemmLaunch a, int n_tg) {
    constexpr int AHEAD = T <= 2 && groups_per_cu<TYPE, T, HOLD>() == 1 ? 2 : 1, R = tile_rows<PAIR>(), GTB = batch_tiles<T>();
    __shared__ WLds<TYPE> ws[GNW];
    __shared__ long long tot[GTB][T][4][WAVE];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nb = a.cols / 32, ns = nb / GS;
    WLds<TYPE> & wl = ws[wave];
    const int total = n_tg * a.n_tiles;
    const int begin = int((long long)(blockIdx.x) * total / gridDim.x), end = int((long long)(blockIdx.x + 1) * total / gridDim.x);
    const auto batch = [&](int at) { return min(min(GTB, end - at), a.n_tiles - at % a.n_tiles); };  // tiles of the batch at `at`
    // the products still to request, in the order they are summed: batch, step, tile; the member of the last one requested
    int r_at = begin, r_n = begin < end ? batch(begin) : 0, r_step = wave, r_j = 0, r_lo = 0, r_hi = 0;
    GemmMember rm{};
    WStep<TYPE> wn[AHEAD];
    float wb[AHEAD];  // their members' term bounds
    const auto request = [&](WStep<TYPE> & o, float & bound) {
        if (r_at >= end) return;
        const int t = r_at % a.n_tiles + r_j;
        if (t < r_lo || t >= r_hi) {
            const int mi = member_of(a, t);
            rm = a.m[mi];
            r_lo = rm.tile0;
            r_hi = mi + 1 < a.n_members ? a.m[mi + 1].tile0 : a.n_tiles;
        }
        const int r0 = (t - r_lo) * R, top = rm.rows - 1;
        const uint32_t s0 = r_step * GS;
        const WAt at{uint32_t(min(r0 + (lane >> 3), top)) * nb + s0, uint32_t(min(r0 + (PAIR ? 0 : 8) + (lane >> 3), top)) * nb + s0,
                     uint32_t(min(r0 + (lane >> 2 & (R - 1)), top)) * nb + s0};
        load_wstep<TYPE, PAIR>(rm.w, a.w2, at, lane, o);
        bound = rm.wbound;
        if (++r_j < r_n) return;
        r_j = 0;
        r_step += GNW;
        if (r_step < ns) return;
        r_step = wave;
        r_at += r_n;
        if (r_at < end) r_n = batch(r_at);
    };
    XStep<TYPE, T> x[HOLD ? HOLD : 1];
    int held = -1;  // the token group whose operands x holds (HOLD > 0)
    if (wave < ns) {
        if (HOLD > 0 && begin < end) {
            held = begin / a.n_tiles;
#pragma unroll
            for (int h = 0; h < HOLD; ++h)
                if (wave + GNW * h < ns) load_xstep<TYPE, T>(a, ns, lane, held * T, wave + GNW * h, x[h]);
        }
#pragma unroll
        for (int k = 0; k < AHEAD; ++k) request(wn[k], wb[k]);
    }
    for (int at = begin; at < end;) {
        const int tg = at / a.n_tiles, t0 = at % a.n_tiles, n = batch(at);
        for (int i = tid; i < n * T * 4 * WAVE; i += GNT) (&tot[0][0][0][0])[i] = 0;
        __syncthreads();
        GQ_ROUND_F64(2);
        const auto chunk = [&](int step, XStep<TYPE, T> & xs) {
            for (int j = 0; j < n; ++j) {
                stage<TYPE>(wn[0], lane, wl);
                const float wbd = wb[0];
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                if constexpr (AHEAD == 2) {
                    wn[0] = wn[1];
                    wb[0] = wb[1];
                }
                request(wn[AHEAD - 1], wb[AHEAD - 1]);
                const float bound = (wbd < __builtin_inff() ? wbd : step_bound<TYPE>(wl, lane)) * xs.bound;
                const bool exact = __builtin_amdgcn_ballot_w64(!(bound < 1125899906842624.0f)) != 0;  // 2^50 LSB
                if (TYPE != T_Q6_K && exact) {
                    if constexpr (TYPE != T_Q6_K) step_terms_exact<TYPE, T>(a, wl, ns, lane, tg * T, step, tot[j]);
                } else {
                    double acc[T][4];
#pragma unroll
                    for (int k = 0; k < T; ++k)
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            acc[k][i] = acc_base<TYPE>();
                            asm volatile("" : "+v"(acc[k][i]));  // the sums stay between the mode switches
                        }
                    if constexpr (TYPE == T_Q6_K) step_terms_k<T>(wl, xs, lane, exact, acc, tot[j]);
                    else step_terms<TYPE, T>(wl, xs, lane, acc);
#pragma unroll
                    for (int k = 0; k < T; ++k)
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            asm volatile("" : "+v"(acc[k][i]));
                            add_total(&tot[j][k][i][lane], __builtin_bit_cast(long long, acc[k][i]) -
                                                               __builtin_bit_cast(long long, acc_base<TYPE>()));
                        }
                }
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
            }
        };
        if constexpr (HOLD > 0) {
            if (held != tg && wave < ns) {
                held = tg;
#pragma unroll
                for (int h = 0; h < HOLD; ++h)
                    if (wave + GNW * h < ns) load_xstep<TYPE, T>(a, ns, lane, tg * T, wave + GNW * h, x[h]);
            }
#pragma unroll
            for (int h = 0; h < HOLD; ++h)
                if (wave + GNW * h < ns) chunk(wave + GNW * h, x[h]);
        } else {
            for (int step = wave; step < ns; step += GNW) {
                load_xstep<TYPE, T>(a, ns, lane, tg * T, step, x[0]);
                chunk(step, x[0]);
            }
        }
        GQ_ROUND_F64(0);
        __syncthreads();
        // element e: row e % R of tile e / (R tokens), its token in between (consecutive rows are stored together); four
        // elements a thread at a time, their residuals requested together
        for (int e0 = tid; e0 < n * R * T * GT; e0 += 4 * GNT) {
            float res[4];
            float * y[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int e = e0 + k * GNT, rr = e % R, tk = e / R % (T * GT), b = t0 + e / (R * T * GT), tok = tg * T * GT + tk;
                const GemmMember & t = a.m[member_of(a, min(b, a.n_tiles - 1))];
                const int row = (b - t.tile0) * R + rr;
                const bool on = e < n * R * T * GT && tok < a.n_tok && row < t.rows;
                y[k] = on ? t.y + size_t(tok) * t.y_stride + row : nullptr;
                res[k] = on && !PAIR && t.epi == EPI_ADD ? t.res[size_t(tok) * t.res_stride + row] : 0.0f;
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (!y[k]) continue;
                const int e = e0 + k * GNT, rr = e % R, tk = e / R % (T * GT), j = e / (R * T * GT);
                const int epi = PAIR ? int(EPI_SWIGLU) : a.m[member_of(a, t0 + j)].epi;
                *y[k] = tile_output<PAIR>(epi, tot[j][tk >> 4], rr, tk & 15, res[k]);
            }
        }
        __syncthreads();
        at += n;
    }
}

template <int TYPE, bool PAIR, int T, int HOLD>
void launch_one(const GemmLaunch & a, hipStream_t st) {
    // as many workgroups as the 256 CUs hold at once
    const int n_tg = (a.n_tok + T * GT - 1) / (T * GT);
    const int grid = std::min(n_tg * a.n_tiles, 256 * groups_per_cu<TYPE, T, HOLD>());
    GQ_LAUNCH((gemm_kernel<TYPE, PAIR, T, HOLD>), dim3(grid), dim3(GNT), 0, st, a, n_tg);
}

template <int TYPE, bool PAIR>
hipError_t launch_tiles(const GemmArgs & g, hipStream_t st) {
    GemmLaunch a{g.q, g.d, g.s, g.bound, g.cols, g.n_tok, 1 + g.n_more, 0, g.w2, {}};
    for (int i = 0; i <= g.n_more; ++i) {  // members follow each other, every one at least a tile
        const GemmMore f{g.w, g.y, g.res, g.rows, g.y_stride, g.res_stride, g.epi};
        const GemmMore & o = i ? g.more[i - 1] : f;
        if (o.rows < 1 || (uint64_t(o.rows) * unsigned(g.cols / 32)) >> 32) return hipErrorInvalidValue;
        a.m[i] = GemmMember{o.w, o.y, o.res, o.rows, o.y_stride, o.res_stride, o.epi, a.n_tiles, g.wbound[i]};
        a.n_tiles += (o.rows + tile_rows<PAIR>() - 1) / tile_rows<PAIR>();
    }
    const int chunks = (a.cols / (32 * GS) + GNW - 1) / GNW;
    if (a.n_tok <= GT) {
        if (chunks == 1) launch_one<TYPE, PAIR, 1, 1>(a, st);
        else if (chunks <= 3) launch_one<TYPE, PAIR, 1, 3>(a, st);
        else launch_one<TYPE, PAIR, 1, 0>(a, st);
    } else if (a.n_tok <= 2 * GT) {
        if (chunks == 1) launch_one<TYPE, PAIR, 2, 1>(a, st);
        else launch_one<TYPE, PAIR, 2, 0>(a, st);
    } else if constexpr (TYPE == T_Q6_K) {
        return hipErrorInvalidValue;
    } else {
        if (chunks == 1) launch_one<TYPE, PAIR, 4, 1>(a, st);
        else launch_one<TYPE, PAIR, 4, 0>(a, st);
    }
    return hipGetLastError();
}

template <int TYPE>
hipError_t launch_type(const GemmArgs & a, hipStream_t st) {
    return a.epi == EPI_SWIGLU ? launch_tiles<TYPE, true>(a, st) : launch_tiles<TYPE, false>(a, st);
}

}  // namespace

hipError_t launch_gemm_quant(const GemmQuantArgs & a, hipStream_t s) {
    if (a.n_tok < 1 || a.n_pad != gemm_pad(a.n_tok) || a.n_tok > GEMM_WIDE_TOK || a.cols % 512 ||
        a.cols > GEMV_MAXK || a.x_stride < a.cols || a.x_stride % 16)
        return hipErrorInvalidValue;
    if (a.kq) GQ_LAUNCH(gemm_quant_k_kernel, dim3(a.n_pad), dim3(NT), 0, s, a);
    else GQ_LAUNCH(gemm_quant_kernel, dim3(a.n_pad), dim3(NT), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_gemm(const GemmArgs & a, int type, hipStream_t s) {
    // shapes the kernels assume: whole steps of GS blocks
    if (a.rows < 1 || a.n_tok < 1 || a.n_tok > GEMM_WIDE_TOK || a.cols % 512 || a.cols > GEMV_MAXK ||
        a.y_stride < a.rows || (a.epi == EPI_ADD && a.res_stride < a.rows) || a.n_more < 0 || a.n_more > GEMM_MAX_MORE ||
        (a.n_more && a.epi == EPI_SWIGLU))
        return hipErrorInvalidValue;
    for (int i = 0; i < a.n_more; ++i) {
        const GemmMore & o = a.more[i];
        if (o.epi == EPI_SWIGLU || o.y_stride < o.rows || (o.epi == EPI_ADD && o.res_stride < o.rows)) return hipErrorInvalidValue;
    }
    switch (type) {
    case T_Q4_0: return launch_type<T_Q4_0>(a, s);
    case T_Q4_1: return launch_type<T_Q4_1>(a, s);
    case T_Q8_0: return launch_type<T_Q8_0>(a, s);
    case T_Q6_K: return a.epi == EPI_SWIGLU ? hipErrorInvalidValue : launch_tiles<T_Q6_K, false>(a, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace gq
