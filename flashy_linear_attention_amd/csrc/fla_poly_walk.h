// Chunk-wise evaluation of the polynomial score map, O = tril(f(Xq Xk^T)) V with f(u) = c0 + c1 u + c2 u^2, for rows of
// at most 16 columns over values of at most 64 (two halves of 128: PolyWalkParams::vhalf; of 32 columns in three parts: part): the quadratic kernels' work grows with N^2, this one's with N.
//
// f(x . y) is the product of feature rows phi_w(x) . phi(y) of F = 153 entries (the order of PolyFeatures below): the
// quadratic terms x_a x_b, every pair of columns once (a pair of two counts twice), the columns themselves and a one.  With the running sums of phi(k_j) [v_j, 1]^T over the rows before a chunk
// (T), and of phi(q_i) [g_i, dn_i]^T over the rows after it (U),
//
//   O_i   = f-scores of the chunk . V + phi_w(q_i) T                      n_i the same with the column of ones
//   dV_j  = f-scores^T of the chunk . g + phi_w(k_j) U
//   dq_i  = ((M f'(u)) of the chunk) k   + the gradient of phi_w(q) (T [g_i, dn_i]) at q_i        M_ij = g_i . v_j + dn_i
//   dk_j  = ((M f'(u))^T of the chunk) q + the gradient of phi_w(k) (U [v_j, 1]) at k_j
//
// (g = dO / n, dn_i = -(dO_i . O_i) / n_i formed here from dO, O and n; without the normaliser g = dO and no dn).
// Nothing of width F goes to memory but the states at the ends of a walk's segments, and no feature row to LDS: MFMA
// operands of features are formed in registers, along the row from a row of the x tile (phi_w) and down the rows
// from two rows of its transposed copy (the state's update).  Feature values stay what fp32 gives, as two bf16 numbers
// each (poly_split8), and what is rounded to bf16 is what the quadratic evaluation rounds -- the scores of the chunk -- and
// the running sums once per chunk: errors against fp64 0.87 to 1.01 times the quadratic kernels', the normaliser's 1e-7.
//
// What bounds it: the matrix instructions and the VALU work that forms features together (an update's fragment of eight
// features costs 32 VALU instructions and serves ten MFMAs of 16 x 16 x 32, one along the row 32 and four of 32 x 32 x 16): the VALU
// issues two thirds of the walks' time, the matrix unit is busy a quarter; HBM is far away
// (40 KiB per 128-row chunk).  Hence eight waves, two per SIMD, so that one wave's VALU work runs under the other's MFMAs: wave w owns
// rows 32 (w % 4) .. of the chunk, and of their work one half: half of the features and of the score blocks (forward
// and dq), the rows after the chunk in dV against dk and the chunk's own rows in dV; the two waves of a row
// block exchange one half of the sums through LDS.  (Halves of the output columns instead formed every feature row and
// every score twice.)  Of a state a wave owns one or two of the ten blocks of 16 features, over all value columns, so that every
// feature is formed once.  A workgroup has a CU to itself; the next chunk's rows are fetched into registers a chunk ahead.  The split
// into segments and the forms of their entry states are the walk kernels' (fla_chunk_walk.h).  Backward is a walk in
// forward direction for dq, from the entry states forward formed, and one in reverse for dk and dv, so that nothing of a
// row reaches the dq of the chunks before it.
// Measured, B 4 H 16 N 4096, 16 over 64 columns, normalised, forward + backward: 605 us quadratic, 200 us this way (kernels
// under the profiler 20 totals, 52 forward, 71 dq with the reverse walk's totals, 77 dk and dv).  With the pairs taken by blocks of eight columns -- 209
// features in seven blocks of 32 -- and a barrier more per chunk 239 us.  With T for dq going backwards, by subtraction, in the reverse walk
// 228 us, but a late row that is infinite, NaN or huge spoiled dq before it; with feature rows rounded to one bf16 number on
// both sides as well, from tiles of them in LDS, 200 us, and errors up to 1.28 times the quadratic kernels'.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>

#include "fla_chunk_walk.h"

namespace fla {

struct PolyWalkParams {
    const void *q, *k, *v, *go, *o;  // rows of width r (q, k) and dv (v, go: dO, o: forward's result, read by backward)
    void *out, *dq, *dk, *dv;        // forward: out; backward: dq, dk, dv
    int64_t qs_b, qs_h, qs_n, ks_b, ks_h, ks_n, vs_b, vs_h, vs_n, gs_b, gs_h, gs_n, os_b, os_h, os_n;
    int64_t us_b, us_h, us_n;  // out
    int64_t dqs_b, dqs_h, dqs_n, dks_b, dks_h, dks_n, dvs_b, dvs_h, dvs_n;
    int32_t H, N, BH, r, wv, n_chunks, seg_chunks, n_seg;
    float c0, c1, c2, eps;
    int32_t wide_out;  // dq, dk, dv are floats (and receive the bf16-rounded values)
    float *denom;  // fp32 [BH][N], or null: not normalised.  Forward writes it, backward reads it
    // states [BH][n_seg][PolyFeatures::kState] in fp32
    float *totals;       // totals kernel: receives the segments' sums; walks: those (sum_entries) or the entry states, of
                         // T (forward) / U (backward); null with a single segment
    int32_t sum_entries;
    float *entries;      // T before every segment but the first: written by forward (null: nowhere), read by dq's walk
    // dq's walk (sum_entries, three segments or more: a kernel of its own) adds up its segment's total of U beside dq and writes it to
    // totals for the walk behind -- g and dn are in LDS already.  Forward + backward, a totals kernel in front -> this:
    // B 4 H 16 N 4096 211 -> 200 us; B H 16, N 4096 83.7 -> 77.1, N 16384 219 -> 210; B H 80, N 4096 268 -> 258; 8 over 32 columns, B H 24,
    // N 4096 112.9 -> 107.4
    int32_t u_totals;
    // 1: v of 65 to 128 columns.  BH counts halves of its columns, a (b, h)'s two next to each other, each a head of its own with states of
    // its own: O, dV and the sums are column by column, dq and dk (and dn, a sum over columns) are the halves' added up.  The halves write
    // theirs in fp32 to dq_part / dk_part [BH][N][16] (32 over 16 columns), poly_add_halves_kernel adds and rounds once.  So are the scores'
    // gradients below them, which a half keeps as two bf16 numbers (rounded to one, as the quadratic kernels round the whole, dq and dk were 0.97 to 1.07 of those
    // kernels' errors with few rows, single heads up to 1.2; this way 0.70 to 0.72 up to 128 rows, 0.80 to 0.99 beyond, for 2 to 4 % of a pair's time).  Forward +
    // backward, 16 over 128 columns, normalised, quadratic -> this: B H 16, N 4096 415 -> 126 us, B H 2, N 16384 1546 -> 100, B H 64, N 4096
    // 1014 -> 417 (a v of 64 columns there: 192; both halves form every feature).
    int32_t vhalf;
    float *dq_part, *dk_part;
    // Rows of 17 to 32 columns, as two halves a and b: the features are those of a, those of b and the 256 products of a column of each, and a walk is
    // three launches, one for each part (PolyPart), with states of its own.  What a part adds up goes on in fp32 from launch to launch: of O or
    // dV in acc [BH][N][64], of n in acc_n [BH][N], of dq and dk in acc_q, acc_k [BH][N][32]; the last part, which has the chunk's own scores
    // as well, rounds.  Forward + backward, normalised, quadratic -> this: 32 / 64, B H 2, N 16384 1062 -> 258 us, B H 16, N 16384 2154 -> 747, B H
    // 64, N 8192 2212 -> 1384 (N 4096 634 -> 735: quadratic).  (One launch with all 576 features would need 144 KiB of a CU's registers for a state and 72 KiB of LDS for its copy.)
    int32_t part;
    float *acc, *acc_n, *acc_q, *acc_k;
    int32_t place;  // which workgroup takes which segment (xcd_place) and xcd_item's factor for n_seg, filled by the launcher
    uint32_t n_seg_inv;
};

enum PolyPart {
    kPolyWhole = 0,   // rows of at most 16 columns
    kPolyFirst = 1,   // a's features and the scores over all columns; adds what the others left and stores the results
    kPolySecond = 2,  // b's (without the one): adds to the sums
    kPolyCross = 3,   // a_i b_j: starts the sums
    kPolyHalves = 4,  // as kPolyWhole, over a v of two halves (vhalf; the parts look it up): a variant, as the test cost the others 1 %
};

// Feature order: groups of eight.  Groups 0 .. 15: x_a x_b with a = 8h + j and b = (a + d) % 16 for d = 0 .. 7, h = 0, 1 (group
// 2d + h, feature j of it); group 16: d = 8, a = 0 .. 7; groups 17, 18: the row itself; group 19: a one and zeros.  Going round
// the columns by differences d every pair is there once (17 groups where pairs by blocks of eight columns took 24), and which
// column a feature's factors are is the same for all features of a lane but for a rotation of the row by 8h.
struct PolyFeatures {
    static constexpr int kGroups = 20, kBlocks = 5, kF = 160;  // blocks of 32 features
    static constexpr int kSteps = kGroups / 2;                 // 16-wide k steps of a contraction over the features
    static constexpr int kHalves = kF / 16;                    // blocks of 16 features: the units in which waves own a state
    static constexpr int kV = 64;                              // value columns of a state
    static constexpr int kState = kF * kV + kF;                // [feature][value column], then the column of ones / dn
    static constexpr int kStateRoom = 224 * 65;                // floats per segment of a state buffer: a state of 224 features,
                                                               // by which the size query still answers; the rest is not touched
    // products of a column of a and one of b: group 2d + h (32 of them), feature j of it: a_{8h + j} b_{(8h + j + d) % 16}
    static constexpr int kCross = 256;
};

struct PolyLds {  // byte offsets
    // XTR: an x tile transposed, in fp32 (rows of 528 bytes: the sixteen columns, a one per row of the sequence, zeros): the state's update
    // multiplies two of its rows, and as 16-bit rows the unpacking was a third of its VALU instructions.  16-bit rows -> this, same
    // bits: B H 64, N 4096 203.6 -> 200.6 us forward + backward, 67.0 -> 65.2 forward (totals 22.1 -> 20.4, walk 53.1 -> 51.9); B H 80
    // 256.2 -> 253.6; B H 300, N 1024 291.8 -> 287.5.
    // XTB: the sixteen columns as they are, operands of the chunk's own scores (poly_col_frag)
    static constexpr int C = 128, XT = C * 32, VT = C * 128, ST = 2 * 64 * 256, XR = 528, XTR = 18 * XR, XTB = 16 * 272, EX = 8 * 4096;
    static constexpr int Z = PolyFeatures::kF * 4, DN = C * 4;
    // totals: two sets of the x tile transposed, the v tile, dn
    static constexpr int tX = 0, tV = tX + XTR, tDn = tV + VT, tSet = tDn + DN, tTotal = 2 * tSet;
    // forward
    static constexpr int fQ = 0, fK = fQ + XT, fKt = fK + XT, fV = fKt + XTR, fS = fV + VT, fEx = fS + ST, fZ = fEx + EX,
                         fSum = fZ + Z, fTotal = fSum + 2 * C * 4;
    // (rows of two halves: b's tiles, and z of 256 features)
    static constexpr int ZX = PolyFeatures::kCross * 4;
    static constexpr int tX2 = 2 * tSet, tTotalTwo = tX2 + 2 * XTR;
    static constexpr int fQ2 = fTotal, fK2 = fQ2 + XT, fKt2 = fK2 + XT, fZ2 = fKt2 + XTR, fTotalTwo = fZ2 + ZX;
    // dq (the exchange: sixteen floats a row)
    static constexpr int qQ = 0, qK = qQ + XT, qKt = qK + XT, qKb = qKt + XTR, qV = qKb + XTB, qG = qV + VT, qS = qG + VT, qEx = qS + ST,
                         qZ = qEx + C * 64, qDn = qZ + Z, qDx = qDn + DN, qTotal = qDx + DN, qQt = qTotal, qTotalSums = qQt + XTR;
    static constexpr int qQ2 = qTotal, qK2 = qQ2 + XT, qKt2 = qK2 + XT, qKb2 = qKt2 + XTR, qZ2 = qKb2 + XTB, qEx2 = qZ2 + ZX,
                         qTotalTwo = qEx2 + C * 128;
    // dk, dv
    static constexpr int kQ = 0, kQt = kQ + XT, kQb = kQt + XTR, kK = kQb + XTB, kV = kK + XT, kG = kV + VT, kU = kG + VT, kY = kU + ST,
                         kDn = kY + Z, kDx = kDn + DN, kEx = kDx + DN, kTotal = kEx + EX;
    static constexpr int kQ2 = kTotal, kK2 = kQ2 + XT, kQt2 = kK2 + XT, kQb2 = kQt2 + XTR, kY2 = kQb2 + XTB, kTotalTwo = kY2 + ZX;
    static_assert(XTR % 16 == 0 && tTotal >= 8 * 5 * 1024 && fTotal <= 160 * 1024 && qTotalSums <= 160 * 1024 && kTotal <= 160 * 1024 && qTotalTwo <= 160 * 1024 &&
                  kTotalTwo <= 160 * 1024, "a CU's LDS");
};

// (a select of two values: written between two elements of an array it would become one load with a computed index, and
// the array would go to scratch memory)
__device__ __forceinline__ float poly_pick(int g, float one, float zero) { return g ? one : zero; }

// rounded pairs: eight floats to an operand fragment
template <typename T>
__device__ __forceinline__ typename Mma<T>::V8 poly_round8(const float (&f)[8]) {
    typename Mma<T>::V8 r;
#pragma unroll
    for (int j = 0; j < 8; ++j) r[j] = static_cast<T>(f[j]);
    return r;
}

// the sixteen columns of one row of an x tile, in fp32
template <typename T>
__device__ __forceinline__ void poly_row(const unsigned char *xt, int row, float (&x)[16]) {
    using V8 = typename Mma<T>::V8;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const V8 e = __builtin_bit_cast(V8, *reinterpret_cast<const u32x4 *>(xt + row * 32 + h * 16));
#pragma unroll
        for (int j = 0; j < 8; ++j) x[8 * h + j] = static_cast<float>(e[j]);
    }
}

// this lane's eight columns of a row of an x tile: an MFMA operand with k along the row
template <typename T>
__device__ __forceinline__ typename Mma<T>::V8 poly_row_frag(const unsigned char *xt, int row, int g) {
    return __builtin_bit_cast(typename Mma<T>::V8, *reinterpret_cast<const u32x4 *>(xt + row * 32 + g * 16));
}

// column r of an x tile from its transposed copy, rows R0 + {4g .., 8 + 4g ..}: the k order of a rounded score
template <typename T>
__device__ __forceinline__ typename Mma<T>::V8 poly_col_frag(const unsigned char *xtb, int r, int R0, int g) {
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    const u32x2 lo = *reinterpret_cast<const u32x2 *>(xtb + r * 272 + (R0 + 4 * g) * 2);
    const u32x2 hi = *reinterpret_cast<const u32x2 *>(xtb + r * 272 + (R0 + 8 + 4 * g) * 2);
    return __builtin_bit_cast(typename Mma<T>::V8, u32x4{lo[0], lo[1], hi[0], hi[1]});
}

// ---- operand fragments of the walk kernels' tile layouts (walk_row_frag, walk_col_frag, walk_col_frag_perm), with their
// addresses split into what depends on the lane, computed once per chunk, an XOR that picks a chunk of a row or a column
// block, and a constant offset -- the swizzle of a row depends on the row modulo 16 only.  (As one expression per
// fragment the addresses took a third of the kernels' VALU instructions.)
struct PolyPair {
    uint32_t lo, hi;
};
// rows 8g .. 8g + 7, plain column mapping, column block 0 (block cb: XOR cb << 6)
template <int RB>
__device__ __forceinline__ PolyPair poly_col_base(int lane) {
    const int lam = lane & 15, g = lane >> 5, beta = (lane >> 4) & 1;
    const int row = 8 * g + (lam >> 2), ch = 2 * beta + ((lam & 3) >> 1), sub = 8 * (lam & 1);
    return {(uint32_t)(row * RB + ((ch ^ walk_swizzle<RB / 16>(row)) << 4) + sub),
            (uint32_t)((row + 4) * RB + ((ch ^ walk_swizzle<RB / 16>(row + 4)) << 4) + sub)};
}
// permuted column mapping, column block 0 (block cb: XOR cb << 6); CONS: rows 8g .. 8g + 7, else {4g .., 8 + 4g ..}
template <int RB, bool CONS>
__device__ __forceinline__ PolyPair poly_perm_base(int lane) {
    const int lam = lane & 15, g = lane >> 5, beta = (lane >> 4) & 1, zc = lam & 3;
    const int lo = (CONS ? 8 : 4) * g + (lam >> 2), hi = lo + (CONS ? 4 : 8), ch = 2 * (zc & 1) + beta, byte = 8 * (zc >> 1);
    return {(uint32_t)(lo * RB + ((ch ^ walk_swizzle<RB / 16>(lo)) << 4) + byte),
            (uint32_t)(hi * RB + ((ch ^ walk_swizzle<RB / 16>(hi)) << 4) + byte)};
}
// chunk g of row `row` (k chunk kc: XOR kc << 5)
template <int RB>
__device__ __forceinline__ uint32_t poly_row_base(int row, int g) {
    return (uint32_t)(row * RB + ((g ^ walk_swizzle<RB / 16>(row)) << 4));
}
template <typename T>
__device__ __forceinline__ typename Mma<T>::V8 poly_tr(const unsigned char *tile, PolyPair at, uint32_t flip = 0) {
    const s16x4 lo = walk_tr_read(tile + (at.lo ^ flip)), hi = walk_tr_read(tile + (at.hi ^ flip));
    return __builtin_bit_cast(typename Mma<T>::V8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}
template <typename T>
__device__ __forceinline__ typename Mma<T>::V8 poly_rd(const unsigned char *tile, uint32_t at) {
    return __builtin_bit_cast(typename Mma<T>::V8, *reinterpret_cast<const u32x4 *>(tile + at));
}

// The mask of a 32 x 32 block on the diagonal for a lane's score i (Y row 8 (i / 4) + 4g + i % 4 against X row l32) as
// bits to AND with
template <bool UPPER>
__device__ __forceinline__ uint32_t poly_mask(int i, int l32, int g) {
    const int jl = 8 * (i / 4) + 4 * g + (i % 4);
    return (UPPER ? jl >= l32 : l32 >= jl) ? ~0u : 0u;
}
// sixteen values rounded to two fragments and masked as pairs (all: ~0 off the diagonal)
template <typename T, bool UPPER>
__device__ __forceinline__ void poly_round_masked(const float (&d)[16], uint32_t all, int l32, int g, typename Mma<T>::V8 (&out)[2]) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        float e[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) e[j] = d[8 * t + j];
        u32x4 w = __builtin_bit_cast(u32x4, poly_round8<T>(e));
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint32_t m = (poly_mask<UPPER>(8 * t + 2 * k, l32, g) & 0xffffu) | (poly_mask<UPPER>(8 * t + 2 * k + 1, l32, g) & 0xffff0000u);
            w[k] &= m | all;
        }
        out[t] = __builtin_bit_cast(typename Mma<T>::V8, w);
    }
}

// ... what that left of the values (the masked ones whole: to be masked again)
template <typename T>
__device__ __forceinline__ void poly_left_over(float (&d)[16], const typename Mma<T>::V8 (&rounded)[2]) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int j = 0; j < 8; ++j) d[8 * t + j] -= static_cast<float>(rounded[t][j]);
}

// Eight fp32 numbers as sums of two bf16 ones each: the upper half of the bits, and what is left, rounded (EXACT: of a
// product of two bf16 numbers, whose sixteen significant bits both halves hold without rounding: the upper half as well)
struct PolyTwo {
    Mma<__bf16>::V8 hi, lo;
};
template <bool EXACT>
__device__ __forceinline__ PolyTwo poly_split8(const float (&f)[8]) {
    PolyTwo t;
    u32x4 hi, lo;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        uint32_t bits[2];
        float rest[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            bits[e] = __builtin_bit_cast(uint32_t, f[2 * k + e]);
            rest[e] = f[2 * k + e] - __builtin_bit_cast(float, bits[e] & 0xffff0000u);
        }
        hi[k] = __builtin_amdgcn_perm(bits[1], bits[0], 0x07060302u);
        if constexpr (EXACT) {
            lo[k] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, rest[1]), __builtin_bit_cast(uint32_t, rest[0]), 0x07060302u);
        } else {
            typedef __bf16 t2 __attribute__((ext_vector_type(2)));
            lo[k] = __builtin_bit_cast(uint32_t, t2{static_cast<__bf16>(rest[0]), static_cast<__bf16>(rest[1])});
        }
    }
    t.hi = __builtin_bit_cast(Mma<__bf16>::V8, hi), t.lo = __builtin_bit_cast(Mma<__bf16>::V8, lo);
    return t;
}

// A row as the features along it take it: turned by 8 g columns, and its first half weighted for the phi_w side
struct PolyTurned {
    float x[16], w[8];  // x[(8g + i) % 16]; 2 c2 times the first eight
};
__device__ __forceinline__ PolyTurned poly_turn(const float (&x)[16], int g, float c2) {
    PolyTurned t;
#pragma unroll
    for (int i = 0; i < 16; ++i) t.x[i] = poly_pick(g, x[(i + 8) & 15], x[i]);
#pragma unroll
    for (int i = 0; i < 8; ++i) t.w[i] = 2.f * c2 * t.x[i];
    return t;
}

// Feature fragment KS (features 16 KS + 8 g ..) of a row, weighted for the phi_w side; `raw` receives it in fp32.
template <int KS>
__device__ __forceinline__ PolyTwo poly_feature_frag(const PolyTurned &t, int g, float c0, float c1, float (&raw)[8]) {
    if constexpr (KS == 0) {  // squares count once
#pragma unroll
        for (int j = 0; j < 8; ++j) raw[j] = 0.5f * t.w[j] * t.x[j];
    } else if constexpr (KS < 8) {
#pragma unroll
        for (int j = 0; j < 8; ++j) raw[j] = t.w[j] * t.x[j + KS];
    } else if constexpr (KS == 8) {  // d = 8; the row's first half
#pragma unroll
        for (int j = 0; j < 8; ++j) raw[j] = (g ? c1 : t.w[j]) * t.x[j + 8];
    } else {  // its second half; the one
#pragma unroll
        for (int j = 0; j < 8; ++j) raw[j] = g ? (j == 0 ? c0 : 0.f) : c1 * t.x[j + 8];
    }
    return poly_split8<false>(raw);
}

// ... of the products of the two halves: a's turned first half, weighted, b turned
template <int KS>
__device__ __forceinline__ PolyTwo poly_cross_frag(const PolyTurned &a, const PolyTurned &b, float (&raw)[8]) {
#pragma unroll
    for (int j = 0; j < 8; ++j) raw[j] = a.w[j] * b.x[(j + KS) & 15];
    return poly_split8<false>(raw);
}

// The two rows of a transposed x tile whose product is feature f, as byte offsets
struct PolyFactors {
    uint32_t a, b;
};
__device__ __forceinline__ PolyFactors poly_factors(int f) {
    const int group = f >> 3, j = f & 7;
    int a, b;
    if (group < 17) {
        a = 8 * (group & 1) + j, b = (a + (group >> 1)) & 15;
    } else {  // the row itself; a one and zeros
        a = group < 19 ? 8 * (group - 17) + j : 16, b = group < 19 || j == 0 ? 16 : 17;
    }
    return {(uint32_t)(a * PolyLds::XR), (uint32_t)(b * PolyLds::XR)};
}

__device__ __forceinline__ PolyFactors poly_cross_factors(int f) {
    const int group = f >> 3, a = 8 * (group & 1) + (f & 7), b = (a + (group >> 1)) & 15;
    return {(uint32_t)(a * PolyLds::XR), (uint32_t)(b * PolyLds::XR)};
}

// A state's blocks of this wave: up to two blocks of 16 features (`first`, `second`, < 0: none) over the four 16-column blocks of
// the values, and -- NORM -- the column of ones (of dn), the same in every lane column.  Register v of a block: feature
// 4 (lane / 16) + v, value column lane % 16.
template <int F>
struct PolyStateOf {
    static constexpr int kState = F * PolyFeatures::kV + F;
    f32x4 st[2][4], ex[2];
    int own[2];
    __device__ __forceinline__ void clear(int first, int second) {
        own[0] = first, own[1] = second;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            ex[u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int cb = 0; cb < 4; ++cb) st[u][cb] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
    // ten blocks on eight waves, two waves to a SIMD: the waves of the row blocks with the least other work take two
    __device__ __forceinline__ void clear_lower(int wave) { clear(wave, wave < 2 ? 8 + wave : -1); }
    // (a second state beside one of clear_lower: on the other two SIMDs.  Waves 4 and 5, on the first two again: B 5 H 16 N 4096 270 us in
    // place of 264)
    __device__ __forceinline__ void clear_beside_lower(int wave) { clear(wave, wave == 2 || wave == 3 ? 6 + wave : -1); }
    __device__ __forceinline__ void clear_upper(int wave) {
        clear(wave < 4 ? 2 * wave : wave >= 6 ? wave + 2 : -1, wave < 4 ? 2 * wave + 1 : -1);
    }
    // += the state at `s` in memory
    template <bool NORM>
    __device__ __forceinline__ void add(const float *s, int lane) {
        const int l16 = lane & 15, kq = lane >> 4;
#pragma unroll
        for (int u = 0; u < 2; ++u)
            if (own[u] >= 0) {
#pragma unroll
                for (int cb = 0; cb < 4; ++cb)
#pragma unroll
                    for (int v = 0; v < 4; ++v) st[u][cb][v] += s[(16 * own[u] + 4 * kq + v) * PolyFeatures::kV + 16 * cb + l16];
                if (NORM) ex[u] += *reinterpret_cast<const f32x4 *>(s + F * PolyFeatures::kV + 16 * own[u] + 4 * kq);
            }
    }
    // += the states `lo` .. `hi` - 1 at `s` in their order, the loads of three in flight together (one at a time is a memory latency
    // per segment as a walk starts)
    template <bool NORM>
    __device__ __forceinline__ void add_range(const float *s, int lo, int hi, int lane) {
        const int l16 = lane & 15, kq = lane >> 4;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            if (own[u] < 0) continue;
#pragma unroll 1
            for (int f0 = lo; f0 < hi; f0 += 3) {
                float t[3][4][4];
                f32x4 e[3];
#pragma unroll
                for (int g = 0; g < 3; ++g) {
                    // (past the range: the last state once more, not added)
                    const float *sf = s + (int64_t)(f0 + g < hi ? f0 + g : hi - 1) * kState;
#pragma unroll
                    for (int cb = 0; cb < 4; ++cb)
#pragma unroll
                        for (int v = 0; v < 4; ++v) t[g][cb][v] = sf[(16 * own[u] + 4 * kq + v) * PolyFeatures::kV + 16 * cb + l16];
                    if (NORM) e[g] = *reinterpret_cast<const f32x4 *>(sf + F * PolyFeatures::kV + 16 * own[u] + 4 * kq);
                }
                walk_all_requested();
#pragma unroll
                for (int g = 0; g < 3; ++g)
                    if (f0 + g < hi) {
#pragma unroll
                        for (int cb = 0; cb < 4; ++cb)
#pragma unroll
                            for (int v = 0; v < 4; ++v) st[u][cb][v] += t[g][cb][v];
                        if (NORM) ex[u] += e[g];
                    }
            }
        }
    }
    template <bool NORM>
    __device__ __forceinline__ void store(float *s, int lane) const {
        const int l16 = lane & 15, kq = lane >> 4;
#pragma unroll
        for (int u = 0; u < 2; ++u)
            if (own[u] >= 0) {
#pragma unroll
                for (int cb = 0; cb < 4; ++cb)
#pragma unroll
                    for (int v = 0; v < 4; ++v) s[(16 * own[u] + 4 * kq + v) * PolyFeatures::kV + 16 * cb + l16] = st[u][cb][v];
                if (NORM && l16 == 0)
                    *reinterpret_cast<f32x4 *>(s + F * PolyFeatures::kV + 16 * own[u] + 4 * kq) = ex[u];
            }
    }
    // rounded to the storage type as rows of value columns, features 0 .. 127 and 128 .. in two tiles; ex in fp32 to z
    template <typename T, bool NORM>
    __device__ __forceinline__ void to_lds(unsigned char *tile, float *z, int lane) const {
        typedef T t4 __attribute__((ext_vector_type(4)));
        const int l16 = lane & 15, kq = lane >> 4;
#pragma unroll
        for (int u = 0; u < 2; ++u)
            if (own[u] >= 0) {
                unsigned char *t = tile + (own[u] >> 3) * 64 * 256;
                const int ch = 2 * (own[u] & 7) + (kq >> 1);
#pragma unroll
                for (int cb = 0; cb < 4; ++cb) {
                    const int row = 16 * cb + l16;
                    t4 w;
#pragma unroll
                    for (int v = 0; v < 4; ++v) w[v] = static_cast<T>(st[u][cb][v]);
                    *reinterpret_cast<t4 *>(t + row * 256 + ((ch ^ walk_swizzle<16>(row)) << 4) + 8 * (kq & 1)) = w;
                }
                if (NORM && l16 == 0) *reinterpret_cast<f32x4 *>(z + 16 * own[u] + 4 * kq) = ex[u];
            }
    }
    // What a step of 32 rows reads; requested a step ahead of its use, block after block (both blocks in one loop of
    // branches: the forward walk 53.6 us in place of 53.1, dk and dv 75.3 in place of 74.1).
    struct Rows {
        f32x4 a[2], b[2];
        u32x4 e[2];
        Mma<__bf16>::V8 z[4];
    };
    template <bool NORM>
    __device__ __forceinline__ void request(Rows &r, const unsigned char *fa, const unsigned char *fb, const unsigned char *zt, PolyPair za,
                                            const float *extra) const {
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) r.z[cb] = poly_tr<__bf16>(zt, za, cb << 5);
#pragma unroll
        for (int h = 0; h < 2; ++h)
            r.a[h] = *reinterpret_cast<const f32x4 *>(fa + 16 * h), r.b[h] = *reinterpret_cast<const f32x4 *>(fb + 16 * h);
        if constexpr (NORM)
            if (extra) r.e[0] = *reinterpret_cast<const u32x4 *>(extra), r.e[1] = *reinterpret_cast<const u32x4 *>(extra + 4);
    }
    template <bool NORM>
    __device__ __forceinline__ void add_rows(const Rows &r, bool ones, f32x4 (&acc)[4], f32x4 &e) {
        float f[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) f[k] = r.a[k / 4][k % 4] * r.b[k / 4][k % 4];
        const PolyTwo y = poly_split8<true>(f);
        Mma<__bf16>::V8 ef;
        if constexpr (NORM) {
            u32x4 w = {0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};
            if (!ones) {
#pragma unroll
                for (int h = 0; h < 4; ++h)
                    w[h] = __builtin_amdgcn_perm(r.e[h >> 1][2 * (h & 1) + 1], r.e[h >> 1][2 * (h & 1)], 0x07060302u);
            }
            ef = __builtin_bit_cast(Mma<__bf16>::V8, w);
        }
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) acc[cb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(y.hi, r.z[cb], acc[cb], 0, 0, 0);
        if constexpr (NORM) e = __builtin_amdgcn_mfma_f32_16x16x32_bf16(y.hi, ef, e, 0, 0, 0);
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) acc[cb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(y.lo, r.z[cb], acc[cb], 0, 0, 0);
        if constexpr (NORM) e = __builtin_amdgcn_mfma_f32_16x16x32_bf16(y.lo, ef, e, 0, 0, 0);
    }
    // += phi^T [z tile, extra column] over the chunk's 128 rows.  Feature rows are formed here, as products of two
    // rows of the transposed x tile: a lane's eight rows of one feature, exactly, in two bf16 numbers each.
    // extra: the extra column, 128 floats in LDS that bf16 holds exactly (null: ones).  xtr2: the second half's transposed tile (F 256).
    // ONE: of the second block the 32 rows of step `step` alone.
    // (Rounded to one bf16 number, from a tile of feature rows, they and the weighted ones along the rows made the errors of
    // O, dq, dk and dv 1.2 times the quadratic kernels', and those of the normaliser 1e-3 in place of 1e-7.)
    template <bool NORM, bool ONE = false>
    __device__ __forceinline__ void update(const unsigned char *xtr, const unsigned char *zt, const float *extra, int lane, int step = 0,
                                           const unsigned char *xtr2 = nullptr) {
        const int l16 = lane & 15, kq = lane >> 4;
        const int row = 8 * kq + (l16 >> 2), ch = (l16 & 3) >> 1, sub = 8 * (l16 & 1);
        const PolyPair za{(uint32_t)(row * 128 + ((ch ^ walk_swizzle<8>(row)) << 4) + sub),
                          (uint32_t)((row + 4) * 128 + ((ch ^ walk_swizzle<8>(row + 4)) << 4) + sub)};
        const float *ex_at = extra ? extra + 8 * kq : nullptr;
        constexpr int STEPS = PolyLds::C / 32;
        auto block = [&](auto uc, auto steps, int first) {
            constexpr int U = decltype(uc)::value, NS = decltype(steps)::value;
            const PolyFactors at = F == PolyFeatures::kCross ? poly_cross_factors(16 * own[U] + l16) : poly_factors(16 * own[U] + l16);
            const unsigned char *fa = xtr + 32 * kq + at.a + 128 * first;
            const unsigned char *fb = (F == PolyFeatures::kCross ? xtr2 : xtr) + 32 * kq + at.b + 128 * first;
            const unsigned char *z0 = zt + 32 * 128 * first;
            const float *e0 = extra ? ex_at + 32 * first : nullptr;
            Rows r[2];
            request<NORM>(r[0], fa, fb, z0, za, e0);
            static_for<0, NS>([&](auto sc) {
                constexpr int S = decltype(sc)::value;
                if constexpr (S + 1 < NS)
                    request<NORM>(r[(S + 1) & 1], fa + 128 * (S + 1), fb + 128 * (S + 1), z0 + 32 * 128 * (S + 1), za, extra ? e0 + 32 * (S + 1) : nullptr);
                __builtin_amdgcn_sched_barrier(0);
                add_rows<NORM>(r[S & 1], !extra, st[U], ex[U]);
            });
        };
        using C4 = std::integral_constant<int, STEPS>;
        if (own[0] >= 0) block(std::integral_constant<int, 0>{}, C4{}, 0);
        if constexpr (ONE) {
            block(std::integral_constant<int, 1>{}, std::integral_constant<int, 1>{}, step);
        } else {
            if (own[1] >= 0) block(std::integral_constant<int, 1>{}, C4{}, 0);
        }
    }
};
using PolyState = PolyStateOf<PolyFeatures::kF>;

// The lane's number as a value the compiler cannot follow out of the chunk loop: LDS addresses that depend on the lane alone
// would all be computed ahead of it and held in registers (dozens of them, to the point of spilling).
__device__ __forceinline__ int poly_opaque(int lane) {
    asm volatile("" : "+v"(lane));
    return lane;
}

struct PolySlice {
    int bh, seg, c_lo, c_hi;
    bool valid;
};
__device__ __forceinline__ PolySlice poly_slice(const PolyWalkParams &p) {  // (walk_slice's map)
    const XcdItem item = xcd_item(blockIdx.x, p.BH, p.n_seg, p.place, p.n_seg_inv);
    PolySlice s;
    s.bh = item.bh, s.seg = item.part;
    s.c_lo = s.seg * p.seg_chunks;
    s.c_hi = s.c_lo + p.seg_chunks < p.n_chunks ? s.c_lo + p.seg_chunks : p.n_chunks;
    s.valid = s.bh >= 0 && s.c_lo < p.n_chunks;
    return s;
}

// what a workgroup's head is in the tensors: its (b, h), and its columns of v
struct PolyHead {
    int bh, b, h, col0, wv;
};
template <bool HALVES>
__device__ __forceinline__ PolyHead poly_head(const PolyWalkParams &p, int item) {
    PolyHead t;
    t.bh = HALVES ? item >> p.vhalf : item;
    t.b = t.bh / p.H, t.h = t.bh - t.b * p.H;
    t.col0 = HALVES ? 64 * (item & p.vhalf) : 0;
    t.wv = HALVES && p.wv - t.col0 > 64 ? 64 : p.wv - t.col0;
    return t;
}

// what a part of rows of two halves takes: its own columns of x (the second half's beside them: TWO)
template <int PART>
struct PolyPartOf {
    static constexpr bool PARTS = PART >= kPolyFirst && PART <= kPolyCross, HALVES = PART != kPolyWhole;
    static constexpr bool CROSS = PART == kPolyCross, TWO = PART == kPolyFirst || CROSS, SCORES = !PARTS || PART == kPolyFirst;
    // over half of v's columns (vhalf) a score's gradient is a partial sum: it is kept as two bf16 numbers
    static constexpr bool TWO_TERMS = PART == kPolyHalves || PART == kPolyFirst;
    static constexpr bool ADDS = PART == kPolyFirst || PART == kPolySecond;  // to what the parts before it left
    static constexpr int F = CROSS ? PolyFeatures::kCross : PolyFeatures::kF, kOff = PART == kPolySecond ? 16 : 0;
    static constexpr int kRoom = PARTS ? F * 65 : PolyFeatures::kStateRoom;  // floats per segment of a state buffer
    __device__ static __forceinline__ int width(const PolyWalkParams &p) { return !PARTS ? p.r : PART == kPolySecond ? p.r - 16 : 16; }
};
// sixteen sums of a row carried from part to part: requested ahead of their use
__device__ __forceinline__ void poly_get_sums(const float *at, bool any, float (&f)[16]) {
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        f32x4 t = {0.f, 0.f, 0.f, 0.f};
        if (any) t = *reinterpret_cast<const f32x4 *>(at + 4 * a);
#pragma unroll
        for (int j = 0; j < 4; ++j) f[4 * a + j] = t[j];
    }
}

// A chunk's rows on their way to LDS, in registers: an x operand (two of them: threads 0 .. 255 and 256 .. 511 take one
// each), tiles of 64 columns, and -- for dO -- forward's result and n.
template <typename T>
__device__ __forceinline__ u32x4 poly_fetch_x(const T *base, int64_t stride, int row0, int N, int r, int tid) {
    const int row = row0 + (tid & 127), half = (tid >> 7) & 1;
    u32x4 v = {0u, 0u, 0u, 0u};
    if (row < N && 8 * half < r) v = *reinterpret_cast<const u32x4 *>(base + (int64_t)row * stride + 8 * half);
    return v;
}
__device__ __forceinline__ void poly_put_x(unsigned char *xt, u32x4 v, int tid) {
    *reinterpret_cast<u32x4 *>(xt + (tid & 127) * 32 + ((tid >> 7) & 1) * 16) = v;
}
// the transposed copy in fp32, with its rows of ones (zeros past the sequence's last row) and of zeros, by the same threads
template <typename T>
__device__ __forceinline__ void poly_put_xt(unsigned char *xtr, u32x4 v, int row0, int N, int tid) {
    const int row = tid & 127, half = (tid >> 7) & 1;
    const typename Mma<T>::V8 e = __builtin_bit_cast(typename Mma<T>::V8, v);
#pragma unroll
    for (int j = 0; j < 8; ++j) *reinterpret_cast<float *>(xtr + (8 * half + j) * PolyLds::XR + row * 4) = static_cast<float>(e[j]);
    *reinterpret_cast<float *>(xtr + (16 + half) * PolyLds::XR + row * 4) = half == 0 && row0 + row < N ? 1.f : 0.f;
}
__device__ __forceinline__ void poly_put_xb(unsigned char *xtb, u32x4 v, int tid) {  // the transposed copy in the storage type
    const int row = tid & 127, half = (tid >> 7) & 1;
#pragma unroll
    for (int j = 0; j < 8; ++j)
        *reinterpret_cast<uint16_t *>(xtb + (8 * half + j) * 272 + row * 2) = (uint16_t)(v[j / 2] >> (16 * (j & 1)));
}
template <typename T>
struct PolyTile {
    u32x4 v[2];
    __device__ __forceinline__ void fetch(const T *base, int64_t stride, int row0, int N, int width, int tid) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int u = tid + 512 * i, row = row0 + (u >> 3), ch = u & 7;
            v[i] = u32x4{0u, 0u, 0u, 0u};
            if (row < N && ch * 8 < width) v[i] = *reinterpret_cast<const u32x4 *>(base + (int64_t)row * stride + ch * 8);
        }
    }
    __device__ __forceinline__ void put(unsigned char *tile, int tid) const {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int u = tid + 512 * i, row = u >> 3, ch = u & 7;
            *reinterpret_cast<u32x4 *>(tile + row * 128 + ((ch ^ walk_swizzle<8>(row)) << 4)) = v[i];
        }
    }
};
// dO, with the normaliser forward's result and n beside it: put() writes g = dO / n and dn = -(dO . O) / n
template <typename T, bool NORM>
struct PolyGrad {
    PolyTile<T> g, o;
    float n[2];
    __device__ __forceinline__ void fetch(const T *go, int64_t gstride, const T *out, int64_t ostride, const float *denom, int row0,
                                          int N, int width, int tid) {
        g.fetch(go, gstride, row0, N, width, tid);
        if constexpr (NORM) {
            o.fetch(out, ostride, row0, N, width, tid);
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int row = row0 + ((tid + 512 * i) >> 3);
                n[i] = row < N ? denom[row] : 1.f;
            }
        }
    }
    // dx: dn as the scores take it (null: nowhere)
    __device__ __forceinline__ void put(unsigned char *tile, float *dn, float *dx, int vhalf, int tid) {
        using V8 = typename Mma<T>::V8;
        if constexpr (NORM) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const V8 a = __builtin_bit_cast(V8, g.v[i]), b = __builtin_bit_cast(V8, o.v[i]);
                const float inv = 1.0f / n[i];
                float dot = 0.f, f[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    dot += static_cast<float>(a[j]) * static_cast<float>(b[j]);
                    f[j] = static_cast<float>(a[j]) * inv;
                }
                g.v[i] = __builtin_bit_cast(u32x4, poly_round8<T>(f));
                dot += __shfl_xor(dot, 1, 64);
                dot += __shfl_xor(dot, 2, 64);
                dot += __shfl_xor(dot, 4, 64);
                // (rounded once for every use, as the quadratic evaluation's bias column holds it.  Of half of v's columns the scores take it
                // unrounded: in early rows dO . V cancels it, and a half's may be the larger one -- rounded, dXq of two rows was up to twice
                // as far from fp64 as the quadratic evaluation's)
                if ((tid & 7) == 0) {
                    const float rounded = static_cast<float>(static_cast<T>(-dot * inv));
                    dn[(tid + 512 * i) >> 3] = rounded;
                    if (dx) dx[(tid + 512 * i) >> 3] = vhalf ? -dot * inv : rounded;
                }
            }
        }
        g.put(tile, tid);
    }
};

// one accumulator block per wave through LDS: 4 KiB each, written and read in lane order
__device__ __forceinline__ void poly_put_acc(unsigned char *ex, int wave, int lane, const f32x16 &v) {
#pragma unroll
    for (int a = 0; a < 4; ++a)
        *reinterpret_cast<f32x4 *>(ex + (wave * 4 + a) * 1024 + lane * 16) = f32x4{v[4 * a], v[4 * a + 1], v[4 * a + 2], v[4 * a + 3]};
}
__device__ __forceinline__ void poly_get_acc(const unsigned char *ex, int wave, int lane, f32x16 &v) {
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        const f32x4 t = *reinterpret_cast<const f32x4 *>(ex + (wave * 4 + a) * 1024 + lane * 16);
#pragma unroll
        for (int b = 0; b < 4; ++b) v[4 * a + b] = t[b];
    }
}

// sixteen consecutive columns (from column `col`) of a row, rounded and stored as two chunks; wide: dst and at (of the row) in floats
template <typename T>
__device__ __forceinline__ void poly_store16(void *dst, int64_t at, const float (&f)[16], int col, int width, int wide = 0) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
        if (col + 8 * h < width) {
            float e[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) e[j] = f[8 * h + j];
            const u32x4 w = __builtin_bit_cast(u32x4, poly_round8<T>(e));
            if (wide) {
                u32x4 *to = reinterpret_cast<u32x4 *>(static_cast<float *>(dst) + at + col + 8 * h);
#pragma unroll
                for (int a = 0; a < 2; ++a)
                    to[a] = u32x4{w[2 * a] << 16, w[2 * a] & 0xffff0000u, w[2 * a + 1] << 16, w[2 * a + 1] & 0xffff0000u};
            } else {
                *reinterpret_cast<u32x4 *>(static_cast<T *>(dst) + at + col + 8 * h) = w;
            }
        }
}

__device__ __forceinline__ void poly_store_part(float *dst, int64_t at, const float (&f)[16]) {
#pragma unroll
    for (int a = 0; a < 4; ++a) *reinterpret_cast<f32x4 *>(dst + at + 4 * a) = f32x4{f[4 * a], f[4 * a + 1], f[4 * a + 2], f[4 * a + 3]};
}

// ---- sums of phi(k) [v, 1]^T (BWD: phi(q) [g, dn]^T) over every segment but the last (the first)
template <typename T, bool NORM, bool BWD, int PART = kPolyWhole>
__global__ __launch_bounds__(512, 2) void poly_totals_kernel(const PolyWalkParams p) {
#if defined(__gfx950__)
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    using L = PolyLds;
    using P = PolyPartOf<PART>;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const PolySlice sl = poly_slice(p);
    if (!sl.valid || sl.seg == (BWD ? 0 : p.n_seg - 1)) return;
    const PolyHead hd = poly_head<P::HALVES>(p, sl.bh);
    const int b = hd.b, h = hd.h, N = p.N;
    const T *X = (BWD ? static_cast<const T *>(p.q) + b * p.qs_b + h * p.qs_h : static_cast<const T *>(p.k) + b * p.ks_b + h * p.ks_h) + P::kOff;
    const int rw = P::width(p);
    const int64_t xs = BWD ? p.qs_n : p.ks_n;
    const T *V = static_cast<const T *>(p.v) + b * p.vs_b + h * p.vs_h + hd.col0;
    const T *G = BWD ? static_cast<const T *>(p.go) + b * p.gs_b + h * p.gs_h + hd.col0 : nullptr;
    const T *O = BWD && NORM ? static_cast<const T *>(p.o) + b * p.os_b + h * p.os_h + hd.col0 : nullptr;
    const float *n = NORM && BWD ? p.denom + (int64_t)hd.bh * N : nullptr;
    // Ten blocks of features on eight waves: a wave has one of its own and a quarter of the rows -- one step of every chunk --
    // of one of the last two, whose four parts are added up at the end (B H 64, N 4096: 21.4 -> 20.8 us forward, 29.7 -> 28.6
    // backward together with the second set of tiles; what is left is the chain load -> LDS -> features of two waves a SIMD)
    // (the products of two halves: sixteen blocks, two to a wave)
    PolyStateOf<P::F> s;
    s.clear(wave, P::CROSS ? 8 + wave : 8 + (wave >> 2));
    constexpr int SETS = 2;  // chunks on their way (registers and LDS)
    u32x4 x[SETS];
    PolyTile<T> v[SETS];
    PolyGrad<T, NORM> go[SETS];
    auto fetch = [&](int c, auto set) {
        constexpr int S = decltype(set)::value;
        const int row0 = c * L::C;
        if (tid < 256) {
            x[S] = poly_fetch_x<T>(X, xs, row0, N, rw, tid);
        } else if constexpr (P::CROSS) {
            x[S] = poly_fetch_x<T>(X + 16, xs, row0, N, p.r - 16, tid);
        }
        if constexpr (BWD)
            go[S].fetch(G, p.gs_n, O, p.os_n, n, row0, N, hd.wv, tid);
        else
            v[S].fetch(V, p.vs_n, row0, N, hd.wv, tid);
    };
    static_for<0, SETS>([&](auto set) {
        if (sl.c_lo + decltype(set)::value < sl.c_hi) fetch(sl.c_lo + decltype(set)::value, set);
    });
    auto chunk = [&](int c, auto set) {
        constexpr int S = decltype(set)::value;
        unsigned char *tile = smem + S * L::tSet;
        float *dn = reinterpret_cast<float *>(tile + L::tDn);
        // (every wave has passed the barrier below a chunk ago, behind its reads of this set)
        if (tid < 256) {
            poly_put_xt<T>(tile + L::tX, x[S], c * L::C, N, tid);
        } else if constexpr (P::CROSS) {
            poly_put_xt<T>(smem + L::tX2 + S * L::XTR, x[S], c * L::C, N, tid);
        }
        if constexpr (BWD)
            go[S].put(tile + L::tV, dn, nullptr, 0, tid);
        else
            v[S].put(tile + L::tV, tid);
        if (c + SETS < sl.c_hi) fetch(c + SETS, set);
        __syncthreads();
        s.template update<NORM, !P::CROSS>(tile + L::tX, tile + L::tV, BWD ? dn : nullptr, lane, wave & 3, smem + L::tX2 + S * L::XTR);
    };
#pragma unroll 1
    for (int c = sl.c_lo; c < sl.c_hi; c += SETS)
        static_for<0, SETS>([&](auto set) {
            if (c + decltype(set)::value < sl.c_hi) chunk(c + decltype(set)::value, set);
        });
    if constexpr (!P::CROSS) {
        // the last two blocks: waves 1 .. 3 and 5 .. 7 hand theirs to waves 0 and 4
        __syncthreads();
        f32x4 *part = reinterpret_cast<f32x4 *>(smem);  // [wave][5][lane]
        if (wave & 3) {
#pragma unroll
            for (int cb = 0; cb < 4; ++cb) part[(wave * 5 + cb) * 64 + lane] = s.st[1][cb];
            part[(wave * 5 + 4) * 64 + lane] = s.ex[1];
        }
        __syncthreads();
        if (wave & 3) {
            s.own[1] = -1;
        } else {
#pragma unroll
            for (int u = 1; u < 4; ++u) {
#pragma unroll
                for (int cb = 0; cb < 4; ++cb) s.st[1][cb] += part[((wave + u) * 5 + cb) * 64 + lane];
                s.ex[1] += part[((wave + u) * 5 + 4) * 64 + lane];
            }
        }
    }
    s.template store<NORM>(p.totals + ((int64_t)sl.bh * p.n_seg + sl.seg) * s.kState, lane);
#else
    (void)p;
#endif
}

// entry states from totals, in place: entry[s] = sum over f < s (reverse: f > s); the loads of eight segments together
// (a template only so that the header can be included by several translation units)
template <int kUnused = 0>
__global__ __launch_bounds__(256) void poly_scan_kernel(float *totals, int n_seg, int64_t total, int reverse, int state) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= total) return;
    const int64_t bh = i / state, e = i - bh * state;
    float *at = totals + (bh * n_seg + (reverse ? n_seg - 1 : 0)) * state + e;
    const int64_t step = reverse ? -(int64_t)state : (int64_t)state;
    float run = 0.f;
    for (int s = 0; s < n_seg; s += 8) {
        float t[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) t[u] = s + u < n_seg - 1 ? at[(s + u) * step] : 0.f;  // (the last one's is not needed)
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (s + u < n_seg) {
                at[(s + u) * step] = run;
                run += t[u];
            }
    }
}

// the entry state of a segment: zeros, one state in memory, or the sum of the totals before (after) it
template <bool NORM, int F>
__device__ __forceinline__ void poly_entry(const PolyWalkParams &p, const PolySlice &sl, bool reverse, int lane, PolyStateOf<F> &s) {
    if (!p.totals) return;
    const float *base = p.totals + (int64_t)sl.bh * p.n_seg * s.kState;
    if (!p.sum_entries) {
        s.template add<NORM>(base + (int64_t)sl.seg * s.kState, lane);
        return;
    }
    s.template add_range<NORM>(base, reverse ? sl.seg + 1 : 0, reverse ? p.n_seg : sl.seg, lane);
}

template <typename T, bool NORM, int PART = kPolyWhole>
__global__ __launch_bounds__(512, 2) void poly_walk_fwd_kernel(const PolyWalkParams p) {
#if defined(__gfx950__)
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    using L = PolyLds;
    using P = PolyPartOf<PART>;
    using M = Mma<T>;
    using V8 = typename M::V8;
    const int tid0 = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid0 >> 6), rb = wave & 3, kh = wave >> 2;
    const PolySlice sl = poly_slice(p);
    if (!sl.valid) return;
    const PolyHead hd = poly_head<P::HALVES>(p, sl.bh);
    const int b = hd.b, h = hd.h, N = p.N;
    const T *Q = static_cast<const T *>(p.q) + b * p.qs_b + h * p.qs_h + P::kOff;
    const T *K = static_cast<const T *>(p.k) + b * p.ks_b + h * p.ks_h + P::kOff;
    const T *V = static_cast<const T *>(p.v) + b * p.vs_b + h * p.vs_h + hd.col0;
    T *O = static_cast<T *>(p.out) + b * p.us_b + h * p.us_h + hd.col0;
    const float c0 = PART == kPolySecond ? 0.f : p.c0, c1 = p.c1, c2 = p.c2;
    const int rw = P::width(p);
    unsigned char *tq = smem + L::fQ, *tk = smem + L::fK, *tkt = smem + L::fKt, *tv = smem + L::fV, *ts = smem + L::fS;
    unsigned char *tq2 = smem + L::fQ2, *tk2 = smem + L::fK2, *tkt2 = smem + L::fKt2;
    float *z = reinterpret_cast<float *>(smem + (P::CROSS ? L::fZ2 : L::fZ)), *sums = reinterpret_cast<float *>(smem + L::fSum);
    unsigned char *exch = smem + L::fEx;
    PolyStateOf<P::F> s;
    if constexpr (P::CROSS)
        s.clear(wave, 8 + wave);
    else
        s.clear_lower(wave);
    poly_entry<NORM>(p, sl, false, tid0 & 63, s);
    if (p.entries && sl.seg > 0)
        s.template store<NORM>(p.entries + ((int64_t)sl.bh * p.n_seg + sl.seg) * P::kRoom, tid0 & 63);
    u32x4 x, x2;
    PolyTile<T> v;
    auto fetch = [&](int c, int tid) {
        const int row0 = c * L::C;
        x = tid < 256 ? poly_fetch_x<T>(Q, p.qs_n, row0, N, rw, tid) : poly_fetch_x<T>(K, p.ks_n, row0, N, rw, tid);
        if constexpr (P::TWO)
            x2 = tid < 256 ? poly_fetch_x<T>(Q + 16, p.qs_n, row0, N, p.r - 16, tid) : poly_fetch_x<T>(K + 16, p.ks_n, row0, N, p.r - 16, tid);
        v.fetch(V, p.vs_n, row0, N, hd.wv, tid);
    };
    fetch(sl.c_lo, tid0);
#pragma unroll 1
    for (int c = sl.c_lo; c < sl.c_hi; ++c) {
        const int tid = poly_opaque(tid0), lane = tid & 63, l32 = lane & 31, g = lane >> 5;
        // (every wave is past the barrier behind its last reads of the tiles and of the state's copy)
        poly_put_x(tid < 256 ? tq : tk, x, tid);
        if (tid >= 256) poly_put_xt<T>(tkt, x, c * L::C, N, tid);
        if constexpr (P::TWO) poly_put_x(tid < 256 ? tq2 : tk2, x2, tid);
        if constexpr (P::CROSS)
            if (tid >= 256) poly_put_xt<T>(tkt2, x2, c * L::C, N, tid);
        v.put(tv, tid);
        s.template to_lds<T, NORM>(ts, z, lane);
        if (c + 1 < sl.c_hi) fetch(c + 1, tid);
        __syncthreads();

        const int trow = 32 * rb + l32, row = c * L::C + trow;
        float *const acc_at = P::PARTS ? p.acc + ((int64_t)sl.bh * N + row) * 64 + 32 * kh + 16 * g : nullptr;
        f32x16 acc[2];
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[0][i] = acc[1][i] = 0.f;
        float rsum = 0.f;
        if (c > 0) {  // phi_w(q) T, this half of the features
            float xr[16];
            poly_row<T>(tq, trow, xr);
            const PolyTurned xt = poly_turn(xr, g, c2);
            PolyTurned xt2;
            if constexpr (P::CROSS) {
                float xr2[16];
                poly_row<T>(tq2, trow, xr2);
                xt2 = poly_turn(xr2, g, c2);
            }
            const uint32_t sa = poly_row_base<256>(walk_e_lane(l32), g);
            auto step = [&](auto ksc) {
                constexpr int KS = decltype(ksc)::value;
                float raw[8];
                PolyTwo f;
                if constexpr (P::CROSS)
                    f = poly_cross_frag<KS>(xt, xt2, raw);
                else
                    f = poly_feature_frag<KS>(xt, g, c0, c1, raw);
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const V8 sf = poly_rd<T>(ts + (KS >> 3) * 64 * 256 + 32 * 256 * e, sa ^ ((KS & 7) << 5));
                    acc[e] = M::mma(sf, f.hi, acc[e]);
                    acc[e] = M::mma(sf, f.lo, acc[e]);
                }
                if constexpr (NORM) {
#pragma unroll
                    for (int a = 0; a < 2; ++a) {
                        const f32x4 zz = *reinterpret_cast<const f32x4 *>(z + 16 * KS + 8 * g + 4 * a);
#pragma unroll
                        for (int j = 0; j < 4; ++j) rsum += raw[4 * a + j] * zz[j];
                    }
                }
            };
            constexpr int H = P::F / 32;
            if (kh == 0)
                static_for<0, H>(step);
            else
                static_for<H, 2 * H>(step);
        }
        if constexpr (P::SCORES) {
            const V8 xq = poly_row_frag<T>(tq, trow, g);
            V8 xq2;
            if constexpr (P::TWO) xq2 = poly_row_frag<T>(tq2, trow, g);
            const PolyPair va = poly_perm_base<128, false>(lane);
#pragma unroll 1
            for (int sb = kh; sb <= rb; sb += 2) {  // every other block of the chunk's scores
                // (the mask as bits, not a branch: see fla_tri_pair.h on scores and branches)
                const uint32_t all = sb < rb ? ~0u : 0u;
                f32x16 sc;
#pragma unroll
                for (int i = 0; i < 16; ++i) sc[i] = 0.f;
                sc = M::mma(poly_row_frag<T>(tk, 32 * sb + l32, g), xq, sc);
                if constexpr (P::TWO) sc = M::mma(poly_row_frag<T>(tk2, 32 * sb + l32, g), xq2, sc);
                float u[16];
                V8 pf[2];
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const float t = c0 + sc[i] * (c1 + c2 * sc[i]);
                    if constexpr (NORM) {
                        u[i] = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, t) & (poly_mask<false>(i, l32, g) | all));
                        rsum += u[i];
                    } else {
                        u[i] = t;
                    }
                }
                poly_round_masked<T, false>(u, NORM ? ~0u : all, l32, g, pf);
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int e = 0; e < 2; ++e)
                        acc[e] = M::mma(poly_tr<T>(tv + 128 * (32 * sb + 16 * t), va, e << 6), pf[t], acc[e]);
            }
        }
        float had[16], had_n = 0.f;  // (on their way under the state's update)
        if constexpr (P::ADDS) {
            poly_get_sums(acc_at, row < N, had);
            if (NORM && row < N) had_n = p.acc_n[(int64_t)sl.bh * N + row];
        }
        if (c + 1 < sl.c_hi) s.template update<NORM>(tkt, tv, nullptr, lane, 0, tkt2);
        // each of the two waves of these rows finishes one half of the columns: the other half's sums go to the other wave
        {
            f32x16 mine;
#pragma unroll
            for (int i = 0; i < 16; ++i) mine[i] = poly_pick(kh, acc[0][i], acc[1][i]);
            poly_put_acc(exch, wave, lane, mine);
        }
        if constexpr (NORM) {
            rsum += __shfl_xor(rsum, 32, 64);
            if (g == 0) sums[kh * L::C + trow] = rsum;
        }
        __syncthreads();
        f32x16 other;
        poly_get_acc(exch, wave ^ 4, lane, other);
        float f[16], inv = 1.f;
        if constexpr (NORM) {
            float own = sums[trow] + sums[L::C + trow];
            if constexpr (P::PARTS) own += had_n;
            if constexpr (P::SCORES) {
                const float n = own + p.eps;
                inv = 1.0f / n;
                if (kh == 0 && g == 0 && row < N && hd.col0 == 0) p.denom[(int64_t)hd.bh * N + row] = n;
            } else {
                if (kh == 0 && g == 0 && row < N) p.acc_n[(int64_t)sl.bh * N + row] = own;
            }
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            f[i] = poly_pick(kh, acc[1][i], acc[0][i]) + other[i];
            if constexpr (P::ADDS) f[i] += had[i];
            f[i] *= inv;
        }
        if constexpr (P::SCORES) {
            if (row < N) poly_store16<T>(O, (int64_t)row * p.us_n, f, 32 * kh + 16 * g, hd.wv);
        } else {
            if (row < N) poly_store_part(acc_at, 0, f);
        }
    }
#else
    (void)p;
#endif
}

// dx += the gradient at x of phi_w(x) . (S [g, extra]): H = S g for the row's feature blocks FB0 .. FB1 - 1, contracted with
// the row.
// S: the rounded state's tiles; gf: the row's g (v) as operands; z, extra: the state's last column and its factor.
// Returns this lane's part of it (the other part is in the lane of the other g) in dx.
template <typename T, bool NORM, int FB0, int FB1>
__device__ __forceinline__ void poly_contract(const unsigned char *S, const float *z, float extra, const typename Mma<T>::V8 (&gf)[4],
                                              const float (&x)[16], int lane, float c1, float c2, float (&dx)[16]) {
    using M = Mma<T>;
    const int g = lane >> 5;
    const PolyPair sa = poly_perm_base<256, true>(lane);
    // of a block's feature v with the difference d = 2 FB + g: a = v, b = (v + 2 FB + g) % 16.  q1: sums of H x_b by a; q2: of
    // H x_a by b - g; y: the row turned by g
    float q1[16], q2[16], y[16], lin[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) q1[i] = q2[i] = lin[i] = 0.f, y[i] = poly_pick(g, x[(i + 1) & 15], x[i]);
    static_for<FB0, FB1>([&](auto fbc) {
        constexpr int FB = decltype(fbc)::value;
        f32x16 hh;
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            f32x4 zz = {0.f, 0.f, 0.f, 0.f};
            if constexpr (NORM) zz = *reinterpret_cast<const f32x4 *>(z + 32 * FB + 16 * g + 4 * a);
#pragma unroll
            for (int j = 0; j < 4; ++j) hh[4 * a + j] = NORM ? zz[j] * extra : 0.f;
        }
#pragma unroll
        for (int kc = 0; kc < 4; ++kc)
            hh = M::mma(poly_tr<T>(S + (FB >> 2) * 64 * 256 + 16 * 256 * kc, sa, (FB & 3) << 6), gf[kc], hh);
        // hh[v]: feature 32 FB + 16 g + v
        if constexpr (FB < 4) {
            const float once = FB == 0 ? (g ? 1.f : 0.5f) : 1.f;  // (d = 0: both sums meet in x_v)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const float t = FB == 0 ? hh[v] * once : hh[v];
                q1[v] += t * y[(v + 2 * FB) & 15];
                q2[(v + 2 * FB) & 15] += t * x[v];
            }
        } else {  // g = 0: d = 8, the row's first half; g = 1: its second half, the one
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float t = poly_pick(g, 0.f, hh[j]);
                q1[j] += t * x[j + 8], q1[j + 8] += t * x[j];
                lin[j] = poly_pick(g, 0.f, hh[j + 8]), lin[j + 8] = poly_pick(g, hh[j], 0.f);
            }
        }
        if constexpr (FB % 2 == 1) __builtin_amdgcn_sched_barrier(0);  // (two blocks at a time: registers)
    });
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        dx[j] = 2.f * c2 * (q1[j] + poly_pick(g, q2[(j + 15) & 15], q2[j]));
        if constexpr (FB1 == PolyFeatures::kBlocks) dx[j] += c1 * lin[j];
    }
}

// ... of the products of a column of each half: the row's halves a and b, their parts of the gradient da and db; feature blocks FB0 ..
template <typename T, bool NORM, int FB0, int FB1>
__device__ __forceinline__ void poly_contract_cross(const unsigned char *S, const float *z, float extra, const typename Mma<T>::V8 (&gf)[4],
                                                    const float (&a)[16], const float (&b)[16], int lane, float c2, float (&da)[16],
                                                    float (&db)[16]) {
    using M = Mma<T>;
    const int g = lane >> 5;
    const PolyPair sa = poly_perm_base<256, true>(lane);
    float q1[16], q2[16], y[16];  // as above: sums of H b by a; of H a by b - g; b turned by g
#pragma unroll
    for (int i = 0; i < 16; ++i) q1[i] = q2[i] = 0.f, y[i] = poly_pick(g, b[(i + 1) & 15], b[i]);
    static_for<FB0, FB1>([&](auto fbc) {
        constexpr int FB = decltype(fbc)::value;
        f32x16 hh;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            f32x4 zz = {0.f, 0.f, 0.f, 0.f};
            if constexpr (NORM) zz = *reinterpret_cast<const f32x4 *>(z + 32 * FB + 16 * g + 4 * u);
#pragma unroll
            for (int j = 0; j < 4; ++j) hh[4 * u + j] = NORM ? zz[j] * extra : 0.f;
        }
#pragma unroll
        for (int kc = 0; kc < 4; ++kc)
            hh = M::mma(poly_tr<T>(S + (FB >> 2) * 64 * 256 + 16 * 256 * kc, sa, (FB & 3) << 6), gf[kc], hh);
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            q1[v] += hh[v] * y[(v + 2 * FB) & 15];
            q2[(v + 2 * FB) & 15] += hh[v] * a[v];
        }
        if constexpr (FB % 2 == 1) __builtin_amdgcn_sched_barrier(0);  // (two blocks at a time: registers)
    });
#pragma unroll
    for (int j = 0; j < 16; ++j) da[j] = 2.f * c2 * q1[j], db[j] = 2.f * c2 * poly_pick(g, q2[(j + 15) & 15], q2[j]);
}
// the sums of a row's two lanes, each lane with the sixteen columns it has of the row: da in those of g = 0, db in those of g = 1
__device__ __forceinline__ void poly_row_sums(const float (&da)[16], const float (&db)[16], int g, float (&f)[16]) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const float give = poly_pick(g, da[i], db[i]), own = poly_pick(g, db[i], da[i]);
        f[i] = own + __shfl_xor(give, 32, 64);
    }
}

// dq: chunks ascending, T += phi(k) [v, 1]^T as in forward.  Each of the two waves of a row block takes a part of the feature
// blocks and every other score block.
template <typename T, bool NORM, bool SUMS, int PART = kPolyWhole>
__global__ __launch_bounds__(512, 2) void poly_walk_dq_kernel(const PolyWalkParams p) {
#if defined(__gfx950__)
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    using L = PolyLds;
    using P = PolyPartOf<PART>;
    static_assert(!SUMS || !P::PARTS, "parts take a totals kernel");
    using M = Mma<T>;
    using V8 = typename M::V8;
    const int tid0 = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid0 >> 6), rb = wave & 3, kh = wave >> 2;
    const PolySlice sl = poly_slice(p);
    if (!sl.valid) return;
    const PolyHead hd = poly_head<P::HALVES>(p, sl.bh);
    const int b = hd.b, h = hd.h, N = p.N;
    const T *Q = static_cast<const T *>(p.q) + b * p.qs_b + h * p.qs_h + P::kOff;
    const T *K = static_cast<const T *>(p.k) + b * p.ks_b + h * p.ks_h + P::kOff;
    const T *V = static_cast<const T *>(p.v) + b * p.vs_b + h * p.vs_h + hd.col0;
    const T *G = static_cast<const T *>(p.go) + b * p.gs_b + h * p.gs_h + hd.col0;
    const T *O = NORM ? static_cast<const T *>(p.o) + b * p.os_b + h * p.os_h + hd.col0 : nullptr;
    const float *den = NORM ? p.denom + (int64_t)hd.bh * N : nullptr;
    const int64_t dq_at = b * p.dqs_b + h * p.dqs_h;
    const float c1 = p.c1, c2 = p.c2;
    const int rw = P::width(p);
    unsigned char *tq = smem + L::qQ, *tk = smem + L::qK, *tkt = smem + L::qKt, *tkb = smem + L::qKb, *tv = smem + L::qV, *tg = smem + L::qG,
                  *ts = smem + L::qS, *exch = smem + (P::PARTS ? L::qEx2 : L::qEx);
    unsigned char *tq2 = smem + L::qQ2, *tk2 = smem + L::qK2, *tkt2 = smem + L::qKt2, *tkb2 = smem + L::qKb2;
    float *z = reinterpret_cast<float *>(smem + (P::CROSS ? L::qZ2 : L::qZ)), *dn = reinterpret_cast<float *>(smem + L::qDn), *dnx = P::HALVES ? reinterpret_cast<float *>(smem + L::qDx) : dn;
    unsigned char *tqt = smem + L::qQt;
    PolyStateOf<P::F> s;
    PolyState sums;
    if constexpr (P::CROSS)
        s.clear(wave, 8 + wave);
    else
        s.clear_lower(wave);
    if constexpr (SUMS) sums.clear_beside_lower(wave);
    const bool with_sums = SUMS && sl.seg > 0;  // (the first segment's total is under no sum)
    if (sl.seg > 0) s.template add<NORM>(p.entries + ((int64_t)sl.bh * p.n_seg + sl.seg) * P::kRoom, tid0 & 63);
    u32x4 x, x2;
    PolyTile<T> v;
    PolyGrad<T, NORM> go;
    auto fetch = [&](int c, int tid) {
        const int row0 = c * L::C;
        x = tid < 256 ? poly_fetch_x<T>(Q, p.qs_n, row0, N, rw, tid) : poly_fetch_x<T>(K, p.ks_n, row0, N, rw, tid);
        if constexpr (P::TWO)
            x2 = tid < 256 ? poly_fetch_x<T>(Q + 16, p.qs_n, row0, N, p.r - 16, tid) : poly_fetch_x<T>(K + 16, p.ks_n, row0, N, p.r - 16, tid);
        v.fetch(V, p.vs_n, row0, N, hd.wv, tid);
        go.fetch(G, p.gs_n, O, p.os_n, den, row0, N, hd.wv, tid);
    };
    fetch(sl.c_lo, tid0);
#pragma unroll 1
    for (int c = sl.c_lo; c < sl.c_hi; ++c) {
        const int tid = poly_opaque(tid0), lane = tid & 63, l32 = lane & 31, g = lane >> 5;
        // (every wave is past the barrier behind its last reads of the tiles and of the state's copy)
        poly_put_x(tid < 256 ? tq : tk, x, tid);
        if constexpr (P::TWO) poly_put_x(tid < 256 ? tq2 : tk2, x2, tid);
        if (tid >= 256) {
            poly_put_xt<T>(tkt, x, c * L::C, N, tid);
            if constexpr (P::SCORES) poly_put_xb(tkb, x, tid);
            if constexpr (P::CROSS) poly_put_xt<T>(tkt2, x2, c * L::C, N, tid);
            if constexpr (PART == kPolyFirst) poly_put_xb(tkb2, x2, tid);
        } else if (with_sums) {
            poly_put_xt<T>(tqt, x, c * L::C, N, tid);
        }
        v.put(tv, tid);
        go.put(tg, dn, P::HALVES ? dnx : nullptr, p.vhalf, tid);
        s.template to_lds<T, NORM>(ts, z, lane);
        if (c + 1 < sl.c_hi) fetch(c + 1, tid);
        __syncthreads();

        const int trow = 32 * rb + l32, row = c * L::C + trow;
        const uint32_t ra = poly_row_base<128>(l32, g);
        V8 gf[4];
#pragma unroll
        for (int kc = 0; kc < 4; ++kc) gf[kc] = poly_rd<T>(tg + 32 * 128 * rb, ra ^ (kc << 5));
        const float dni = NORM ? dnx[trow] : 0.f;
        float *const acc_at = P::PARTS ? p.acc_q + ((int64_t)sl.bh * N + row) * 32 + 16 * g : nullptr;
        float dxs[16], dxb[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) dxs[i] = dxb[i] = 0.f;
        if (c > 0) {
            float xr[16];
            poly_row<T>(tq, trow, xr);
            if constexpr (P::CROSS) {
                float xr2[16];
                poly_row<T>(tq2, trow, xr2);
                if (kh == 0)
                    poly_contract_cross<T, NORM, 0, 4>(ts, z, dni, gf, xr, xr2, lane, c2, dxs, dxb);
                else
                    poly_contract_cross<T, NORM, 4, 8>(ts, z, dni, gf, xr, xr2, lane, c2, dxs, dxb);
            } else if (kh == 0)
                poly_contract<T, NORM, 0, 2>(ts, z, dni, gf, xr, lane, c1, c2, dxs);
            else
                poly_contract<T, NORM, 2, PolyFeatures::kBlocks>(ts, z, dni, gf, xr, lane, c1, c2, dxs);
        }
        f32x16 dx;
#pragma unroll
        for (int i = 0; i < 16; ++i) dx[i] = 0.f;
        if constexpr (P::SCORES) {
            const V8 xq = poly_row_frag<T>(tq, trow, g);
            V8 xq2;
            if constexpr (P::TWO) xq2 = poly_row_frag<T>(tq2, trow, g);
            const int rc = walk_e_lane(l32) & 15;  // (columns 16 .. of the 32-wide block of dq: the second half's, or not used)
            const unsigned char *kb = PART == kPolyFirst && walk_e_lane(l32) >= 16 ? tkb2 : tkb;
#pragma unroll 1
            for (int sb = kh; sb <= rb; sb += 2) {
                const uint32_t all = sb < rb ? ~0u : 0u;
                f32x16 m, u;
#pragma unroll
                for (int i = 0; i < 16; ++i) m[i] = dni, u[i] = 0.f;
                u = M::mma(poly_row_frag<T>(tk, 32 * sb + l32, g), xq, u);
                if constexpr (P::TWO) u = M::mma(poly_row_frag<T>(tk2, 32 * sb + l32, g), xq2, u);
#pragma unroll
                for (int kc = 0; kc < 4; ++kc) m = M::mma(poly_rd<T>(tv + 32 * 128 * sb, ra ^ (kc << 5)), gf[kc], m);
                V8 df[2];
                float d[16];
#pragma unroll
                for (int i = 0; i < 16; ++i) d[i] = m[i] * (c1 + 2.f * c2 * u[i]);
                poly_round_masked<T, false>(d, all, l32, g, df);
#pragma unroll
                for (int t = 0; t < 2; ++t) dx = M::mma(poly_col_frag<T>(kb, rc, 32 * sb + 16 * t, g), df[t], dx);
                if constexpr (P::TWO_TERMS)
                    if (p.vhalf) {
                        poly_left_over<T>(d, df);
                        poly_round_masked<T, false>(d, all, l32, g, df);
#pragma unroll
                        for (int t = 0; t < 2; ++t) dx = M::mma(poly_col_frag<T>(kb, rc, 32 * sb + 16 * t, g), df[t], dx);
                    }
            }
        }
        float f[16];  // (lanes of g = 0 hold the block's columns 0 .. 15)
        if constexpr (!P::PARTS) {
#pragma unroll
            for (int i = 0; i < 16; ++i) f[i] = dxs[i] + __shfl_xor(dxs[i], 32, 64) + dx[i];
        } else {
            if constexpr (PART == kPolySecond)
                poly_row_sums(dxb, dxs, g, f);
            else
                poly_row_sums(dxs, dxb, g, f);
#pragma unroll
            for (int i = 0; i < 16; ++i) f[i] += dx[i];
        }
        if (kh == 1 && (P::PARTS || g == 0)) {
#pragma unroll
            for (int a = 0; a < 4; ++a)
                *reinterpret_cast<f32x4 *>(exch + ((4 * g + a) * L::C + trow) * 16) = f32x4{f[4 * a], f[4 * a + 1], f[4 * a + 2], f[4 * a + 3]};
        }
        float had[16];
        if constexpr (P::ADDS) poly_get_sums(acc_at, kh == 0 && row < N, had);
        if (c + 1 < sl.c_hi) s.template update<NORM>(tkt, tv, nullptr, lane, 0, tkt2);
        if constexpr (SUMS)
            if (with_sums) sums.template update<NORM>(tqt, tg, dn, lane);
        __syncthreads();
        if (kh == 0 && (P::PARTS || g == 0)) {
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                const f32x4 t = *reinterpret_cast<const f32x4 *>(exch + ((4 * g + a) * L::C + trow) * 16);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    f[4 * a + j] += t[j];
                    if constexpr (P::ADDS) f[4 * a + j] += had[4 * a + j];
                }
            }
            if (row < N) {
                if constexpr (!P::SCORES)
                    poly_store_part(acc_at, 0, f);
                else if (P::HALVES && p.vhalf)
                    poly_store_part(p.dq_part, P::PARTS ? ((int64_t)sl.bh * N + row) * 32 + 16 * g : ((int64_t)sl.bh * N + row) * 16, f);
                else
                    poly_store16<T>(p.dq, dq_at + (int64_t)row * p.dqs_n, f, P::PARTS ? 16 * g : 0, p.r, p.wide_out);
            }
        }
    }
    if constexpr (SUMS)
        if (with_sums) sums.template store<NORM>(p.totals + ((int64_t)sl.bh * p.n_seg + sl.seg) * PolyFeatures::kState, tid0 & 63);
#else
    (void)p;
#endif
}

// dk and dV: chunks descending, U += phi(q) [g, dn]^T
template <typename T, bool NORM, int PART = kPolyWhole>
__global__ __launch_bounds__(512, 2) void poly_walk_dkdv_kernel(const PolyWalkParams p) {
#if defined(__gfx950__)
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    using L = PolyLds;
    using P = PolyPartOf<PART>;
    using M = Mma<T>;
    using V8 = typename M::V8;
    const int tid0 = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid0 >> 6), rb = wave & 3, half = wave >> 2;
    const PolySlice sl = poly_slice(p);
    if (!sl.valid) return;
    const PolyHead hd = poly_head<P::HALVES>(p, sl.bh);
    const int b = hd.b, h = hd.h, N = p.N;
    const T *Q = static_cast<const T *>(p.q) + b * p.qs_b + h * p.qs_h + P::kOff;
    const T *K = static_cast<const T *>(p.k) + b * p.ks_b + h * p.ks_h + P::kOff;
    const T *V = static_cast<const T *>(p.v) + b * p.vs_b + h * p.vs_h + hd.col0;
    const T *G = static_cast<const T *>(p.go) + b * p.gs_b + h * p.gs_h + hd.col0;
    const T *O = NORM ? static_cast<const T *>(p.o) + b * p.os_b + h * p.os_h + hd.col0 : nullptr;
    const float *den = NORM ? p.denom + (int64_t)hd.bh * N : nullptr;
    const int64_t dk_at = b * p.dks_b + h * p.dks_h, dv_at = b * p.dvs_b + h * p.dvs_h + hd.col0;
    const float c0 = PART == kPolySecond ? 0.f : p.c0, c1 = p.c1, c2 = p.c2;
    const int rw = P::width(p);
    unsigned char *tq = smem + L::kQ, *tqt = smem + L::kQt, *tqb = smem + L::kQb, *tk = smem + L::kK, *tv = smem + L::kV, *tg = smem + L::kG,
                  *us = smem + L::kU, *exch = smem + L::kEx;
    unsigned char *tq2 = smem + L::kQ2, *tk2 = smem + L::kK2, *tqt2 = smem + L::kQt2, *tqb2 = smem + L::kQb2;
    float *y = reinterpret_cast<float *>(smem + (P::CROSS ? L::kY2 : L::kY)), *dn = reinterpret_cast<float *>(smem + L::kDn), *dnx = P::HALVES ? reinterpret_cast<float *>(smem + L::kDx) : dn;
    PolyStateOf<P::F> su;
    if constexpr (P::CROSS)
        su.clear(wave, 8 + wave);
    else
        su.clear_upper(wave);
    poly_entry<NORM>(p, sl, true, tid0 & 63, su);
    u32x4 x, x2;
    PolyTile<T> v;
    PolyGrad<T, NORM> go;
    auto fetch = [&](int c, int tid) {
        const int row0 = c * L::C;
        x = tid < 256 ? poly_fetch_x<T>(Q, p.qs_n, row0, N, rw, tid) : poly_fetch_x<T>(K, p.ks_n, row0, N, rw, tid);
        if constexpr (P::TWO)
            x2 = tid < 256 ? poly_fetch_x<T>(Q + 16, p.qs_n, row0, N, p.r - 16, tid) : poly_fetch_x<T>(K + 16, p.ks_n, row0, N, p.r - 16, tid);
        v.fetch(V, p.vs_n, row0, N, hd.wv, tid);
        go.fetch(G, p.gs_n, O, p.os_n, den, row0, N, hd.wv, tid);
    };
    fetch(sl.c_hi - 1, tid0);
#pragma unroll 1
    for (int c = sl.c_hi - 1; c >= sl.c_lo; --c) {
        const int tid = poly_opaque(tid0), lane = tid & 63, l32 = lane & 31, g = lane >> 5;
        const bool after = c + 1 < p.n_chunks;  // (U of this chunk holds anything)
        // (every wave is past the barrier behind its last reads of the tiles and of the state's copy)
        poly_put_x(tid < 256 ? tq : tk, x, tid);
        if constexpr (P::TWO) poly_put_x(tid < 256 ? tq2 : tk2, x2, tid);
        if (tid < 256) {
            poly_put_xt<T>(tqt, x, c * L::C, N, tid);
            if constexpr (P::SCORES) poly_put_xb(tqb, x, tid);
            if constexpr (P::CROSS) poly_put_xt<T>(tqt2, x2, c * L::C, N, tid);
            if constexpr (PART == kPolyFirst) poly_put_xb(tqb2, x2, tid);
        }
        v.put(tv, tid);
        go.put(tg, dn, P::HALVES ? dnx : nullptr, p.vhalf, tid);
        if (after) su.template to_lds<T, NORM>(us, y, lane);
        if (c > sl.c_lo) fetch(c - 1, tid);
        __syncthreads();

        const int trow = 32 * rb + l32, row = c * L::C + trow;
        // dV: the waves of half 0 form phi_w(k) U, those of half 1 -- after dk -- the chunk's own part; each finishes one
        // half of the columns
        float *const acc_at = P::PARTS ? p.acc + ((int64_t)sl.bh * N + row) * 64 + 32 * half + 16 * g : nullptr;
        float *const acck_at = P::PARTS ? p.acc_k + ((int64_t)sl.bh * N + row) * 32 + 16 * g : nullptr;
        float had_k[16];
        if constexpr (PART == kPolySecond) poly_get_sums(acck_at, half == 1 && row < N, had_k);
        f32x16 acc[2];
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[0][i] = acc[1][i] = 0.f;
        if (half == 0) {
            if (after) {
                float xr[16];
                poly_row<T>(tk, trow, xr);
                const PolyTurned xt = poly_turn(xr, g, c2);
                PolyTurned xt2;
                if constexpr (P::CROSS) {
                    float xr2[16];
                    poly_row<T>(tk2, trow, xr2);
                    xt2 = poly_turn(xr2, g, c2);
                }
                const uint32_t sa = poly_row_base<256>(walk_e_lane(l32), g);
                static_for<0, P::F / 16>([&](auto ksc) {
                    constexpr int KS = decltype(ksc)::value;
                    float raw[8];
                    PolyTwo f;
                    if constexpr (P::CROSS)
                        f = poly_cross_frag<KS>(xt, xt2, raw);
                    else
                        f = poly_feature_frag<KS>(xt, g, c0, c1, raw);
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        const V8 uf = poly_rd<T>(us + (KS >> 3) * 64 * 256 + 32 * 256 * e, sa ^ ((KS & 7) << 5));
                        acc[e] = M::mma(uf, f.hi, acc[e]);
                        acc[e] = M::mma(uf, f.lo, acc[e]);
                    }
                });
            }
        } else {
            const V8 xk = poly_row_frag<T>(tk, trow, g);
            V8 xk2;
            if constexpr (P::TWO) xk2 = poly_row_frag<T>(tk2, trow, g);
            const uint32_t ra = poly_row_base<128>(l32, g);
            const int rc = walk_e_lane(l32) & 15;  // (columns 16 .. of the 32-wide block of dk: the second half's, or not used)
            const unsigned char *qb = PART == kPolyFirst && walk_e_lane(l32) >= 16 ? tqb2 : tqb;
            const PolyPair ga = poly_perm_base<128, false>(lane);
            V8 vf[4];
#pragma unroll
            for (int kc = 0; kc < 4; ++kc) vf[kc] = poly_rd<T>(tv + 32 * 128 * rb, ra ^ (kc << 5));
            float dxs[16], dxb[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) dxs[i] = dxb[i] = 0.f;
            if (after) {
                float xr[16];
                poly_row<T>(tk, trow, xr);
                if constexpr (P::CROSS) {
                    float xr2[16];
                    poly_row<T>(tk2, trow, xr2);
                    poly_contract_cross<T, NORM, 0, 8>(us, y, 1.f, vf, xr, xr2, lane, c2, dxs, dxb);
                } else {
                    poly_contract<T, NORM, 0, PolyFeatures::kBlocks>(us, y, 1.f, vf, xr, lane, c1, c2, dxs);
                }
            }
            f32x16 dx;
#pragma unroll
            for (int i = 0; i < 16; ++i) dx[i] = 0.f;
#pragma unroll 1
            for (int sb = P::SCORES ? rb : 4; sb < 4; ++sb) {
                const uint32_t all = sb > rb ? ~0u : 0u;
                f32x16 m, u;
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    f32x4 d = {0.f, 0.f, 0.f, 0.f};
                    if constexpr (NORM) d = *reinterpret_cast<const f32x4 *>(dnx + 32 * sb + 8 * a + 4 * g);
#pragma unroll
                    for (int j = 0; j < 4; ++j) m[4 * a + j] = d[j], u[4 * a + j] = 0.f;
                }
                u = M::mma(poly_row_frag<T>(tq, 32 * sb + l32, g), xk, u);
                if constexpr (P::TWO) u = M::mma(poly_row_frag<T>(tq2, 32 * sb + l32, g), xk2, u);
#pragma unroll
                for (int kc = 0; kc < 4; ++kc) m = M::mma(poly_rd<T>(tg + 32 * 128 * sb, ra ^ (kc << 5)), vf[kc], m);
                V8 df[2], pf[2];
                float d[16], f[16];
#pragma unroll
                for (int i = 0; i < 16; ++i) d[i] = m[i] * (c1 + 2.f * c2 * u[i]), f[i] = c0 + u[i] * (c1 + c2 * u[i]);
                poly_round_masked<T, true>(d, all, l32, g, df);
                poly_round_masked<T, true>(f, all, l32, g, pf);
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    dx = M::mma(poly_col_frag<T>(qb, rc, 32 * sb + 16 * t, g), df[t], dx);
#pragma unroll
                    for (int e = 0; e < 2; ++e)
                        acc[e] = M::mma(poly_tr<T>(tg + 128 * (32 * sb + 16 * t), ga, e << 6), pf[t], acc[e]);
                }
                if constexpr (P::TWO_TERMS)
                    if (p.vhalf) {
                        poly_left_over<T>(d, df);
                        poly_round_masked<T, true>(d, all, l32, g, df);
#pragma unroll
                        for (int t = 0; t < 2; ++t) dx = M::mma(poly_col_frag<T>(qb, rc, 32 * sb + 16 * t, g), df[t], dx);
                    }
            }
            if constexpr (PART == kPolyFirst) poly_get_sums(acck_at, row < N, had_k);  // (earlier: 16 registers spilled)
            float f[16];
            if constexpr (!P::PARTS) {
#pragma unroll
                for (int i = 0; i < 16; ++i) f[i] = dxs[i] + __shfl_xor(dxs[i], 32, 64) + dx[i];
            } else {
                if constexpr (PART == kPolySecond)
                    poly_row_sums(dxb, dxs, g, f);
                else
                    poly_row_sums(dxs, dxb, g, f);
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    f[i] += dx[i];
                    if constexpr (PART != kPolyCross) f[i] += had_k[i];
                }
            }
            if (row < N && (P::PARTS || g == 0)) {
                if constexpr (!P::SCORES)
                    poly_store_part(acck_at, 0, f);
                else if (P::HALVES && p.vhalf)
                    poly_store_part(p.dk_part, P::PARTS ? ((int64_t)sl.bh * N + row) * 32 + 16 * g : ((int64_t)sl.bh * N + row) * 16, f);
                else
                    poly_store16<T>(p.dk, dk_at + (int64_t)row * p.dks_n, f, P::PARTS ? 16 * g : 0, p.r, p.wide_out);
            }
        }
        float had[16];
        if constexpr (P::ADDS) poly_get_sums(acc_at, row < N, had);
        if (c > sl.c_lo) su.template update<NORM>(tqt, tg, dn, lane, 0, tqt2);
        {
            f32x16 mine;
#pragma unroll
            for (int i = 0; i < 16; ++i) mine[i] = poly_pick(half, acc[0][i], acc[1][i]);
            poly_put_acc(exch, wave, lane, mine);
        }
        __syncthreads();
        {
            f32x16 other;
            poly_get_acc(exch, wave ^ 4, lane, other);
            float f[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                f[i] = poly_pick(half, acc[1][i], acc[0][i]) + other[i];
                if constexpr (P::ADDS) f[i] += had[i];
            }
            if constexpr (!P::SCORES) {
                if (row < N) poly_store_part(acc_at, 0, f);
            } else {
                if (row < N) poly_store16<T>(p.dv, dv_at + (int64_t)row * p.dvs_n, f, 32 * half + 16 * g, hd.wv, p.wide_out);
            }
        }
    }
#else
    (void)p;
#endif
}

// dq (grid y 1: dk) of a v of two halves: their parts added and rounded; a thread has eight columns of a row.  Bound by memory: 128 bytes in
// and 32 out a row
template <typename T>
__global__ __launch_bounds__(256) void poly_add_halves_kernel(const PolyWalkParams p, int64_t total) {
#if defined(__gfx950__)
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= total) return;
    const int chunks = p.r >> 3, N = p.N;
    const int64_t rows = i / chunks, bh = rows / N, row = rows - bh * N;
    const int col = 8 * (int)(i - rows * chunks);
    const int64_t b = bh / p.H, h = bh - b * p.H;
    const bool second = blockIdx.y != 0;
    const int pitch = p.r > 16 ? 32 : 16;
    const float *part = (second ? p.dk_part : p.dq_part) + (2 * bh * N + row) * pitch + col;
    float f[16];
#pragma unroll
    for (int a = 0; a < 2; ++a) {
        const f32x4 x = *reinterpret_cast<const f32x4 *>(part + 4 * a), y = *reinterpret_cast<const f32x4 *>(part + (int64_t)N * pitch + 4 * a);
#pragma unroll
        for (int j = 0; j < 4; ++j) f[4 * a + j] = x[j] + y[j], f[8 + 4 * a + j] = 0.f;
    }
    if (second)
        poly_store16<T>(p.dk, b * p.dks_b + h * p.dks_h + row * p.dks_n, f, col, col + 8, p.wide_out);
    else
        poly_store16<T>(p.dq, b * p.dqs_b + h * p.dqs_h + row * p.dqs_n, f, col, col + 8, p.wide_out);
#else
    (void)p, (void)total;
#endif
}

template <auto kern>
hipError_t launch_poly_kernel(PolyWalkParams p, int smem, hipStream_t stream) {
    p.place = xcd_place(p.BH, p.n_seg, p.ks_h, kWholeHeadParts, p.n_seg <= 20 ? 32 : 0), p.n_seg_inv = xcd_inverse(p.n_seg);  // (kSumOnLoadPoly)
    const int64_t grid = (int64_t)8 * ((p.BH + 7) / 8) * p.n_seg;
    if (grid > 0x7fffffffLL) return hipErrorInvalidConfiguration;
    if (hipError_t e = ensure_dynamic_lds<kern>(smem)) return e;
    return launch_kernel<kern>(dim3((unsigned)grid), dim3(512), smem, stream, p);
}

// a kernel's instantiation for the plan: pick(part)
template <typename Pick>
hipError_t poly_by_part(const PolyWalkParams &p, Pick &&pick) {
    switch (p.part) {
        case kPolyWhole: return p.vhalf ? pick(std::integral_constant<int, kPolyHalves>{}) : pick(std::integral_constant<int, kPolyWhole>{});
        case kPolyFirst: return pick(std::integral_constant<int, kPolyFirst>{});
        case kPolySecond: return pick(std::integral_constant<int, kPolySecond>{});
        case kPolyCross: return pick(std::integral_constant<int, kPolyCross>{});
    }
    return hipErrorInvalidValue;
}

template <typename T>
hipError_t launch_poly_totals(const PolyWalkParams &p, bool bwd, hipStream_t stream) {
    return poly_by_part(p, [&](auto part) {
        constexpr int P = decltype(part)::value, smem = P == kPolyCross ? PolyLds::tTotalTwo : PolyLds::tTotal;
        if (bwd)
            return p.denom ? launch_poly_kernel<poly_totals_kernel<T, true, true, P>>(p, smem, stream)
                           : launch_poly_kernel<poly_totals_kernel<T, false, true, P>>(p, smem, stream);
        return p.denom ? launch_poly_kernel<poly_totals_kernel<T, true, false, P>>(p, smem, stream)
                       : launch_poly_kernel<poly_totals_kernel<T, false, false, P>>(p, smem, stream);
    });
}

template <typename T>
hipError_t launch_poly_walk(const PolyWalkParams &p, bool bwd, hipStream_t stream) {
    if (p.part && (p.r <= 16 || p.u_totals || !p.acc || !(bwd ? p.acc_q && p.acc_k : p.acc_n != nullptr))) return hipErrorInvalidValue;
    if (!bwd)
        return poly_by_part(p, [&](auto part) {
            constexpr int P = decltype(part)::value, smem = PolyPartOf<P>::PARTS ? PolyLds::fTotalTwo : PolyLds::fTotal;
            return p.denom ? launch_poly_kernel<poly_walk_fwd_kernel<T, true, P>>(p, smem, stream)
                           : launch_poly_kernel<poly_walk_fwd_kernel<T, false, P>>(p, smem, stream);
        });
    if (p.n_seg > 1 && !p.entries) return hipErrorInvalidValue;
    if (p.vhalf && (!p.dq_part || !p.dk_part || p.BH % 2)) return hipErrorInvalidValue;
    if (p.u_totals && (!p.sum_entries || !p.totals || p.n_seg < 3)) return hipErrorInvalidValue;
    const hipError_t dq = poly_by_part(p, [&](auto part) {
        constexpr int P = decltype(part)::value, smem = PolyPartOf<P>::PARTS ? PolyLds::qTotalTwo : PolyLds::qTotal;
        if constexpr (!PolyPartOf<P>::PARTS)
            if (p.u_totals)
                return p.denom ? launch_poly_kernel<poly_walk_dq_kernel<T, true, true, P>>(p, PolyLds::qTotalSums, stream)
                               : launch_poly_kernel<poly_walk_dq_kernel<T, false, true, P>>(p, PolyLds::qTotalSums, stream);
        return p.denom ? launch_poly_kernel<poly_walk_dq_kernel<T, true, false, P>>(p, smem, stream)
                       : launch_poly_kernel<poly_walk_dq_kernel<T, false, false, P>>(p, smem, stream);
    });
    if (dq != hipSuccess) return dq;
    if (hipError_t e = poly_by_part(p, [&](auto part) {
            constexpr int P = decltype(part)::value, smem = PolyPartOf<P>::PARTS ? PolyLds::kTotalTwo : PolyLds::kTotal;
            return p.denom ? launch_poly_kernel<poly_walk_dkdv_kernel<T, true, P>>(p, smem, stream)
                           : launch_poly_kernel<poly_walk_dkdv_kernel<T, false, P>>(p, smem, stream);
        }))
        return e;
    if (!p.vhalf || p.part > kPolyFirst) return hipSuccess;
    const int64_t total = (int64_t)(p.BH / 2) * p.N * (p.r / 8), blocks = (total + 255) / 256;
    if (blocks > 0x7fffffffLL) return hipErrorInvalidConfiguration;
    return launch_kernel<poly_add_halves_kernel<T>>(dim3((unsigned)blocks, 2), dim3(256), 0, stream, p, total);
}

inline hipError_t launch_poly_scan(float *totals, int64_t BH, int n_seg, int reverse, int part, hipStream_t stream) {
    const int state = part == kPolyCross ? PolyFeatures::kCross * 65 : PolyFeatures::kState;
    const int64_t total = BH * state;
    return launch_kernel<poly_scan_kernel<0>>(dim3((unsigned)((total + 255) / 256)), dim3(256), 0, stream, totals, n_seg, total,
                                              reverse, state);
}

}  // namespace fla
