// Chunk-wise evaluation of the polynomial score map, O = tril(f(Xq Xk^T)) V with f(u) = c0 + c1 u + c2 u^2, for rows of
// at most 16 columns over values of at most 64: the quadratic kernels' work grows with N^2, this one's with N.
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
    int32_t place;  // which workgroup takes which segment (xcd_place) and xcd_item's factor for n_seg, filled by the launcher
    uint32_t n_seg_inv;
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
    // dq (the exchange: sixteen floats a row)
    static constexpr int qQ = 0, qK = qQ + XT, qKt = qK + XT, qKb = qKt + XTR, qV = qKb + XTB, qG = qV + VT, qS = qG + VT, qEx = qS + ST,
                         qZ = qEx + C * 64, qDn = qZ + Z, qTotal = qDn + DN, qQt = qTotal, qTotalSums = qQt + XTR;
    // dk, dv
    static constexpr int kQ = 0, kQt = kQ + XT, kQb = kQt + XTR, kK = kQb + XTB, kV = kK + XT, kG = kV + VT, kU = kG + VT, kY = kU + ST,
                         kDn = kY + Z, kEx = kDn + DN, kTotal = kEx + EX;
    static_assert(XTR % 16 == 0 && tTotal >= 8 * 5 * 1024 && fTotal <= 160 * 1024 && qTotalSums <= 160 * 1024 && kTotal <= 160 * 1024, "a CU's LDS");
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

// A state's blocks of this wave: up to two blocks of 16 features (`first`, `second`, < 0: none) over the four 16-column blocks of
// the values, and -- NORM -- the column of ones (of dn), the same in every lane column.  Register v of a block: feature
// 4 (lane / 16) + v, value column lane % 16.
struct PolyState {
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
                if (NORM) ex[u] += *reinterpret_cast<const f32x4 *>(s + PolyFeatures::kF * PolyFeatures::kV + 16 * own[u] + 4 * kq);
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
                    const float *sf = s + (int64_t)(f0 + g < hi ? f0 + g : hi - 1) * PolyFeatures::kState;
#pragma unroll
                    for (int cb = 0; cb < 4; ++cb)
#pragma unroll
                        for (int v = 0; v < 4; ++v) t[g][cb][v] = sf[(16 * own[u] + 4 * kq + v) * PolyFeatures::kV + 16 * cb + l16];
                    if (NORM) e[g] = *reinterpret_cast<const f32x4 *>(sf + PolyFeatures::kF * PolyFeatures::kV + 16 * own[u] + 4 * kq);
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
                    *reinterpret_cast<f32x4 *>(s + PolyFeatures::kF * PolyFeatures::kV + 16 * own[u] + 4 * kq) = ex[u];
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
    // extra: the extra column, 128 floats in LDS that bf16 holds exactly (null: ones).
    // ONE: of the second block the 32 rows of step `step` alone.
    // (Rounded to one bf16 number, from a tile of feature rows, they and the weighted ones along the rows made the errors of
    // O, dq, dk and dv 1.2 times the quadratic kernels', and those of the normaliser 1e-3 in place of 1e-7.)
    template <bool NORM, bool ONE = false>
    __device__ __forceinline__ void update(const unsigned char *xtr, const unsigned char *zt, const float *extra, int lane, int step = 0) {
        const int l16 = lane & 15, kq = lane >> 4;
        const int row = 8 * kq + (l16 >> 2), ch = (l16 & 3) >> 1, sub = 8 * (l16 & 1);
        const PolyPair za{(uint32_t)(row * 128 + ((ch ^ walk_swizzle<8>(row)) << 4) + sub),
                          (uint32_t)((row + 4) * 128 + ((ch ^ walk_swizzle<8>(row + 4)) << 4) + sub)};
        const float *ex_at = extra ? extra + 8 * kq : nullptr;
        constexpr int STEPS = PolyLds::C / 32;
        auto block = [&](auto uc, auto steps, int first) {
            constexpr int U = decltype(uc)::value, NS = decltype(steps)::value;
            const PolyFactors at = poly_factors(16 * own[U] + l16);
            const unsigned char *fa = xtr + 32 * kq + at.a + 128 * first, *fb = xtr + 32 * kq + at.b + 128 * first;
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
    __device__ __forceinline__ void put(unsigned char *tile, float *dn, int tid) {
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
                // (rounded once for every use, as the quadratic evaluation's bias column holds it)
                if ((tid & 7) == 0) dn[(tid + 512 * i) >> 3] = static_cast<float>(static_cast<T>(-dot * inv));
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

// ---- sums of phi(k) [v, 1]^T (BWD: phi(q) [g, dn]^T) over every segment but the last (the first)
template <typename T, bool NORM, bool BWD>
__global__ __launch_bounds__(512, 2) void poly_totals_kernel(const PolyWalkParams p) {
#if defined(__gfx950__)
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    using L = PolyLds;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const PolySlice sl = poly_slice(p);
    if (!sl.valid || sl.seg == (BWD ? 0 : p.n_seg - 1)) return;
    const int b = sl.bh / p.H, h = sl.bh - b * p.H, N = p.N;
    const T *X = BWD ? static_cast<const T *>(p.q) + b * p.qs_b + h * p.qs_h : static_cast<const T *>(p.k) + b * p.ks_b + h * p.ks_h;
    const int64_t xs = BWD ? p.qs_n : p.ks_n;
    const T *V = static_cast<const T *>(p.v) + b * p.vs_b + h * p.vs_h;
    const T *G = BWD ? static_cast<const T *>(p.go) + b * p.gs_b + h * p.gs_h : nullptr;
    const T *O = BWD && NORM ? static_cast<const T *>(p.o) + b * p.os_b + h * p.os_h : nullptr;
    const float *n = NORM && BWD ? p.denom + (int64_t)sl.bh * N : nullptr;
    // Ten blocks of features on eight waves: a wave has one of its own and a quarter of the rows -- one step of every chunk --
    // of one of the last two, whose four parts are added up at the end (B H 64, N 4096: 21.4 -> 20.8 us forward, 29.7 -> 28.6
    // backward together with the second set of tiles; what is left is the chain load -> LDS -> features of two waves a SIMD)
    PolyState s;
    s.clear(wave, 8 + (wave >> 2));
    constexpr int SETS = 2;  // chunks on their way (registers and LDS)
    u32x4 x[SETS];
    PolyTile<T> v[SETS];
    PolyGrad<T, NORM> go[SETS];
    auto fetch = [&](int c, auto set) {
        constexpr int S = decltype(set)::value;
        const int row0 = c * L::C;
        if (tid < 256) x[S] = poly_fetch_x<T>(X, xs, row0, N, p.r, tid);
        if constexpr (BWD)
            go[S].fetch(G, p.gs_n, O, p.os_n, n, row0, N, p.wv, tid);
        else
            v[S].fetch(V, p.vs_n, row0, N, p.wv, tid);
    };
    static_for<0, SETS>([&](auto set) {
        if (sl.c_lo + decltype(set)::value < sl.c_hi) fetch(sl.c_lo + decltype(set)::value, set);
    });
    auto chunk = [&](int c, auto set) {
        constexpr int S = decltype(set)::value;
        unsigned char *tile = smem + S * L::tSet;
        float *dn = reinterpret_cast<float *>(tile + L::tDn);
        // (every wave has passed the barrier below a chunk ago, behind its reads of this set)
        if (tid < 256) poly_put_xt<T>(tile + L::tX, x[S], c * L::C, N, tid);
        if constexpr (BWD)
            go[S].put(tile + L::tV, dn, tid);
        else
            v[S].put(tile + L::tV, tid);
        if (c + SETS < sl.c_hi) fetch(c + SETS, set);
        __syncthreads();
        s.template update<NORM, true>(tile + L::tX, tile + L::tV, BWD ? dn : nullptr, lane, wave & 3);
    };
#pragma unroll 1
    for (int c = sl.c_lo; c < sl.c_hi; c += SETS)
        static_for<0, SETS>([&](auto set) {
            if (c + decltype(set)::value < sl.c_hi) chunk(c + decltype(set)::value, set);
        });
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
    s.template store<NORM>(p.totals + ((int64_t)sl.bh * p.n_seg + sl.seg) * PolyFeatures::kState, lane);
#else
    (void)p;
#endif
}

// entry states from totals, in place: entry[s] = sum over f < s (reverse: f > s); the loads of eight segments together
// (a template only so that the header can be included by several translation units)
template <int kUnused = 0>
__global__ __launch_bounds__(256) void poly_scan_kernel(float *totals, int n_seg, int64_t total, int reverse) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= total) return;
    const int64_t bh = i / PolyFeatures::kState, e = i - bh * PolyFeatures::kState;
    float *at = totals + (bh * n_seg + (reverse ? n_seg - 1 : 0)) * PolyFeatures::kState + e;
    const int64_t step = reverse ? -(int64_t)PolyFeatures::kState : (int64_t)PolyFeatures::kState;
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
template <bool NORM>
__device__ __forceinline__ void poly_entry(const PolyWalkParams &p, const PolySlice &sl, bool reverse, int lane, PolyState &s) {
    if (!p.totals) return;
    const float *base = p.totals + (int64_t)sl.bh * p.n_seg * PolyFeatures::kState;
    if (!p.sum_entries) {
        s.template add<NORM>(base + (int64_t)sl.seg * PolyFeatures::kState, lane);
        return;
    }
    s.template add_range<NORM>(base, reverse ? sl.seg + 1 : 0, reverse ? p.n_seg : sl.seg, lane);
}

template <typename T, bool NORM>
__global__ __launch_bounds__(512, 2) void poly_walk_fwd_kernel(const PolyWalkParams p) {
#if defined(__gfx950__)
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    using L = PolyLds;
    using M = Mma<T>;
    using V8 = typename M::V8;
    const int tid0 = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid0 >> 6), rb = wave & 3, kh = wave >> 2;
    const PolySlice sl = poly_slice(p);
    if (!sl.valid) return;
    const int b = sl.bh / p.H, h = sl.bh - b * p.H, N = p.N;
    const T *Q = static_cast<const T *>(p.q) + b * p.qs_b + h * p.qs_h;
    const T *K = static_cast<const T *>(p.k) + b * p.ks_b + h * p.ks_h;
    const T *V = static_cast<const T *>(p.v) + b * p.vs_b + h * p.vs_h;
    T *O = static_cast<T *>(p.out) + b * p.us_b + h * p.us_h;
    const float c0 = p.c0, c1 = p.c1, c2 = p.c2;
    unsigned char *tq = smem + L::fQ, *tk = smem + L::fK, *tkt = smem + L::fKt, *tv = smem + L::fV, *ts = smem + L::fS;
    float *z = reinterpret_cast<float *>(smem + L::fZ), *sums = reinterpret_cast<float *>(smem + L::fSum);
    unsigned char *exch = smem + L::fEx;
    PolyState s;
    s.clear_lower(wave);
    poly_entry<NORM>(p, sl, false, tid0 & 63, s);
    if (p.entries && sl.seg > 0)
        s.template store<NORM>(p.entries + ((int64_t)sl.bh * p.n_seg + sl.seg) * PolyFeatures::kStateRoom, tid0 & 63);
    u32x4 x;
    PolyTile<T> v;
    auto fetch = [&](int c, int tid) {
        const int row0 = c * L::C;
        x = tid < 256 ? poly_fetch_x<T>(Q, p.qs_n, row0, N, p.r, tid) : poly_fetch_x<T>(K, p.ks_n, row0, N, p.r, tid);
        v.fetch(V, p.vs_n, row0, N, p.wv, tid);
    };
    fetch(sl.c_lo, tid0);
#pragma unroll 1
    for (int c = sl.c_lo; c < sl.c_hi; ++c) {
        const int tid = poly_opaque(tid0), lane = tid & 63, l32 = lane & 31, g = lane >> 5;
        // (every wave is past the barrier behind its last reads of the tiles and of the state's copy)
        poly_put_x(tid < 256 ? tq : tk, x, tid);
        if (tid >= 256) poly_put_xt<T>(tkt, x, c * L::C, N, tid);
        v.put(tv, tid);
        s.template to_lds<T, NORM>(ts, z, lane);
        if (c + 1 < sl.c_hi) fetch(c + 1, tid);
        __syncthreads();

        const int trow = 32 * rb + l32, row = c * L::C + trow;
        f32x16 acc[2];
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[0][i] = acc[1][i] = 0.f;
        float rsum = 0.f;
        if (c > 0) {  // phi_w(q) T, this half of the features
            float xr[16];
            poly_row<T>(tq, trow, xr);
            const PolyTurned xt = poly_turn(xr, g, c2);
            const uint32_t sa = poly_row_base<256>(walk_e_lane(l32), g);
            auto step = [&](auto ksc) {
                constexpr int KS = decltype(ksc)::value;
                float raw[8];
                const PolyTwo f = poly_feature_frag<KS>(xt, g, c0, c1, raw);
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
            constexpr int H = PolyFeatures::kSteps / 2;
            if (kh == 0)
                static_for<0, H>(step);
            else
                static_for<H, 2 * H>(step);
        }
        const V8 xq = poly_row_frag<T>(tq, trow, g);
        const PolyPair va = poly_perm_base<128, false>(lane);
#pragma unroll 1
        for (int sb = kh; sb <= rb; sb += 2) {  // every other block of the chunk's scores
            // (the mask as bits, not a branch: see fla_tri_pair.h on scores and branches)
            const uint32_t all = sb < rb ? ~0u : 0u;
            f32x16 sc;
#pragma unroll
            for (int i = 0; i < 16; ++i) sc[i] = 0.f;
            sc = M::mma(poly_row_frag<T>(tk, 32 * sb + l32, g), xq, sc);
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
        if (c + 1 < sl.c_hi) s.template update<NORM>(tkt, tv, nullptr, lane);
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
            const float n = sums[trow] + sums[L::C + trow] + p.eps;
            inv = 1.0f / n;
            if (kh == 0 && g == 0 && row < N) p.denom[(int64_t)sl.bh * N + row] = n;
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) f[i] = (poly_pick(kh, acc[1][i], acc[0][i]) + other[i]) * inv;
        if (row < N) poly_store16<T>(O, (int64_t)row * p.us_n, f, 32 * kh + 16 * g, p.wv);
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

// dq: chunks ascending, T += phi(k) [v, 1]^T as in forward.  Each of the two waves of a row block takes a part of the feature
// blocks and every other score block.
template <typename T, bool NORM, bool SUMS>
__global__ __launch_bounds__(512, 2) void poly_walk_dq_kernel(const PolyWalkParams p) {
#if defined(__gfx950__)
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    using L = PolyLds;
    using M = Mma<T>;
    using V8 = typename M::V8;
    const int tid0 = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid0 >> 6), rb = wave & 3, kh = wave >> 2;
    const PolySlice sl = poly_slice(p);
    if (!sl.valid) return;
    const int b = sl.bh / p.H, h = sl.bh - b * p.H, N = p.N;
    const T *Q = static_cast<const T *>(p.q) + b * p.qs_b + h * p.qs_h;
    const T *K = static_cast<const T *>(p.k) + b * p.ks_b + h * p.ks_h;
    const T *V = static_cast<const T *>(p.v) + b * p.vs_b + h * p.vs_h;
    const T *G = static_cast<const T *>(p.go) + b * p.gs_b + h * p.gs_h;
    const T *O = NORM ? static_cast<const T *>(p.o) + b * p.os_b + h * p.os_h : nullptr;
    const float *den = NORM ? p.denom + (int64_t)sl.bh * N : nullptr;
    const int64_t dq_at = b * p.dqs_b + h * p.dqs_h;
    const float c1 = p.c1, c2 = p.c2;
    unsigned char *tq = smem + L::qQ, *tk = smem + L::qK, *tkt = smem + L::qKt, *tkb = smem + L::qKb, *tv = smem + L::qV, *tg = smem + L::qG,
                  *ts = smem + L::qS, *exch = smem + L::qEx;
    float *z = reinterpret_cast<float *>(smem + L::qZ), *dn = reinterpret_cast<float *>(smem + L::qDn);
    unsigned char *tqt = smem + L::qQt;
    PolyState s, sums;
    s.clear_lower(wave);
    if constexpr (SUMS) sums.clear_beside_lower(wave);
    const bool with_sums = SUMS && sl.seg > 0;  // (the first segment's total is under no sum)
    if (sl.seg > 0) s.template add<NORM>(p.entries + ((int64_t)sl.bh * p.n_seg + sl.seg) * PolyFeatures::kStateRoom, tid0 & 63);
    u32x4 x;
    PolyTile<T> v;
    PolyGrad<T, NORM> go;
    auto fetch = [&](int c, int tid) {
        const int row0 = c * L::C;
        x = tid < 256 ? poly_fetch_x<T>(Q, p.qs_n, row0, N, p.r, tid) : poly_fetch_x<T>(K, p.ks_n, row0, N, p.r, tid);
        v.fetch(V, p.vs_n, row0, N, p.wv, tid);
        go.fetch(G, p.gs_n, O, p.os_n, den, row0, N, p.wv, tid);
    };
    fetch(sl.c_lo, tid0);
#pragma unroll 1
    for (int c = sl.c_lo; c < sl.c_hi; ++c) {
        const int tid = poly_opaque(tid0), lane = tid & 63, l32 = lane & 31, g = lane >> 5;
        // (every wave is past the barrier behind its last reads of the tiles and of the state's copy)
        poly_put_x(tid < 256 ? tq : tk, x, tid);
        if (tid >= 256) {
            poly_put_xt<T>(tkt, x, c * L::C, N, tid), poly_put_xb(tkb, x, tid);
        } else if (with_sums) {
            poly_put_xt<T>(tqt, x, c * L::C, N, tid);
        }
        v.put(tv, tid);
        go.put(tg, dn, tid);
        s.template to_lds<T, NORM>(ts, z, lane);
        if (c + 1 < sl.c_hi) fetch(c + 1, tid);
        __syncthreads();

        const int trow = 32 * rb + l32, row = c * L::C + trow;
        const uint32_t ra = poly_row_base<128>(l32, g);
        V8 gf[4];
#pragma unroll
        for (int kc = 0; kc < 4; ++kc) gf[kc] = poly_rd<T>(tg + 32 * 128 * rb, ra ^ (kc << 5));
        const float dni = NORM ? dn[trow] : 0.f;
        float dxs[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) dxs[i] = 0.f;
        if (c > 0) {
            float xr[16];
            poly_row<T>(tq, trow, xr);
            if (kh == 0)
                poly_contract<T, NORM, 0, 2>(ts, z, dni, gf, xr, lane, c1, c2, dxs);
            else
                poly_contract<T, NORM, 2, PolyFeatures::kBlocks>(ts, z, dni, gf, xr, lane, c1, c2, dxs);
        }
        const V8 xq = poly_row_frag<T>(tq, trow, g);
        const int rc = walk_e_lane(l32) & 15;  // (columns 16 .. of the 32-wide block of dq are not used)
        f32x16 dx;
#pragma unroll
        for (int i = 0; i < 16; ++i) dx[i] = 0.f;
#pragma unroll 1
        for (int sb = kh; sb <= rb; sb += 2) {
            const uint32_t all = sb < rb ? ~0u : 0u;
            f32x16 m, u;
#pragma unroll
            for (int i = 0; i < 16; ++i) m[i] = dni, u[i] = 0.f;
            u = M::mma(poly_row_frag<T>(tk, 32 * sb + l32, g), xq, u);
#pragma unroll
            for (int kc = 0; kc < 4; ++kc) m = M::mma(poly_rd<T>(tv + 32 * 128 * sb, ra ^ (kc << 5)), gf[kc], m);
            V8 df[2];
            float d[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) d[i] = m[i] * (c1 + 2.f * c2 * u[i]);
            poly_round_masked<T, false>(d, all, l32, g, df);
#pragma unroll
            for (int t = 0; t < 2; ++t) dx = M::mma(poly_col_frag<T>(tkb, rc, 32 * sb + 16 * t, g), df[t], dx);
        }
        float f[16];  // (lanes of g = 0 hold the block's columns 0 .. 15)
#pragma unroll
        for (int i = 0; i < 16; ++i) f[i] = dxs[i] + __shfl_xor(dxs[i], 32, 64) + dx[i];
        if (kh == 1 && g == 0) {
#pragma unroll
            for (int a = 0; a < 4; ++a)
                *reinterpret_cast<f32x4 *>(exch + (a * L::C + trow) * 16) = f32x4{f[4 * a], f[4 * a + 1], f[4 * a + 2], f[4 * a + 3]};
        }
        if (c + 1 < sl.c_hi) s.template update<NORM>(tkt, tv, nullptr, lane);
        if constexpr (SUMS)
            if (with_sums) sums.template update<NORM>(tqt, tg, dn, lane);
        __syncthreads();
        if (kh == 0 && g == 0) {
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                const f32x4 t = *reinterpret_cast<const f32x4 *>(exch + (a * L::C + trow) * 16);
#pragma unroll
                for (int j = 0; j < 4; ++j) f[4 * a + j] += t[j];
            }
            if (row < N) poly_store16<T>(p.dq, dq_at + (int64_t)row * p.dqs_n, f, 0, p.r, p.wide_out);
        }
    }
    if constexpr (SUMS)
        if (with_sums) sums.template store<NORM>(p.totals + ((int64_t)sl.bh * p.n_seg + sl.seg) * PolyFeatures::kState, tid0 & 63);
#else
    (void)p;
#endif
}

// dk and dV: chunks descending, U += phi(q) [g, dn]^T
template <typename T, bool NORM>
__global__ __launch_bounds__(512, 2) void poly_walk_dkdv_kernel(const PolyWalkParams p) {
#if defined(__gfx950__)
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    using L = PolyLds;
    using M = Mma<T>;
    using V8 = typename M::V8;
    const int tid0 = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid0 >> 6), rb = wave & 3, half = wave >> 2;
    const PolySlice sl = poly_slice(p);
    if (!sl.valid) return;
    const int b = sl.bh / p.H, h = sl.bh - b * p.H, N = p.N;
    const T *Q = static_cast<const T *>(p.q) + b * p.qs_b + h * p.qs_h;
    const T *K = static_cast<const T *>(p.k) + b * p.ks_b + h * p.ks_h;
    const T *V = static_cast<const T *>(p.v) + b * p.vs_b + h * p.vs_h;
    const T *G = static_cast<const T *>(p.go) + b * p.gs_b + h * p.gs_h;
    const T *O = NORM ? static_cast<const T *>(p.o) + b * p.os_b + h * p.os_h : nullptr;
    const float *den = NORM ? p.denom + (int64_t)sl.bh * N : nullptr;
    const int64_t dk_at = b * p.dks_b + h * p.dks_h, dv_at = b * p.dvs_b + h * p.dvs_h;
    const float c0 = p.c0, c1 = p.c1, c2 = p.c2;
    unsigned char *tq = smem + L::kQ, *tqt = smem + L::kQt, *tqb = smem + L::kQb, *tk = smem + L::kK, *tv = smem + L::kV, *tg = smem + L::kG,
                  *us = smem + L::kU, *exch = smem + L::kEx;
    float *y = reinterpret_cast<float *>(smem + L::kY), *dn = reinterpret_cast<float *>(smem + L::kDn);
    PolyState su;
    su.clear_upper(wave);
    poly_entry<NORM>(p, sl, true, tid0 & 63, su);
    u32x4 x;
    PolyTile<T> v;
    PolyGrad<T, NORM> go;
    auto fetch = [&](int c, int tid) {
        const int row0 = c * L::C;
        x = tid < 256 ? poly_fetch_x<T>(Q, p.qs_n, row0, N, p.r, tid) : poly_fetch_x<T>(K, p.ks_n, row0, N, p.r, tid);
        v.fetch(V, p.vs_n, row0, N, p.wv, tid);
        go.fetch(G, p.gs_n, O, p.os_n, den, row0, N, p.wv, tid);
    };
    fetch(sl.c_hi - 1, tid0);
#pragma unroll 1
    for (int c = sl.c_hi - 1; c >= sl.c_lo; --c) {
        const int tid = poly_opaque(tid0), lane = tid & 63, l32 = lane & 31, g = lane >> 5;
        const bool after = c + 1 < p.n_chunks;  // (U of this chunk holds anything)
        // (every wave is past the barrier behind its last reads of the tiles and of the state's copy)
        poly_put_x(tid < 256 ? tq : tk, x, tid);
        if (tid < 256) poly_put_xt<T>(tqt, x, c * L::C, N, tid), poly_put_xb(tqb, x, tid);
        v.put(tv, tid);
        go.put(tg, dn, tid);
        if (after) su.template to_lds<T, NORM>(us, y, lane);
        if (c > sl.c_lo) fetch(c - 1, tid);
        __syncthreads();

        const int trow = 32 * rb + l32, row = c * L::C + trow;
        // dV: the waves of half 0 form phi_w(k) U, those of half 1 -- after dk -- the chunk's own part; each finishes one
        // half of the columns
        f32x16 acc[2];
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[0][i] = acc[1][i] = 0.f;
        if (half == 0) {
            if (after) {
                float xr[16];
                poly_row<T>(tk, trow, xr);
                const PolyTurned xt = poly_turn(xr, g, c2);
                const uint32_t sa = poly_row_base<256>(walk_e_lane(l32), g);
                static_for<0, PolyFeatures::kSteps>([&](auto ksc) {
                    constexpr int KS = decltype(ksc)::value;
                    float raw[8];
                    const PolyTwo f = poly_feature_frag<KS>(xt, g, c0, c1, raw);
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
            const uint32_t ra = poly_row_base<128>(l32, g);
            const int rc = walk_e_lane(l32) & 15;  // (columns 16 .. of the 32-wide block of dk are not used)
            const PolyPair ga = poly_perm_base<128, false>(lane);
            V8 vf[4];
#pragma unroll
            for (int kc = 0; kc < 4; ++kc) vf[kc] = poly_rd<T>(tv + 32 * 128 * rb, ra ^ (kc << 5));
            float dxs[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) dxs[i] = 0.f;
            if (after) {
                float xr[16];
                poly_row<T>(tk, trow, xr);
                poly_contract<T, NORM, 0, PolyFeatures::kBlocks>(us, y, 1.f, vf, xr, lane, c1, c2, dxs);
            }
            f32x16 dx;
#pragma unroll
            for (int i = 0; i < 16; ++i) dx[i] = 0.f;
#pragma unroll 1
            for (int sb = rb; sb < 4; ++sb) {
                const uint32_t all = sb > rb ? ~0u : 0u;
                f32x16 m, u;
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    f32x4 d = {0.f, 0.f, 0.f, 0.f};
                    if constexpr (NORM) d = *reinterpret_cast<const f32x4 *>(dn + 32 * sb + 8 * a + 4 * g);
#pragma unroll
                    for (int j = 0; j < 4; ++j) m[4 * a + j] = d[j], u[4 * a + j] = 0.f;
                }
                u = M::mma(poly_row_frag<T>(tq, 32 * sb + l32, g), xk, u);
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
                    dx = M::mma(poly_col_frag<T>(tqb, rc, 32 * sb + 16 * t, g), df[t], dx);
#pragma unroll
                    for (int e = 0; e < 2; ++e)
                        acc[e] = M::mma(poly_tr<T>(tg + 128 * (32 * sb + 16 * t), ga, e << 6), pf[t], acc[e]);
                }
            }
            float f[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) f[i] = dxs[i] + __shfl_xor(dxs[i], 32, 64) + dx[i];
            if (row < N && g == 0) poly_store16<T>(p.dk, dk_at + (int64_t)row * p.dks_n, f, 0, p.r, p.wide_out);
        }
        if (c > sl.c_lo) su.template update<NORM>(tqt, tg, dn, lane);
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
            for (int i = 0; i < 16; ++i) f[i] = poly_pick(half, acc[1][i], acc[0][i]) + other[i];
            if (row < N) poly_store16<T>(p.dv, dv_at + (int64_t)row * p.dvs_n, f, 32 * half + 16 * g, p.wv, p.wide_out);
        }
    }
#else
    (void)p;
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

template <typename T>
hipError_t launch_poly_totals(const PolyWalkParams &p, bool bwd, hipStream_t stream) {
    if (bwd)
        return p.denom ? launch_poly_kernel<poly_totals_kernel<T, true, true>>(p, PolyLds::tTotal, stream)
                       : launch_poly_kernel<poly_totals_kernel<T, false, true>>(p, PolyLds::tTotal, stream);
    return p.denom ? launch_poly_kernel<poly_totals_kernel<T, true, false>>(p, PolyLds::tTotal, stream)
                   : launch_poly_kernel<poly_totals_kernel<T, false, false>>(p, PolyLds::tTotal, stream);
}

template <typename T>
hipError_t launch_poly_walk(const PolyWalkParams &p, bool bwd, hipStream_t stream) {
    if (bwd) {
        if (p.n_seg > 1 && !p.entries) return hipErrorInvalidValue;
        if (p.u_totals && (!p.sum_entries || !p.totals || p.n_seg < 3)) return hipErrorInvalidValue;
        if (hipError_t e = p.u_totals ? (p.denom ? launch_poly_kernel<poly_walk_dq_kernel<T, true, true>>(p, PolyLds::qTotalSums, stream)
                                                 : launch_poly_kernel<poly_walk_dq_kernel<T, false, true>>(p, PolyLds::qTotalSums, stream))
                           : p.denom ? launch_poly_kernel<poly_walk_dq_kernel<T, true, false>>(p, PolyLds::qTotal, stream)
                                     : launch_poly_kernel<poly_walk_dq_kernel<T, false, false>>(p, PolyLds::qTotal, stream))
            return e;
        return p.denom ? launch_poly_kernel<poly_walk_dkdv_kernel<T, true>>(p, PolyLds::kTotal, stream)
                       : launch_poly_kernel<poly_walk_dkdv_kernel<T, false>>(p, PolyLds::kTotal, stream);
    }
    return p.denom ? launch_poly_kernel<poly_walk_fwd_kernel<T, true>>(p, PolyLds::fTotal, stream)
                   : launch_poly_kernel<poly_walk_fwd_kernel<T, false>>(p, PolyLds::fTotal, stream);
}

inline hipError_t launch_poly_scan(float *totals, int64_t BH, int n_seg, int reverse, hipStream_t stream) {
    const int64_t total = BH * PolyFeatures::kState;
    return launch_kernel<poly_scan_kernel<0>>(dim3((unsigned)((total + 255) / 256)), dim3(256), 0, stream, totals, n_seg, total,
                                              reverse);
}

}  // namespace fla
