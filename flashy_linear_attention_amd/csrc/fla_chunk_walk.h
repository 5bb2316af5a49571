// Chunk-wise causal linear attention with the running state kept inside the kernel, for equal
// padded head dims D = 32, 64 or 128 (shapes bound by memory traffic, not by the matrix units).
//
// The chunk-wise evaluation of fla_chunk_state.h / fla_tri_fast.h computes every per-chunk
// state, writes it in fp32, scans it, writes the running sums in 16 bit and reads them back in
// each consumer, and its backward reads q, k, v and dO once per product.  Here a workgroup walks
// a *segment* of consecutive chunks in sequence order and carries the running state
//
//     S = sum over the chunks before of K_c^T V_c      (forward, lower mask: ascending walk)
//     R = sum over the chunks after  of Q_c^T dO_c     (backward, upper mask: descending walk)
//
// in fp32 accumulators; per chunk it is rounded once to the storage type (as before) into LDS,
// where the MFMAs of the state products read it.  Every operand tile of a chunk is brought to
// LDS once and serves all products of that chunk:
//
//   forward   O_c  = lower(Q_c K_c^T) V_c   + Q_c S          then S += K_c^T V_c
//   backward  dQ_c = lower(dO_c V_c^T) K_c  + dO_c S_c^T
//             dV_c = upper(K_c Q_c^T) dO_c  + K_c R
//             dK_c = upper(V_c dO_c^T) Q_c  + V_c R^T        then R += Q_c^T dO_c
//
// Segments make the walk parallel: a first kernel adds up K^T V (Q^T dO) over segments, a small
// one turns the totals into each segment's entry state (exclusive prefix / suffix sums), and
// each walking workgroup starts from its segment's entry state.  No fp32 per-chunk state ever
// goes to memory.
//
//   D <= 64: 128-row chunks, two workgroups per CU.  ONE backward kernel (walk_bwd_kernel)
//            computes dQ, dV and dK of a chunk from one set of tiles; dQ's state -- the sum of
//            K^T V over the chunks BEFORE -- is the 16-bit copy that forward multiplied q by, saved at
//            the entry of every chunk (half the bytes of one operand at D = 64).  Nothing of a row
//            reaches the dQ of the chunks before it.
//   D = 128: tiles and state must share the 160 KiB of LDS: 64-row chunks, one workgroup per CU
//            with two sets of tiles (the next chunk's loads are in flight while this one is
//            multiplied).  A saved per-chunk state would cost as much traffic as an operand, so
//            forward hands over its segments' fp32 entry states and the state after the last chunk.
//            Backward is dQ as the forward walk over (dO, V, K), whose states V^T K start from the
//            transposed entry states, and walk_dkdv_kernel, the reverse walk for dV and dK -- or, for
//            callers that ask for it, ONE reverse walk (walk_bwd_rev_kernel) with dQ's state by
//            subtracting every chunk's K^T V from the state at the segment's end: 4 to 15 % less
//            backward time, but late rows that are infinite, NaN or huge spoil the dQ of earlier ones.
//
// Options of the walks: an element-wise feature map applied to q, k as they are loaded, with its
// slope multiplied into dQ, dK (WalkParams::fmap); the normaliser of linear attention and its
// gradient terms as rank-one additions to the products (WalkParams::denom ...); at D = 128,
// operands of at most 64 true columns on a side without the MFMAs on their padding (WalkExt).
//
// Scheduling.  With one wave per SIMD nothing hides the latency of an LDS read but the wave's own
// instruction order, and the compiler, short of registers, moves every operand read down to the
// MFMA that uses it.  The products therefore name their order themselves (walk_pipe: fragment
// j + 4 is read before fragment j is used, kept in place by scheduling barriers), the state
// product's MFMAs go between the score MFMAs of the first block (D = 128), running sums that only
// MFMAs touch live in accumulation registers (Mma::mma_acc), and code for feature maps is compiled
// only into the instantiations that use it.
//
// Layout.  An operand tile is C rows x D 16-bit values, row-major, the 16-byte chunk index of
// a row XORed with walk_swizzle(row) -- one layout, free of bank conflicts for the 16-byte row
// reads (MFMA operands with k along the row) and for the transposing column reads (k down the rows).  A wave
// owns one 32-row block of the chunk as the "X rows" of every product (and, at D = 128, one half
// of the output columns; the two waves of a row block then form the same scores); the MFMA
// operand chaining is that of the other kernels: S^T = Y X^T leaves a lane holding one X row
// and eight-row groups of Y rows, which is the B operand of Out^T += Z^T P^T.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "fla_launch.h"
#include "fla_tri_fast.h"

namespace fla {

// rows per chunk of the walk kernels: 128, or 64 at D = 128 (tiles and state must share the LDS)
constexpr int walk_rows(int D) { return D <= 64 ? 128 : 64; }

// a result's place: pointer, element strides, true width
struct WalkRowsOut {
    void *ptr;
    int64_t s_b, s_h, s_n;
    int32_t width;
};

struct WalkParams {
    const void *q, *k, *v, *go;  // operands (go: backward only); (B, H, N, D)
    void *o, *dq, *dk, *dv;      // results (forward: o; backward: dq, dk, dv)
    int64_t qs_b, qs_h, qs_n, ks_b, ks_h, ks_n, vs_b, vs_h, vs_n, gs_b, gs_h, gs_n;
    int64_t os_b, os_h, os_n, dqs_b, dqs_h, dqs_n, dks_b, dks_h, dks_n, dvs_b, dvs_h, dvs_n;
    int32_t H, N, BH, wqk, wv;   // true widths of q/k and of v (<= D)
    int32_t n_chunks;            // ceil(N / rows per chunk)
    int32_t seg_chunks, n_seg;   // chunks per segment, segments per (b, h)
    // entry state of every segment, fp32 [BH][n_seg][D (q/k index)][D (v index)]: sum of K^T V over
    // the segments before (forward) / of Q^T dO over the segments after (backward); null when
    // there is a single segment (entry state zero).  init_transposed: the buffer holds the
    // transposed matrices ([v index][q/k index]).
    const float *init;
    int32_t init_transposed;
    // forward, D <= 64: where the 16-bit state at the entry of every chunk goes, [BH][n_chunks][D][D], or null; backward:
    // the same buffer, read for dQ.  Laid out as its copy in LDS (unscaled).
    void *saved;
    // Feature map (fla_feature.h), 0: none.  Forward: q holds the argument xq of the map phi; the Q
    // tile is mapped in LDS as it lands and phi(xq) is written to qmap_out (q's shape, element
    // strides qo_*); k already holds phi(xk) (written by the totals kernel).  Backward: q and k
    // hold phi(xq), phi(xk), and dQ, dK are multiplied by the slope of phi, computed from those
    // values in the LDS tiles, before they are rounded and stored.
    int32_t fmap;
    void *qmap_out;
    int64_t qo_b, qo_h, qo_n;
    // walk_fwd_kernel run as the dQ walk of the split backward (q <- dO, k <- V, v <- K, o <- dQ) with
    // a feature map: slope_y holds phi(xq) (o's shape, element strides sy_*) and the result is
    // multiplied by the slope of phi computed from it; null: none.
    const void *slope_y;
    int64_t sy_b, sy_h, sy_n;
    // The normaliser n_i = q_i . (k_0 + ... + k_i) + eps fused into the walks (null pointers: off).
    // Forward (denom): n_i = sum of row i's masked scores + q_i . zc_c, with zc_c carried by the walk beside the
    // state (walk_col_sums; vsum: the segments' totals of k from the totals kernel, null with a single segment) and
    // written to zc_out (null: nowhere) for backward; the result is divided by n_i and n goes to denom.  Backward, with
    // dn_i = -(g_i . out_i) / n_i and dO = g / n from walk_grad_totals_kernel: dQ's scores get + dn_i and its result
    // + dn_i zc_c (dn, zc); dK's scores get + dn_i (i: the dO row) and its result + rc_c, the sum of dn_i q_i over the rows
    // after chunk c, carried by the walk beside R (rc: the segments' totals of dn_i q_i, null with a single one).
    float *denom;     // fp32 [BH][N]
    float eps;
    const float *zc;  // fp32 [BH][n_chunks][D]: sum of k over the rows before chunk c (backward)
    const float *vsum;  // fp32 [BH][n_seg][D], slots as those of `init` (two segments: partial sums in both)
    float *zc_out;      // as zc
    const float *dn;  // fp32 [BH][N]
    const float *rc;  // fp32 [BH][n_seg][D], slots as those of `init`
    // fp16 without the normaliser, up to 64 columns: what each of the saved copies is to be multiplied by, [BH][n_chunks] (walk_state_scale, 1
    // with a feature map on load; null: they were multiplied by it)
    float *saved_scale;
    // walk_bwd_kernel: go holds g, and dO = g / n is formed in its tile as it lands (null: go holds dO).  An operand less for
    // walk_grad_totals_kernel to write: B H 64, N 4096, D 64 that kernel 24.8 -> 19.4 us, the walk 57.3 to 59.9 (55.2 from 54.4 without a
    // feature map); forward + backward with a feature map 151 -> 145, B H 128 283 -> 274, without one B H 512, N 1024 228 -> 221
    const float *gn;  // n, fp32 [BH][N]
    // Forward, D = 128: where the state after the last chunk of every (b, h) goes, fp32 [BH][D][D]
    // ([q/k index][v index]), or null.  walk_bwd_rev_kernel: that buffer (xtotal) and forward's entry
    // states (xinit, the layout of `init`, not transposed; may be null with a single segment).
    float *total_out;
    const float *xinit, *xtotal;
    // The wide walks (walk_fwd_wide_kernel, walk_bwd_rev_wide_kernel): q and k (dq and dk) have 129 .. 256
    // columns.  Columns 128 .. are the second half, of true width wqk2 (wqk = 128 is the first half's), with
    // entry and final states of its own in the layouts of init, total_out, xinit and xtotal.
    int32_t wqk2;
    const float *init2;
    float *total_out2;
    const float *xinit2, *xtotal2;
    // init_is_totals (every D = 128 walk; three segments or more): init (and init2) hold the segments' TOTALS as the
    // totals kernel wrote them, and a workgroup adds up those of the segments before its own (after it, walking in
    // reverse) as it starts, several loads in flight together -- no scan launch between the totals kernel and the
    // walk.  The forward walks (walk_fwd_kernel at D = 128, walk_fwd_wide_kernel) then write the entry
    // state they formed to entry_out / entry_out2 (the layout of init; null: nowhere), for the backward walk.
    int32_t init_is_totals;
    float *entry_out, *entry_out2;
    // walk_fwd_kernel as dQ's walk and the backward walks (but quad, and v wider than 64 beside a wide q / k), bf16: the results
    // are stored in fp32 (o / dq, dk, dv then
    // point to floats; what is stored is rounded to bf16 as always).  Kernels of their own (WIDE): as a branch in front of the
    // stores it cost the others up to 3 %
    int32_t wide_out;
    // walk_fwd_kernel (D = 128), walk_dkdv_kernel and walk_bwd_rev_kernel, plain, and walk_bwd_rev_wide_kernel with v of at most 64
    // columns and without dQ (dk alone): the results go to rows of any alignment and width (WalkAnyRows), in place of o, dq, dk
    // and dv.  Kernels of their own (ROWS)
    int32_t any_rows;
    WalkRowsOut rows_o, rows_dq, rows_dk, rows_dv;
    // walk_fwd_kernel as dQ's walk (D = 128, bf16, plain, q and k above 64 columns; kernels of their own: RSUM), three segments or more:
    // beside dQ it adds up its segment's total of Q^T dO for the reverse walk -- dO is in LDS already -- and writes it to r_totals,
    // as walk_totals_kernel would (r_frags: by fragments).  Null: not.  Forward + backward, a totals kernel in front -> this: D 128, B H
    // 32, N 2048 83.0 -> 78.9 us; B H 64, N 4096 223.8 -> 213.7; B H 16, N 20000 295 -> 287; D 80, B H 24, N 1500 59.9 -> 57.6.  With two
    // segments, where half of the workgroups have that work, B H 128, N 4096 422 -> 418, N 1024 111 -> 113
    const void *r_q;
    int64_t rs_b, rs_h, rs_n;
    int32_t r_frags;
    float *r_totals;
    // A v of 129 .. 256 columns beside a wide q / k (1; 0: none): its columns 128 .. are a second half of true width wv2, and grid y
    // picks a part of the work: the half of v (walk_fwd_wide_kernel); the half of dV, or of dK (walk_rev_wide_kernel).
    // The states of (q / k half i, v half j) are matrices (2 j + i) BH .. of every state buffer.
    int32_t quad, wv2;
    // D = 128, plain, both sides above 64 columns, one segment per (b, h): two workgroups per (b, h) in place of two segments
    // (grid y), so that no totals come before the walk.  cols (walk_fwd_kernel; kernels of their own: COLS): grid y takes columns
    // 64 y .. of v and of the result; q and k are read by both, within one XCD, at the same time.  The state at the entry of chunk
    // mid_chunk goes to mid_out (null: nowhere) in the form of two segments' partial sums, total_out as always.  roles
    // (walk_dkdv_kernel, ROLES): dV is formed by grid y = 0, dK by 1, each with a copy of R; q and dO are read by both.
    int32_t cols, roles, mid_chunk;
    float *mid_out;
    int32_t place;       // which workgroup takes which segment (walk_place) and xcd_item's factor for n_seg, both filled on the way to the
    uint32_t n_seg_inv;  // launcher; here and below
};

template <int D>
struct WalkCfg {
    static constexpr int C = walk_rows(D);  // rows per chunk
    static constexpr int RB = D * 2;        // bytes per tile row
    static constexpr int CR = D / 8;        // 16-byte chunks per row
    static constexpr int TILE = C * RB;     // bytes per operand tile
    static constexpr int KC = D / 16;       // 16-wide k chunks of a contraction over D
    static constexpr int DB = D / 32;       // 32-wide blocks of D
    static constexpr int RPI = 1024 / RB;   // rows covered by one wave-level 1 KiB load
    static constexpr int NI = TILE / 4096;  // such loads per wave and tile
    static constexpr int STATE = D * RB;    // the 16-bit state in LDS
    static constexpr int VEC = 3 * 1024;    // per set of tiles: zc, rc (walk_bwd_kernel), dn of the chunk (fp32, 1 KiB each)
    static constexpr int NID = C / 64;      // wave-level 256-byte loads of a chunk's dn
    static constexpr int NBLK = DB * DB;    // 32 x 32 blocks of the state: block b belongs to wave b % 4
    static constexpr int NBW = (NBLK + 3) / 4;  // state blocks per wave
    // a wave owns one 32-row block of the chunk as the X rows of every product, and -- with fewer
    // than four such blocks -- one part of the output columns
    static constexpr int NRB = C / 32;      // row blocks per chunk
    static constexpr int NCH = 4 / NRB;     // column parts
    static constexpr int DBW = DB / NCH;    // 32-wide output blocks per wave
    static_assert(D == 32 || D == 64 || D == 128, "walk kernels are built for padded head dims 32, 64 and 128");
    static_assert(NRB * NCH == 4 && DBW * NCH == DB, "four waves tile the chunk's rows and output columns");
};

// The 32 x 32 blocks of the state that hold anything: NQ blocks of q/k indices (its rows), NV of v
// indices (its columns).  All D / 32 of each by default; the D = 128 kernels are also built for
// operands of at most 64 true columns on one side (NQ or NV = 2: the other blocks would hold the
// zeros the tiles are padded with, and the MFMAs on them are left out).
// State block i of wave `wave` is block wave + 4 i of the NQ x NV: (dbk, eb) = (block of q/k
// indices, block of v indices); the v block is the same for all blocks of a wave.
template <int D, int NQ = D / 32, int NV = D / 32>
struct WalkExt {
    static_assert(NQ >= 1 && NQ <= D / 32 && NV >= 1 && NV <= D / 32 && (4 % NV == 0 || NV % 4 == 0), "block counts");
    static constexpr int nq = NQ, nv = NV;
    static constexpr int SLOTS = (NQ * NV + 3) / 4;  // state blocks per wave
    static constexpr int KQ = 2 * NQ, KV = 2 * NV;   // 16-wide k chunks over the q/k side, the v side
    // (with a multiple of four blocks every slot of every wave holds one: known at compile time)
    __device__ static __forceinline__ bool valid(int wave, int i) { return (NQ * NV) % 4 == 0 || wave + 4 * i < NQ * NV; }
    __device__ static __forceinline__ int dbk(int wave, int i) { return (wave + 4 * i) / NV; }
    __device__ static __forceinline__ int eb(int wave) { return wave % NV; }
};

// Output blocks of a product whose result has NOB blocks that hold anything: with two column parts
// (D = 128) each part takes half of them -- PER blocks from block db0(wave).
template <int D, int NOB>
struct WalkOut {
    using W = WalkCfg<D>;
    static_assert(NOB % W::NCH == 0, "the column parts share the output blocks evenly");
    static constexpr int PER = NOB / W::NCH;
    __device__ static __forceinline__ int db0(int wave) { return W::NCH == 1 ? 0 : (wave / W::NRB) * PER; }
};

// ---- LDS tile access (tile: row-major [rows][D], chunk index XOR walk_swizzle(row))

// XOR applied to the 16-byte chunk index of tile row `row`.  Every tile is read both ways:
//   * along its rows (walk_row_frag): 16 lanes read the same chunk index of 16 consecutive rows,
//     which must land in the 16 different 16-byte slots of the 256 bytes that 64 banks span;
//   * down its columns (walk_col_frag*, transposing 8-byte reads): 32 lanes read 64 consecutive
//     bytes of each of 4 consecutive rows, which must land in 4 different 64-byte quarters.
// With 256-byte rows (D = 128) the row's low four bits go into the chunk index with its low two
// bits on top -- the bits that pick the 64-byte quarter -- and with 128-byte rows (D = 64, where
// the row's lowest bit already picks a half) bits 1 .. 3, bit 1 on top.  (Folding the bits in
// unpermuted serves the row reads just as well, but the 4 rows of a column read then meet in the
// same quarter: a 4-way bank conflict at D = 128, 2-way at D = 64.)
template <int CR>
__device__ __forceinline__ int walk_swizzle(int row) {
    if constexpr (CR == 4) {
        return (row >> 2) & 3;  // (64-byte rows: the 4 rows of a column read are the 4 quarters)
    } else if constexpr (CR == 8) {
        const int t = (row >> 1) & 7;
        return ((t & 1) << 2) | (t >> 1);
    } else {
        const int t = row & 15;
        return ((t & 3) << 2) | (t >> 2);
    }
}

// whole 128-row tile HBM -> LDS; rows >= N and chunks beyond the true width arrive as zeros
template <int D>
__device__ __forceinline__ void walk_load_tile(u32x4 rsrc, uint32_t lds_tile, int row0, int stride2, int width, int wave,
                                               int lane) {
    using W = WalkCfg<D>;
    const int r = wave * W::RPI + lane / W::CR;
    const int c = (lane % W::CR) ^ walk_swizzle<W::CR>(r);
    const uint32_t voff = (uint32_t)(r * stride2 + c * 16) + (c * 8 < width ? 0u : kOobOffset);
    const uint32_t base = (uint32_t)__builtin_amdgcn_readfirstlane((int)(lds_tile + wave * 1024));
    u32x4 rs = {(uint32_t)__builtin_amdgcn_readfirstlane((int)rsrc[0]), (uint32_t)__builtin_amdgcn_readfirstlane((int)rsrc[1]),
                (uint32_t)__builtin_amdgcn_readfirstlane((int)rsrc[2]), (uint32_t)__builtin_amdgcn_readfirstlane((int)rsrc[3])};
    static_for<0, W::NI>([&](auto u) {
        constexpr int U = decltype(u)::value;
        const uint32_t so = (uint32_t)__builtin_amdgcn_readfirstlane((row0 + U * 4 * W::RPI) * stride2);
        dma_16B_per_lane<U * 4096>(rs, base, voff, so);
    });
}

// eight consecutive columns 16 kc + 8 g .. of one row: an MFMA operand with k along the row
template <typename T, int D>
__device__ __forceinline__ typename Mma<T>::V8 walk_row_frag(const unsigned char *tile, int row, int kc, int g) {
    using W = WalkCfg<D>;
    const int ch = (2 * kc + g) ^ walk_swizzle<W::CR>(row);
    return __builtin_bit_cast(typename Mma<T>::V8, *reinterpret_cast<const u32x4 *>(tile + row * W::RB + (ch << 4)));
}

__device__ __forceinline__ s16x4 walk_tr_read(const unsigned char *p) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(p));
}

// Column fragment with the output-column permutation of the product kernels: rows R0 + {4g .. 4g+3,
// 8+4g .. 8+4g+3} (the k order of a rounded S^T accumulator) of the 32 columns of block cb, taken
// so that MFMA row m = 8a + 4g' + b holds column 16g' + 4a + b -- a lane's 16 accumulator registers
// are then 16 consecutive output columns.  With `consecutive` the rows are R0 + 8g .. 8g+7 instead
// (the k order of a row fragment): the transposed read of the state.
template <typename T, int D>
__device__ __forceinline__ typename Mma<T>::V8 walk_col_frag_perm(const unsigned char *tile, int R0, int cb, int lane,
                                                                  bool consecutive) {
    using W = WalkCfg<D>;
    const int lam = lane & 15, g = lane >> 5, beta = (lane >> 4) & 1, zc = lam & 3;
    const int row_lo = R0 + (consecutive ? 8 * g : 4 * g) + (lam >> 2), row_hi = row_lo + (consecutive ? 4 : 8);
    const int ch = 4 * cb + 2 * (zc & 1) + beta, byte = 8 * (zc >> 1);
    const s16x4 lo = walk_tr_read(tile + row_lo * W::RB + ((ch ^ walk_swizzle<W::CR>(row_lo)) << 4) + byte);
    const s16x4 hi = walk_tr_read(tile + row_hi * W::RB + ((ch ^ walk_swizzle<W::CR>(row_hi)) << 4) + byte);
    return __builtin_bit_cast(typename Mma<T>::V8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

// Column fragment, plain mapping (lane l32 <-> column 32 cb + l32), rows R0 + {4g.., 8+4g..}: both
// operands of the state update Y^T Z, whose contraction runs down the rows.
template <typename T, int D>
__device__ __forceinline__ typename Mma<T>::V8 walk_col_frag(const unsigned char *tile, int R0, int cb, int lane) {
    using W = WalkCfg<D>;
    const int lam = lane & 15, g = lane >> 5, beta = (lane >> 4) & 1;
    const int row_lo = R0 + 4 * g + (lam >> 2), row_hi = row_lo + 8;
    const int ch = 4 * cb + 2 * beta + ((lam & 3) >> 1), sub = 8 * (lam & 1);
    const s16x4 lo = walk_tr_read(tile + row_lo * W::RB + ((ch ^ walk_swizzle<W::CR>(row_lo)) << 4) + sub);
    const s16x4 hi = walk_tr_read(tile + row_hi * W::RB + ((ch ^ walk_swizzle<W::CR>(row_hi)) << 4) + sub);
    return __builtin_bit_cast(typename Mma<T>::V8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

// MFMA row m of a state-product A operand holds output column e_lane(m) of its 32-column block
// (the permutation of walk_col_frag_perm)
__device__ __forceinline__ int walk_e_lane(int l32) { return 16 * ((l32 >> 2) & 1) + 4 * (l32 >> 3) + (l32 & 3); }

// ---- small fp32 vectors of a chunk HBM -> LDS (every wave issues them, to the same place)
template <int LDS_IMM>
__device__ __forceinline__ void dma_4B_per_lane(u32x4 rsrc, uint32_t lds_base, uint32_t voffset, uint32_t soffset) {
    asm volatile("s_add_u32 m0, %0, %4\n\ts_nop 0\n\tbuffer_load_dword %1, %2, %3 offen lds"
                 :
                 : "s"(lds_base), "v"(voffset), "s"(rsrc), "s"(soffset), "n"(LDS_IMM)
                 : "memory", "m0", "scc");
}
__device__ __forceinline__ u32x4 walk_uniform_rsrc(const void *base, uint32_t bytes) {
    const u32x4 r = make_rsrc(base, bytes);
    return u32x4{(uint32_t)__builtin_amdgcn_readfirstlane((int)r[0]), (uint32_t)__builtin_amdgcn_readfirstlane((int)r[1]),
                 (uint32_t)__builtin_amdgcn_readfirstlane((int)r[2]), (uint32_t)__builtin_amdgcn_readfirstlane((int)r[3])};
}
// D floats (16-byte aligned) to lds_dst: one load, lanes beyond D / 4 write zeros (1 KiB is written)
template <int D>
__device__ __forceinline__ void walk_load_vec(const float *src, uint32_t lds_dst, int lane) {
    dma_16B_per_lane<0>(walk_uniform_rsrc(src, D * 4), (uint32_t)__builtin_amdgcn_readfirstlane((int)lds_dst),
                        (uint32_t)lane * 16, 0);
}
// rows row0 .. row0 + C - 1 of a vector of N floats (zeros past the end) to lds_dst
template <int D>
__device__ __forceinline__ void walk_load_rows(const float *vec, int row0, int N, uint32_t lds_dst, int lane) {
    const u32x4 rs = walk_uniform_rsrc(vec + row0, (uint32_t)(N - row0) * 4);
    const uint32_t base = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds_dst);
    static_for<0, WalkCfg<D>::NID>([&](auto u) {
        constexpr int U = decltype(u)::value;
        dma_4B_per_lane<U * 256>(rs, base, (uint32_t)lane * 4 + U * 256, 0);
    });
}

// acc[i][v] += scale * vec[32 (db0 + i) + 16 g + v] (vec: fp32 in LDS)
template <int D>
__device__ __forceinline__ void walk_add_vec(f32x16 (&acc)[WalkCfg<D>::DBW], float scale, const float *vec, int db0, int g) {
    typedef float f32x4 __attribute__((ext_vector_type(4)));  // (declared again below, for the products)
#pragma unroll
    for (int i = 0; i < WalkCfg<D>::DBW; ++i)
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const f32x4 z = *reinterpret_cast<const f32x4 *>(vec + 32 * (db0 + i) + 16 * g + 4 * a);
#pragma unroll
            for (int b = 0; b < 4; ++b) acc[i][4 * a + b] += scale * z[b];
        }
}

// ---- one product of a chunk for this wave's 32 X rows (row block rb = wave % NRB) and its part of
// the output columns (blocks db0 .. db0 + DBW - 1, db0 = (wave / NRB) * DBW):
//   acc = [state: X_w . State]  +  mask(X_w Y^T) Z        (UPPER: keep row <= column, else row >= column)
// xt, yt, zt: LDS tiles; sfrag(db, kc): the state's A-operand fragment for output block db, k chunk kc.
// (With several column parts the waves of one row block each compute the same scores.)
// EX (the normaliser's terms): 1: ex = sum of this row's masked scores + x_row . exv (exv: D floats in
// LDS); 2: every score gets + ex (a value per X row, i.e. per lane) before the mask; 3: every
// score gets + exv[its Y row] (exv: one float per tile row, in LDS).
typedef float f32x4 __attribute__((ext_vector_type(4)));
struct WalkNoRows {
    __device__ __forceinline__ f32x4 operator()(int, int) const { return f32x4{0.f, 0.f, 0.f, 0.f}; }
};
// N operand fragments read from LDS and consumed in order, the read of fragment j + DEPTH issued
// before fragment j is used: use(j, fragment) for j = 0 .. N-1 with read(j + DEPTH) ahead of it.  The
// scheduling barriers keep the compiler from moving a read down to its use again (which it does when
// registers are scarce, and every MFMA then waits out the whole latency of its own LDS read).
template <int N, int DEPTH, typename V8, typename Read, typename Use>
__device__ __forceinline__ void walk_pipe(Read &&read, Use &&use) {
    V8 buf[N];
    static_for<0, (DEPTH < N ? DEPTH : N)>([&](auto j) { buf[decltype(j)::value] = read(j); });
    static_for<0, N>([&](auto j) {
        constexpr int J = decltype(j)::value;
        if constexpr (J + DEPTH < N) buf[J + DEPTH] = read(std::integral_constant<int, J + DEPTH>{});
        __builtin_amdgcn_sched_barrier(0);
        use(j, buf[J]);
    });
    __builtin_amdgcn_sched_barrier(0);
}

// KCL: 16-wide k chunks of the contraction X Y^T that hold anything; NOB: output blocks that do.
// KEEP: the product is added to what acc holds.  SCALED: the state's part is multiplied by sback (walk_state_scale).
template <typename T, int D, bool UPPER, int EX = 0, int KCL = WalkCfg<D>::KC, int NOB = WalkCfg<D>::DB, bool KEEP = false,
          bool SCALED = false, typename SFrag, typename YRows = WalkNoRows>
__device__ __forceinline__ void walk_product(const unsigned char *xt, const unsigned char *yt, const unsigned char *zt,
                                             int wave, int lane, bool has_state, SFrag &&sfrag,
                                             f32x16 (&acc)[WalkCfg<D>::DBW], float *ex = nullptr,
                                             const float *exv = nullptr, YRows &&yrows = WalkNoRows{}, float sback = 1.f) {
    static_assert(!SCALED || !KEEP, "what acc held would be scaled too");
    using W = WalkCfg<D>;
    using M = Mma<T>;
    using V8 = typename M::V8;
    constexpr int PER = WalkOut<D, NOB>::PER;
    const int l32 = lane & 31, g = lane >> 5;
    const int rb = W::NCH == 1 ? wave : wave % W::NRB, db0 = WalkOut<D, NOB>::db0(wave);
    V8 xf[KCL];
#pragma unroll
    for (int kc = 0; kc < KCL; ++kc) xf[kc] = walk_row_frag<T, D>(xt, 32 * rb + l32, kc, g);
    float rsum = 0.f;
    if constexpr (EX == 1) {
#pragma unroll
        for (int kc = 0; kc < KCL; ++kc)
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                const f32x4 z = *reinterpret_cast<const f32x4 *>(exv + 16 * kc + 8 * g + 4 * a);
#pragma unroll
                for (int b = 0; b < 4; ++b) rsum += static_cast<float>(xf[kc][4 * a + b]) * z[b];
            }
    }
    if constexpr (!KEEP) {
#pragma unroll
        for (int i = 0; i < W::DBW; ++i)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][v] = 0.f;
    }
    // One 32-row block s of Y and Z: scores, mask and rounding, second product.  ST: the state product's
    // MFMAs are issued in between -- PER / 2 of them after every score MFMA (they share its X fragment
    // and fill the gaps of the dependent chain), the rest after the last one, where the rounding of the
    // scores runs beneath them.  Operand fragments are read four ahead, in the order of their use.
    auto block = [&](int s, auto with_state) {
        constexpr bool ST = decltype(with_state)::value;
        constexpr int H = ST ? PER / 2 : 0, GA = 1 + H, GB = PER - H;
        constexpr int NA = KCL * GA, NB = ST ? GB * KCL : 0, NC = 2 * PER;
        constexpr int CONV = NB > 2 ? NA + 2 : NA + NB;  // the scores are finished in front of this operation
        f32x16 sc;
#pragma unroll
        for (int v = 0; v < 16; ++v) sc[v] = 0.f;
        V8 pf[2];
        walk_pipe<NA + NB + NC, 4, V8>(
            [&](auto j) {
                constexpr int J = decltype(j)::value;
                if constexpr (J < NA) {
                    if constexpr (J % GA == 0)
                        return walk_row_frag<T, D>(yt, 32 * s + l32, J / GA, g);
                    else
                        return sfrag(db0 + J % GA - 1, J / GA);
                } else if constexpr (J < NA + NB) {
                    return sfrag(db0 + H + (J - NA) % GB, (J - NA) / GB);
                } else {
                    return walk_col_frag_perm<T, D>(zt, 32 * s + 16 * ((J - NA - NB) / PER), db0 + (J - NA - NB) % PER, lane,
                                                    false);
                }
            },
            [&](auto j, V8 f) {
                constexpr int J = decltype(j)::value;
                if constexpr (SCALED && ST && J == NA + NB) {  // (the state product is complete)
#pragma unroll
                    for (int i = 0; i < PER; ++i)
#pragma unroll
                        for (int v = 0; v < 16; ++v) acc[i][v] *= sback;
                }
                if constexpr (J == CONV) {  // normaliser's terms, mask, rounding
                    if constexpr (EX == 2) {
#pragma unroll
                        for (int v = 0; v < 16; ++v) sc[v] += *ex;
                    }
                    if constexpr (EX == 3) {
#pragma unroll
                        for (int a = 0; a < 4; ++a) {
                            const f32x4 y = yrows(s, a);
#pragma unroll
                            for (int b = 0; b < 4; ++b) sc[4 * a + b] += y[b];
                        }
                    }
                    if (s == rb) {  // the 32 x 32 block on the diagonal: lane = X row l32, register v = Y row jl
#pragma unroll
                        for (int v = 0; v < 16; ++v) {
                            const int jl = 8 * (v / 4) + 4 * g + (v % 4);
                            const bool keep = UPPER ? l32 <= jl : l32 >= jl;
                            sc[v] = keep ? sc[v] : 0.f;
                        }
                    }
                    if constexpr (EX == 1) {
#pragma unroll
                        for (int v = 0; v < 16; ++v) rsum += sc[v];
                    }
#pragma unroll
                    for (int t = 0; t < 2; ++t)
#pragma unroll
                        for (int e = 0; e < 8; ++e) pf[t][e] = static_cast<T>(sc[8 * t + e]);
                }
                if constexpr (J < NA) {
                    if constexpr (J % GA == 0)
                        sc = M::mma(f, xf[J / GA], sc);
                    else
                        acc[J % GA - 1] = M::mma(f, xf[J / GA], acc[J % GA - 1]);
                } else if constexpr (J < NA + NB) {
                    acc[H + (J - NA) % GB] = M::mma(f, xf[(J - NA) / GB], acc[H + (J - NA) % GB]);
                } else {
                    acc[(J - NA - NB) % PER] = M::mma(f, pf[(J - NA - NB) / PER], acc[(J - NA - NB) % PER]);
                }
            });
    };
    const int s_lo = UPPER ? rb : 0, s_hi = UPPER ? W::NRB - 1 : rb;
    if constexpr (D == 128) {
        if (has_state)
            block(s_lo, std::true_type{});
        else
            block(s_lo, std::false_type{});
#pragma unroll 1
        for (int s = s_lo + 1; s <= s_hi; ++s) block(s, std::false_type{});
    } else {
        // (two workgroups per CU cover each other's gaps, and the fused backward has no registers to
        // spare for the longer pipeline: the state product on its own, k chunk outer, output block inner)
        if (has_state) {
            walk_pipe<PER * KCL, 4, V8>([&](auto j) { return sfrag(db0 + decltype(j)::value % PER, decltype(j)::value / PER); },
                                        [&](auto j, V8 f) {
                                            constexpr int I = decltype(j)::value % PER, KC_ = decltype(j)::value / PER;
                                            acc[I] = M::mma(f, xf[KC_], acc[I]);
                                        });
            if constexpr (SCALED) {
#pragma unroll
                for (int i = 0; i < PER; ++i)
#pragma unroll
                    for (int v = 0; v < 16; ++v) acc[i][v] *= sback;
            }
        }
#pragma unroll 1
        for (int s = s_lo; s <= s_hi; ++s) block(s, std::false_type{});
    }
    if constexpr (EX == 1) *ex = rsum + __shfl_xor(rsum, 32, 64);  // the two lanes of a row hold half the columns each
}

// Every element of the landed tile replaced by phi(element), in place, and the mapped rows written
// to `out` (rows >= N and chunks beyond the true width arrived as zeros and stay zeros).  The
// caller synchronises before the tile is read.
template <typename T, int D>
__device__ __forceinline__ void walk_map_tile(unsigned char *tile, int fmap, int row0, int N, int width, T *out,
                                              int64_t out_stride, int tid) {
    using W = WalkCfg<D>;
    feature_dispatch(fmap, [&](auto map) {
#pragma unroll
        for (int v = 0; v < W::C * W::CR / 256; ++v) {
            const int u = tid + 256 * v, r = u / W::CR, pos = u % W::CR, c = pos ^ walk_swizzle<W::CR>(r);
            if (row0 + r < N && c * 8 < width) {
                u32x4 *ptr = reinterpret_cast<u32x4 *>(tile + r * W::RB + (pos << 4));
                const u32x4 m = feature_map8_c<T, decltype(map)::value>(*ptr);
                *ptr = m;
                *reinterpret_cast<u32x4 *>(out + (int64_t)(row0 + r) * out_stride + c * 8) = m;
            }
        }
    });
}

// acc[i][v] = Out[row][32 (db0 + i) + 16 g + v] rounded to the storage type: pk[i][hq] = columns
// 32 (db0 + i) + 16 g + 8 hq .. + 7.  With a feature map, `ytile` is the LDS tile holding
// y = phi(x) for the same rows (tile row `trow`) and Out is multiplied by the slope phi'(x),
// computed from y, first.
template <typename T, int D, int PER = WalkCfg<D>::DBW>
__device__ __forceinline__ void walk_pack(const f32x16 (&acc)[WalkCfg<D>::DBW], int g, int db0,
                                          u32x4 (&pk)[WalkCfg<D>::DBW][2], int fmap = 0,
                                          const unsigned char *ytile = nullptr, int trow = 0) {
    using W = WalkCfg<D>;
    using V8 = typename Mma<T>::V8;
    float sl[PER][2][8];  // the slopes (one branch on the map around all of them)
    if (fmap) {
        feature_dispatch(fmap, [&](auto map) {
#pragma unroll
            for (int i = 0; i < PER; ++i)
#pragma unroll
                for (int hq = 0; hq < 2; ++hq) {
                    const int ch = (4 * (db0 + i) + 2 * g + hq) ^ walk_swizzle<W::CR>(trow);
                    const V8 y = __builtin_bit_cast(V8, *reinterpret_cast<const u32x4 *>(ytile + trow * W::RB + (ch << 4)));
#pragma unroll
                    for (int e = 0; e < 8; ++e) sl[i][hq][e] = feature_slope_c<decltype(map)::value>(static_cast<float>(y[e]));
                }
        });
    }
#pragma unroll
    for (int i = 0; i < PER; ++i) {
#pragma unroll
        for (int hq = 0; hq < 2; ++hq) {
            V8 o8;
#pragma unroll
            for (int e = 0; e < 8; ++e) o8[e] = static_cast<T>(fmap ? acc[i][8 * hq + e] * sl[i][hq][e] : acc[i][8 * hq + e]);
            pk[i][hq] = __builtin_bit_cast(u32x4, o8);
        }
    }
}

// two 16-byte stores per block; rows >= N and columns beyond the true width fall outside the
// buffer resource and are dropped
template <int D, int PER = WalkCfg<D>::DBW>
__device__ __forceinline__ void walk_store_packed(__amdgpu_buffer_rsrc_t rs, int stride2, int width, int row, int g,
                                                  int db0, const u32x4 (&pk)[WalkCfg<D>::DBW][2]) {
#pragma unroll
    for (int i = 0; i < PER; ++i)
#pragma unroll
        for (int hq = 0; hq < 2; ++hq) {
            const int col = 32 * (db0 + i) + 16 * g + 8 * hq;
            const uint32_t off = (uint32_t)(row * stride2 + col * 2) + (col < width ? 0u : kOobOffset);
            __builtin_amdgcn_raw_buffer_store_b128(pk[i][hq], rs, off, 0, 0);
        }
}

// ... the same values as fp32 (bf16: its bits with sixteen zeros behind them), four stores per block; stride_b: of a row, in bytes
template <int D, int PER>
__device__ __forceinline__ void walk_store_widened(__amdgpu_buffer_rsrc_t rs, int stride_b, int width, int row, int g, int db0,
                                                   const u32x4 (&pk)[WalkCfg<D>::DBW][2]) {
#pragma unroll
    for (int i = 0; i < PER; ++i)
#pragma unroll
        for (int hq = 0; hq < 2; ++hq)
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                const int col = 32 * (db0 + i) + 16 * g + 8 * hq + 4 * a;
                const uint32_t off = (uint32_t)(row * stride_b + col * 4) + (col < width ? 0u : kOobOffset);
                const uint32_t lo = pk[i][hq][2 * a], hi = pk[i][hq][2 * a + 1];
                __builtin_amdgcn_raw_buffer_store_b128(u32x4{lo << 16, lo & 0xffff0000u, hi << 16, hi & 0xffff0000u}, rs, off, 0, 0);
            }
}

// (PER: the blocks of acc that are this wave's -- the others belong to another wave or hold nothing.  wide: WalkParams::wide_out,
// stride2 then being a row of floats)
template <typename T, int D, int PER = WalkCfg<D>::DBW>
__device__ __forceinline__ void walk_store(__amdgpu_buffer_rsrc_t rs, int stride2, int width, int row, int g, int db0,
                                           const f32x16 (&acc)[WalkCfg<D>::DBW], int fmap = 0,
                                           const unsigned char *ytile = nullptr, int trow = 0, int wide = 0) {
    u32x4 pk[WalkCfg<D>::DBW][2];
    walk_pack<T, D, PER>(acc, g, db0, pk, fmap, ytile, trow);
    if constexpr (std::is_same<T, __bf16>::value) {
        if (wide) {
            walk_store_widened<D, PER>(rs, stride2, width, row, g, db0, pk);
            return;
        }
    }
    walk_store_packed<D, PER>(rs, stride2, width, row, g, db0, pk);
}

// Where a result of (b, h) starts and its rows' stride and descriptor, for 16-bit or fp32 storage
struct WalkResult {
    __amdgpu_buffer_rsrc_t rs;
    int stride;  // bytes
    __device__ __forceinline__ WalkResult(void *base, int64_t at, int64_t stride_n, int width, int N, int wide) {
        const int size = wide ? 4 : 2;
        stride = (int)stride_n * size;
        rs = __builtin_amdgcn_make_buffer_rsrc(static_cast<char *>(base) + at * size, 0, (N - 1) * stride + width * size, 0x00020000);
    }
};

// A result whose rows start at any element: 16-byte stores at the rows' own alignment, what is left of a row element by
// element.  Forward + backward with results in aligned rows that a copy took to the caller's -> this way: B H 32, N 2048, 153 over
// 64 columns (306-byte rows) 139.5 -> 127.3 us; B H 32, N 4096, 100 columns 231 -> 177, by one reverse walk 218 -> 167; B H 128 736 -> 547.
template <typename T>
struct WalkAnyRows {
    T *base;
    int64_t stride;
    int width, N;
    __device__ __forceinline__ WalkAnyRows(const WalkRowsOut &o, int b, int h, int col0, int w, int n)
        : base(static_cast<T *>(o.ptr) + b * o.s_b + h * o.s_h + col0), stride(o.s_n), width(w), N(n) {}
    template <int D, int PER>
    __device__ __forceinline__ void store(int row, int g, int db0, const f32x16 (&acc)[WalkCfg<D>::DBW]) const {
        u32x4 pk[WalkCfg<D>::DBW][2];
        walk_pack<T, D, PER>(acc, g, db0, pk);
        if (row >= N) return;
        T *r = base + row * stride;
#pragma unroll
        for (int i = 0; i < PER; ++i)
#pragma unroll
            for (int hq = 0; hq < 2; ++hq) {
                const int col = 32 * (db0 + i) + 16 * g + 8 * hq;
                if (col + 8 <= width) {
                    __builtin_memcpy(r + col, &pk[i][hq], 16);
                } else if (col < width) {
#pragma unroll
                    for (int e = 0; e < 7; ++e) {
                        const uint16_t x = (uint16_t)(pk[i][hq][e / 2] >> (16 * (e & 1)));
                        if (e < width % 8) __builtin_memcpy(r + col + e, &x, 2);  // (the same for all lanes)
                    }
                }
            }
    }
};

// state += Y^T Z over the rows of the tiles, this wave's 32 x 32 blocks (block i: Y columns of block
// dbk(i), Z columns of block eb): st[i][v] = State[32 dbk(i) + 8(v/4) + 4g + v%4][32 eb + l32]
// (NEG: state -= Y^T Z -- the sign bits of the Z fragments are flipped.  ACC: the state lives in
// accumulation registers, see Mma::mma_acc; the wait states an MFMA's result needs before anything
// but another MFMA reads it are spent at the end, since the compiler does not count them for a
// statement it cannot look into.)
template <typename T, int D, typename B = WalkExt<D>, bool NEG = false, bool ACC = false>
__device__ __forceinline__ void walk_update(const unsigned char *yt, const unsigned char *zt, int wave, int lane,
                                            f32x16 (&st)[WalkCfg<D>::NBW]) {
    using W = WalkCfg<D>;
    using M = Mma<T>;
    using V8 = typename M::V8;
    if (!B::valid(wave, 0)) return;
    // per 16 rows: the Z fragment, then the Y fragment of every block -- one group of reads ahead of the MFMAs
    constexpr int G = 1 + B::SLOTS, KS = W::C / 16;
    V8 zf = {};
    walk_pipe<KS * G, G, V8>(
        [&](auto j) {
            constexpr int ks = decltype(j)::value / G, r = decltype(j)::value % G;
            if constexpr (r == 0) {
                V8 z = walk_col_frag<T, D>(zt, 16 * ks, B::eb(wave), lane);
                if constexpr (NEG) {
                    u32x4 raw = __builtin_bit_cast(u32x4, z);
#pragma unroll
                    for (int e = 0; e < 4; ++e) raw[e] ^= 0x80008000u;
                    z = __builtin_bit_cast(V8, raw);
                }
                return z;
            } else {
                // (a slot without a block -- only in the last one, with fewer than four blocks in all -- reads block 0)
                return walk_col_frag<T, D>(yt, 16 * ks, B::valid(wave, r - 1) ? B::dbk(wave, r - 1) : 0, lane);
            }
        },
        [&](auto j, V8 f) {
            constexpr int r = decltype(j)::value % G;
            if constexpr (r == 0) {
                zf = f;
            } else if (B::valid(wave, r - 1)) {
                if constexpr (ACC)
                    M::mma_acc(f, zf, st[r - 1]);
                else
                    st[r - 1] = M::mma(f, zf, st[r - 1]);
            }
        });
    if constexpr (ACC) {
        static_assert(!ACC || B::SLOTS == 4 || B::SLOTS == 2, "written for two or four blocks per wave");
        if constexpr (B::SLOTS == 4)
            asm volatile("s_nop 15\n\ts_nop 7" : "+a"(st[0]), "+a"(st[1]), "+a"(st[2]), "+a"(st[3]));
        else
            asm volatile("s_nop 15\n\ts_nop 7" : "+a"(st[0]), "+a"(st[1]));
    }
}

// acc += column sums of the tile's rows (all of them, or this wave's part: with fewer than four 32-column blocks the
// waves of a block share the rows), by MFMAs against a fragment of ones: exact products, fp32 sums, four MFMAs per wave
// and chunk.  Every lane column holds the same sums: acc[v] of column 32 (wave % DB) + 8(v/4) + 4g + v%4.
template <typename T, int D>
__device__ __forceinline__ void walk_col_sums(const unsigned char *yt, int wave, int lane, f32x16 &acc) {
    using W = WalkCfg<D>;
    using V8 = typename Mma<T>::V8;
    constexpr int KS = W::C / 16 / (4 / W::DB);  // 16-row steps per wave
    V8 ones;
#pragma unroll
    for (int e = 0; e < 8; ++e) ones[e] = static_cast<T>(1.0f);
    static_for<0, KS>([&](auto j) {
        const int ks = (wave / W::DB) * KS + decltype(j)::value;
        acc = Mma<T>::mma(walk_col_frag<T, D>(yt, 16 * ks, wave % W::DB, lane), ones, acc);
    });
}
// ... to LDS: part[wave / DB][column], 4 / DB parts of D floats
template <int D>
__device__ __forceinline__ void walk_col_sums_to_lds(float *part, int wave, int lane, const f32x16 &acc) {
    constexpr int DB = D / 32;
    typedef float f32x4_ __attribute__((ext_vector_type(4)));
    if ((lane & 31) == 0) {
#pragma unroll
        for (int a = 0; a < 4; ++a)
            *reinterpret_cast<f32x4_ *>(part + (wave / DB) * D + 32 * (wave % DB) + 8 * a + 4 * (lane >> 5)) =
                f32x4_{acc[4 * a], acc[4 * a + 1], acc[4 * a + 2], acc[4 * a + 3]};
    }
}
template <int D>
__device__ __forceinline__ float walk_col_sum_of(const float *part, int col) {
    float t = 0.f;
#pragma unroll
    for (int u = 0; u < 4 / (D / 32); ++u) t += part[u * D + col];
    return t;
}

// this lane's part of the column sums of the tile's rows times w (fp32 in LDS, one value per row): the rows
// R0 + {4g .., 8 + 4g ..} of the steps ks of this wave, of column 32 (wave % DB) + l32.  In fp32 throughout: the fragments
// are the ones an MFMA would take, but w would have to be rounded for it.
template <typename T, int D>
__device__ __forceinline__ float walk_weighted_sums(const unsigned char *yt, const float *w, int wave, int lane) {
    using W = WalkCfg<D>;
    using V8 = typename Mma<T>::V8;
    constexpr int KS = W::C / 16 / (4 / W::DB);  // 16-row steps per wave
    const int g = lane >> 5;
    float sum = 0.f;
    static_for<0, KS>([&](auto j) {
        const int ks = (wave / W::DB) * KS + decltype(j)::value;
        const V8 y = walk_col_frag<T, D>(yt, 16 * ks, wave % W::DB, lane);
#pragma unroll
        for (int a = 0; a < 2; ++a) {
            const f32x4 wv = *reinterpret_cast<const f32x4 *>(w + 16 * ks + 8 * a + 4 * g);
#pragma unroll
            for (int b = 0; b < 4; ++b) sum += wv[b] * static_cast<float>(y[4 * a + b]);
        }
    });
    return sum;
}
// ... to LDS, in the layout of walk_col_sums_to_lds
template <int D>
__device__ __forceinline__ void walk_weighted_sums_to_lds(float *part, int wave, int lane, float sum) {
    constexpr int DB = D / 32;
    sum += __shfl_xor(sum, 32, 64);
    if (lane < 32) part[(wave / DB) * D + 32 * (wave % DB) + lane] = sum;
}

// x as the sum of three bf16 numbers (its 24 significant bits; what is not finite in the first alone), in the k slots 0 .. 2 of
// an MFMA's A operand whose row is this lane's l32; walk_ones3 is the B operand that adds them up.  One MFMA then adds x to
// a row of an accumulator, where handing it round within the wave takes a ds_bpermute per register.
__device__ __forceinline__ Mma<__bf16>::V8 walk_split3(float x, int g) {
    uint32_t hi = __builtin_bit_cast(uint32_t, x) & 0xffff0000u;
    if (x != x) hi = 0x7fc00000u;
    const float r1 = (hi & 0x7f800000u) == 0x7f800000u ? 0.f : x - __builtin_bit_cast(float, hi);
    const uint32_t mid = __builtin_bit_cast(uint32_t, r1) & 0xffff0000u;
    const float r2 = r1 - __builtin_bit_cast(float, mid);
    const u32x4 w = {g ? 0u : (hi >> 16) | mid, g ? 0u : __builtin_bit_cast(uint32_t, r2) >> 16, 0u, 0u};
    return __builtin_bit_cast(Mma<__bf16>::V8, w);
}
__device__ __forceinline__ Mma<__bf16>::V8 walk_ones3(int g) {
    return __builtin_bit_cast(Mma<__bf16>::V8, u32x4{g ? 0u : 0x3f803f80u, g ? 0u : 0x3f80u, 0u, 0u});
}

// the state rounded to 16 bit into LDS as T[v index][q/k index] (row = 32 eb + l32, four consecutive
// columns per register group), in the tile layout
template <typename T, int D, typename B = WalkExt<D>>
__device__ __forceinline__ void walk_state_to_lds(unsigned char *tl, int wave, int lane,
                                                  const f32x16 (&st)[WalkCfg<D>::NBW], float scale = 1.f) {
    using W = WalkCfg<D>;
    typedef T t4 __attribute__((ext_vector_type(4)));
    const int l32 = lane & 31, g = lane >> 5, row = 32 * B::eb(wave) + l32;
#pragma unroll
    for (int i = 0; i < B::SLOTS; ++i) {
        if (!B::valid(wave, i)) continue;
        const int dbk = B::dbk(wave, i);
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            t4 w;
#pragma unroll
            for (int b = 0; b < 4; ++b) w[b] = static_cast<T>(scale * st[i][4 * a + b]);
            *reinterpret_cast<t4 *>(tl + row * W::RB + (((4 * dbk + a) ^ walk_swizzle<W::CR>(row)) << 4) + 8 * g) = w;
        }
    }
}

// a chunk's saved copy (WalkParams::saved) HBM -> LDS, as it lay there
template <int D>
__device__ __forceinline__ void walk_load_state_copy(const void *src, uint32_t lds_dst, int wave, int lane) {
    constexpr int LOADS = WalkCfg<D>::STATE / 1024;  // of a wave each
    const u32x4 rs = walk_uniform_rsrc(src, WalkCfg<D>::STATE);
    const uint32_t base = (uint32_t)__builtin_amdgcn_readfirstlane((int)(lds_dst + wave * 1024));
    static_for<0, (LOADS + 3) / 4>([&](auto u) {
        constexpr int U = decltype(u)::value;
        if (4 * U + wave < LOADS) dma_16B_per_lane<U * 4096>(rs, base, (uint32_t)(wave * 1024 + lane * 16), U * 4096);
    });
}

// fp16: the sums of a long sequence leave its range where results of the operator do not, so the state's 16-bit copy is
// scaled by a power of two that puts its largest finite element at 2^14 (exact; what is 2^28 times smaller than that becomes
// subnormal).  An infinite or NaN element, which stays what it is at any scale, has no say: the other columns' elements would leave
// fp16's range.  Every wave leaves its largest finite |element| in smax[wave]; behind a barrier walk_state_scale gives the factor of
// the copy and, in `back`, its inverse for the product (1 for a state of zeros).
template <int D, typename B, bool FINITE = false>
__device__ __forceinline__ float walk_state_largest(const f32x16 (&st)[WalkCfg<D>::NBW], int wave) {
    float m = 0.f;
#pragma unroll
    for (int i = 0; i < B::SLOTS; ++i)
        if (B::valid(wave, i)) {
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const float x = fabsf(st[i][v]);
                m = fmaxf(m, FINITE && x == __builtin_inff() ? 0.f : x);  // (a NaN is never the larger one)
            }
        }
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) m = fmaxf(m, __shfl_xor(m, d, 64));
    return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, m)));
}
template <int D, typename B>
__device__ __forceinline__ void walk_state_max(float *smax, int wave, int lane, const f32x16 (&st)[WalkCfg<D>::NBW]) {
    float m = walk_state_largest<D, B>(st, wave);
    if (__builtin_expect(__builtin_bit_cast(uint32_t, m) == 0x7f800000u, 0)) m = walk_state_largest<D, B, true>(st, wave);
    if (lane == 0) smax[wave] = m;
}
__device__ __forceinline__ float walk_state_scale(const float *smax, float &back) {
    const float m = fmaxf(fmaxf(smax[0], smax[1]), fmaxf(smax[2], smax[3]));
    const int e = (int)(__builtin_bit_cast(uint32_t, m) >> 23);  // biased exponent: m < 2^(e - 126)
    const int k = m > 0.f ? (e < 40 ? 40 : e) - 141 : 0;
    back = __builtin_bit_cast(float, (uint32_t)(127 + k) << 23);
    return __builtin_bit_cast(float, (uint32_t)(127 - k) << 23);
}

struct WalkSlice {
    int bh, seg, c_lo, c_hi;  // chunks c_lo .. c_hi - 1
    bool valid;
};

// workgroup -> ((b, h), segment)
__device__ __forceinline__ WalkSlice walk_slice(const WalkParams &p) {
    const XcdItem item = xcd_item(blockIdx.x, p.BH, p.n_seg, p.place, p.n_seg_inv);
    WalkSlice s;
    s.bh = item.bh, s.seg = item.part;
    s.c_lo = s.seg * p.seg_chunks;
    s.c_hi = s.c_lo + p.seg_chunks < p.n_chunks ? s.c_lo + p.seg_chunks : p.n_chunks;
    s.valid = s.bh >= 0 && s.c_lo < p.n_chunks;
    return s;
}

// this wave's blocks of an fp32 state [D][D] in memory, assigned to st or (ADD) added to it;
// `transposed`: the buffer holds the transposed matrix ([v index][q/k index])
template <int D, typename B, bool ADD>
__device__ __forceinline__ void walk_read_state(const float *init, bool transposed, int wave, int lane,
                                                f32x16 (&st)[WalkCfg<D>::NBW]) {
    const int l32 = lane & 31, g = lane >> 5;
    // st[i][v] = State[r = 32 dbk(i) + 8 (v/4) + 4g + v%4][c = 32 eb + l32]: element r D + c of the
    // buffer, or c D + r when it holds the transposed matrix (then four consecutive floats per v/4)
    const int c = 32 * B::eb(wave) + l32;
    if (transposed) {
        typedef float f32x4 __attribute__((ext_vector_type(4)));
#pragma unroll
        for (int i = 0; i < B::SLOTS; ++i)
            if (B::valid(wave, i)) {
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    const f32x4 t = *reinterpret_cast<const f32x4 *>(init + c * D + 32 * B::dbk(wave, i) + 8 * a + 4 * g);
#pragma unroll
                    for (int b = 0; b < 4; ++b) st[i][4 * a + b] = ADD ? st[i][4 * a + b] + t[b] : t[b];
                }
            }
    } else {
#pragma unroll
        for (int i = 0; i < B::SLOTS; ++i)
            if (B::valid(wave, i)) {
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const float t = init[(32 * B::dbk(wave, i) + 8 * (v / 4) + 4 * g + (v % 4)) * D + c];
                    st[i][v] = ADD ? st[i][v] + t : t;
                }
            }
    }
}

// A state that is to be added up on load lies in memory by fragments: block (i, j) of 32 x 32 at float 1024 (i D / 32 + j), in it
// the sixteen values that a lane holds, as four runs of four -- a wave moves 1 KiB of consecutive memory with each access.  Row by
// row a lane's values are four bytes apart from the next lane's, and the 63 accesses that a wave may have in flight are one
// D = 128 state: a memory latency per segment.  (Forward walk, D = 128: B H 32, N 2048, eight segments 24.2 -> 22.0 us, with the
// scan's entry states 16.4; normalised, B H 16, N 4096, sixteen segments 53.6 -> 26.0 us, 20.4 behind a scan of 7.)
template <int D, typename B>
__device__ __forceinline__ void walk_read_frags(const float *buf, int wave, int lane, f32x16 (&st)[WalkCfg<D>::NBW]) {
    typedef float f32x4 __attribute__((ext_vector_type(4)));
#pragma unroll
    for (int i = 0; i < B::SLOTS; ++i)
        if (B::valid(wave, i)) {
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                const f32x4 t = *reinterpret_cast<const f32x4 *>(buf + (B::dbk(wave, i) * (D / 32) + B::eb(wave)) * 1024 + a * 256 + lane * 4);
#pragma unroll
                for (int b = 0; b < 4; ++b) st[i][4 * a + b] = t[b];
            }
        }
}
template <int D, typename B>
__device__ __forceinline__ void walk_write_frags(float *out, int wave, int lane, const f32x16 (&st)[WalkCfg<D>::NBW]) {
    typedef float f32x4 __attribute__((ext_vector_type(4)));
#pragma unroll
    for (int i = 0; i < B::SLOTS; ++i)
        if (B::valid(wave, i)) {
#pragma unroll
            for (int a = 0; a < 4; ++a)
                *reinterpret_cast<f32x4 *>(out + (B::dbk(wave, i) * (D / 32) + B::eb(wave)) * 1024 + a * 256 + lane * 4) =
                    f32x4{st[i][4 * a], st[i][4 * a + 1], st[i][4 * a + 2], st[i][4 * a + 3]};
        }
}

// ... zeros for a null pointer; with `init2` the state is the sum of the two buffers
template <int D, typename B = WalkExt<D>>
__device__ __forceinline__ void walk_load_state(const float *init, bool transposed, int wave, int lane,
                                                f32x16 (&st)[WalkCfg<D>::NBW], const float *init2 = nullptr) {
    using W = WalkCfg<D>;
#pragma unroll
    for (int i = 0; i < W::NBW; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) st[i][v] = 0.f;
    if (!init) return;
    walk_read_state<D, B, false>(init, transposed, wave, lane, st);
    if (init2) walk_read_state<D, B, true>(init2, transposed, wave, lane, st);
}

// Entry states in memory, fp32 [D][D] per segment, [bh][seg], in one of three forms that host and
// kernels tell apart by the number of segments and, at D = 128, WalkParams::init_is_totals:
//   * two segments per (b, h): the first segment in walking order starts from zero and the other one
//     from the one total the totals kernel forms; its two workgroups of a (b, h) add up half of that
//     segment each, and the two slots hold their partial sums;
//   * three to walk_sum_on_load_max(D) segments, or with that flag: the slots hold the segments' TOTALS, by fragments
//     (walk_read_frags), and a walk adds up the totals of the segments before it (after it, walking in reverse)
//     as it starts -- a few states of D x D read from L2 per workgroup instead of a scan kernel between
//     the totals kernel and the walk, whose launch costs more than it computes on plans this small
//     (B H = 16, N = 1024, D = 64, forward + backward: 40.7 -> 32.8 us, bound by its six -> four launches).  D = 64, scan
//     against sums on load: 32 segments B H 16 N 4096 84.7 / 77.1 us, N 32768 232.8 / 227.6, B H 12 N 8192 81.9 / 75.0, forward
//     alone B H 12 N 4096 24.2 / 21.5, B H 10 N 8192 25.2 / 25.7; 64 segments (B H 8 N 8192) forward alone 23.3 / 24.9; beyond 32 forward alone B H 12 N 19200
//     (40 columns) 40.8 / 44.3.  D = 32, whose scan is a quarter of that: 32 segments B H 16 N 8503 forward alone 26.2 / 28.3;
//   * more segments: the slots hold the entry states themselves (walk_scan_kernel).
// (At D = 128 a forward walk then writes the entry states it formed, for backward.)
__host__ __device__ constexpr int walk_sum_on_load_max(int D) { return D <= 32 ? 16 : D <= 64 ? 32 : 0; }
__host__ __device__ constexpr bool walk_entries_are_totals(int D, int n_seg) {
    return n_seg >= 3 && n_seg <= walk_sum_on_load_max(D);
}

// the loads above stay above their uses (short of registers the compiler moves every load down to its use otherwise, and two are in
// flight at a time)
__device__ __forceinline__ void walk_all_requested() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// this wave's blocks of the sum of the states buf[f_lo .. f_hi - 1] (zeros for an empty range; by fragments), added in
// ascending order, the loads of several states in flight together (one state at a time is a chain of
// dependent loads: a memory latency per state at the start of every workgroup).
// What a group has room for past the range is not requested.  (The last state once more in its place, not added: all workgroups of a
// plan of eleven segments then read 1.75 times the states they need, from L2 -- backward walk, D = 64, B H 40, N 5184, 41.1 us, this way
// 38.3; forward, D = 32, B H 128, N 1536, four segments 11.1 / 10.2; 128 over 64 columns, B H 64, N 1024, reverse walk 24.8 / 23.5.
// With four blocks per wave, in groups of three, it stays so: the branches take registers that walk_bwd_rev_wide_kernel does not have)
// At D = 32, where one wave has the state's one block and there are at most 16 segments, groups of four: eight take 148 registers in
// place of 110 and leave three wavefronts to a SIMD in place of four, where many heads have more workgroups than that (the build checks
// it).  Forward, B H 2048, N 300 32.0 us with eight, this way 30.7; forward + backward, B H 32, N 2048, 16 segments 31.5 / 28.7.
// TOGETHER: the group's loads stay ahead of its additions (walk_all_requested).  Not in walk_fwd_wide_kernel with a v above 64 columns:
// its loop over the chunks then holds more in accumulation registers than it has to, 300 moves in place of 221 (forward, 192 / 128, B H
// 128, N 2048 106.6 us, this way 105.2; forward + backward, 256 / 128, B H 42, N 1536, six segments 207.7 / 202.6)
template <int D, typename B, bool TOGETHER = true>
__device__ __forceinline__ void walk_sum_states(const float *buf, int f_lo, int f_hi, int wave, int lane,
                                                f32x16 (&st)[WalkCfg<D>::NBW]) {
    using W = WalkCfg<D>;
    constexpr int GROUP = B::SLOTS > 2 ? 3 : B::SLOTS > 1 ? 6 : D == 32 ? 4 : 8;  // (GROUP x SLOTS x 16 registers beside the sum)
#pragma unroll
    for (int i = 0; i < W::NBW; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) st[i][v] = 0.f;
#pragma unroll 1
    for (int f0 = f_lo; f0 < f_hi; f0 += GROUP) {
        f32x16 t[GROUP][W::NBW];
#pragma unroll
        for (int u = 0; u < GROUP; ++u) {
            if constexpr (B::SLOTS > 2) {  // (past the range: the last state once more, not added -- nor times zero: it may be infinite)
                walk_read_frags<D, B>(buf + (int64_t)(f0 + u < f_hi ? f0 + u : f_hi - 1) * (D * D), wave, lane, t[u]);
            } else {
                if (f0 + u < f_hi) walk_read_frags<D, B>(buf + (int64_t)(f0 + u) * (D * D), wave, lane, t[u]);
            }
        }
        if constexpr (TOGETHER) walk_all_requested();
#pragma unroll
        for (int u = 0; u < GROUP; ++u) {
            if (f0 + u >= f_hi) continue;
#pragma unroll
            for (int i = 0; i < B::SLOTS; ++i)
                if (B::valid(wave, i)) {
#pragma unroll
                    for (int v = 0; v < 16; ++v) st[i][v] += t[u][i][v];
                }
        }
    }
}

// st_a, st_b = this wave's blocks of the sums of the states a[f_lo .. f_hi - 1], b[f_lo .. f_hi - 1], the loads of
// up to three states of each in flight together (a chain of dependent loads costs a memory latency per state).  Past the range
// nothing is requested, as above (forward + backward with the last state once more in its place -> this: 256 / 64, B H 64,
// N 1024 90.8 -> 89.3 us; 153 / 64, B H 80, N 640 98.7 -> 96.9)
template <int D, typename B, typename B2 = B>
__device__ __forceinline__ void walk_sum_two(const float *a, const float *b, int f_lo, int f_hi, int wave, int lane,
                                             f32x16 (&st_a)[WalkCfg<D>::NBW], f32x16 (&st_b)[WalkCfg<D>::NBW]) {
    using W = WalkCfg<D>;
    constexpr int E = D * D, GROUP = 3;
    static_assert(B::SLOTS <= 2, "2 x GROUP x SLOTS x 16 registers beside the two sums: for states of two blocks per wave");
#pragma unroll
    for (int i = 0; i < W::NBW; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) st_a[i][v] = 0.f, st_b[i][v] = 0.f;
#pragma unroll 1
    for (int f0 = f_lo; f0 < f_hi; f0 += GROUP) {
        f32x16 ta[GROUP][W::NBW], tb[GROUP][W::NBW];
#pragma unroll
        for (int u = 0; u < GROUP; ++u) {
            if (f0 + u >= f_hi) continue;
            walk_read_frags<D, B>(a + (int64_t)(f0 + u) * E, wave, lane, ta[u]);
            walk_read_frags<D, B2>(b + (int64_t)(f0 + u) * E, wave, lane, tb[u]);
        }
        walk_all_requested();
#pragma unroll
        for (int u = 0; u < GROUP; ++u) {
            if (f0 + u >= f_hi) continue;
#pragma unroll
            for (int i = 0; i < B::SLOTS; ++i)
                if (B::valid(wave, i)) {
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        st_a[i][v] += ta[u][i][v];
                        if constexpr (std::is_same<B, B2>::value) st_b[i][v] += tb[u][i][v];
                    }
                }
#pragma unroll
            for (int i = 0; i < (std::is_same<B, B2>::value ? 0 : B2::SLOTS); ++i)
                if (B2::valid(wave, i)) {
#pragma unroll
                    for (int v = 0; v < 16; ++v) st_b[i][v] += tb[u][i][v];
                }
        }
    }
}

// this wave's blocks of the entry state of segment sl.seg (zeros without a buffer) of a walk in
// ascending (`reverse` false) or descending order of the chunks; `buf`: the entry states of one operand
template <int D, typename B = WalkExt<D>>
__device__ __forceinline__ void walk_load_init_from(const float *buf, const WalkParams &p, const WalkSlice &sl, int wave,
                                                    int lane, f32x16 (&st)[WalkCfg<D>::NBW], bool reverse, bool transposed) {
    const float *init = nullptr, *init2 = nullptr;
    if (buf) {
        if (p.n_seg == 2) {
            if (sl.seg != (reverse ? 1 : 0)) init = buf + (int64_t)sl.bh * 2 * (D * D), init2 = init + D * D;
        } else if (walk_entries_are_totals(D, p.n_seg) || p.init_is_totals) {
            walk_sum_states<D, B>(buf + (int64_t)sl.bh * p.n_seg * (D * D), reverse ? sl.seg + 1 : 0,
                                  reverse ? p.n_seg : sl.seg, wave, lane, st);
            return;
        } else if (sl.seg != (reverse ? p.n_seg - 1 : 0)) {  // (the first one in walking order starts from zero)
            init = buf + ((int64_t)sl.bh * p.n_seg + sl.seg) * (D * D);
        }
    }
    walk_load_state<D, B>(init, transposed, wave, lane, st, init2);
}
template <int D, typename B = WalkExt<D>>
__device__ __forceinline__ void walk_load_init(const WalkParams &p, const WalkSlice &sl, int wave, int lane,
                                               f32x16 (&st)[WalkCfg<D>::NBW], bool reverse) {
    walk_load_init_from<D, B>(p.init, p, sl, wave, lane, st, reverse, p.init_transposed != 0);
}

// the forward state at the end of segment sl.seg from what forward handed over: the entry state of
// the next segment (xinit, in the forms above) or, for the last one, the final state (xtotal)
template <int D, typename B = WalkExt<D>>
__device__ __forceinline__ void walk_load_end_state_from(const float *xinit, const float *xtotal, const WalkParams &p,
                                                         const WalkSlice &sl, int wave, int lane,
                                                         f32x16 (&xs)[WalkCfg<D>::NBW]) {
    const float *x = xtotal + (int64_t)sl.bh * (D * D), *x2 = nullptr;
    if (sl.c_hi < p.n_chunks) {
        if (p.n_seg == 2) {
            x = xinit + (int64_t)sl.bh * 2 * (D * D), x2 = x + D * D;
        } else if (walk_entries_are_totals(D, p.n_seg)) {
            walk_sum_states<D, B>(xinit + (int64_t)sl.bh * p.n_seg * (D * D), 0, sl.seg + 1, wave, lane, xs);
            return;
        } else {
            x = xinit + ((int64_t)sl.bh * p.n_seg + sl.seg + 1) * (D * D);
        }
    }
    walk_load_state<D, B>(x, false, wave, lane, xs, x2);
}
template <int D, typename B = WalkExt<D>>
__device__ __forceinline__ void walk_load_end_state(const WalkParams &p, const WalkSlice &sl, int wave, int lane,
                                                    f32x16 (&xs)[WalkCfg<D>::NBW]) {
    walk_load_end_state_from<D, B>(p.xinit, p.xtotal, p, sl, wave, lane, xs);
}

// The state transposed, through LDS (`turn`: D rows of D + 4 floats, read and written by nobody else; square states)
template <int D, typename B>
__device__ __forceinline__ void walk_transpose_state(float *turn, int wave, int lane, f32x16 (&st)[WalkCfg<D>::NBW]) {
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    constexpr int P = D + 4;
    const int l32 = lane & 31, g = lane >> 5, c = 32 * B::eb(wave) + l32;
#pragma unroll
    for (int i = 0; i < B::SLOTS; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) turn[(32 * B::dbk(wave, i) + 8 * (v / 4) + 4 * g + (v % 4)) * P + c] = st[i][v];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < B::SLOTS; ++i)
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const f32x4 t = *reinterpret_cast<const f32x4 *>(turn + c * P + 32 * B::dbk(wave, i) + 8 * a + 4 * g);
#pragma unroll
            for (int b = 0; b < 4; ++b) st[i][4 * a + b] = t[b];
        }
    __syncthreads();
}

// this wave's blocks of a state to an fp32 buffer [D][D] ([q/k index][v index]); blocks outside B stay unwritten
template <int D, typename B>
__device__ __forceinline__ void walk_write_state(float *out, int wave, int lane, const f32x16 (&st)[WalkCfg<D>::NBW]) {
    const int l32 = lane & 31, g = lane >> 5;
#pragma unroll
    for (int i = 0; i < B::SLOTS; ++i)
        if (B::valid(wave, i)) {
#pragma unroll
            for (int v = 0; v < 16; ++v)
                out[(32 * B::dbk(wave, i) + 8 * (v / 4) + 4 * g + (v % 4)) * D + 32 * B::eb(wave) + l32] = st[i][v];
        }
}

// ---- one product with its running state, chunks ascending:
//   O_c = lower(Q_c K_c^T) V_c + Q_c S, then S += K_c^T V_c
// (forward as named; dQ of the split backward with q <- dO, k <- V, v <- K, o <- dQ and the entry
// states read transposed)
// DOUBLE: one workgroup per CU with two sets of tiles -- the loads of the next chunk are in flight
// while this one is multiplied.  (Holding a chunk's results back and storing them after the next
// chunk's tiles have been awaited, so that the wait for the tiles never includes fresh stores,
// measured 20 % slower: the stores then compete with the loads in flight instead of filling the
// gap after them.)
// NORM: the instantiations that take the normaliser's terms: 1 forward (WalkParams::denom), 2 dQ (dn).
// FM: the instantiations that know of feature maps (WalkParams::fmap, slope_y); the others ignore both.
// NQ, NV: blocks of the state [q/k index][v index] that hold anything (WalkExt).
// the plain fp16 forward: walk_state_scale
template <typename T, int NORM, bool FM>
constexpr bool walk_fwd_scaled = std::is_same<T, _Float16>::value && NORM == 0 && !FM;

template <typename T, int D, bool DOUBLE, int NORM, bool FM, int NQ = D / 32, int NV = D / 32, bool WIDE = false, bool ROWS = false,
          bool RSUM = false, bool COLS = false>
__global__ __launch_bounds__(256, DOUBLE ? 1 : 2) void walk_fwd_kernel(const WalkParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
    using W = WalkCfg<D>;
    using V8 = typename Mma<T>::V8;
    using B = WalkExt<D, NQ, NV>;
    using OB = WalkOut<D, NV>;  // the result is as wide as v
    static_assert(NORM == 0 || (NQ == W::DB && NV == W::DB), "the normaliser's variants are built for full widths");
    constexpr int SETS = DOUBLE ? 2 : 1, TPS = RSUM ? 4 : 3;  // (tiles per set)
    static_assert(!RSUM || (DOUBLE && NORM == 0 && !FM), "the plain dQ walk");
    static_assert(!COLS || (DOUBLE && NORM == 0 && !FM && !RSUM && NQ == 4 && NV == 2), "64 of the columns of a plain walk");
    using RB = WalkExt<D, D / 32, NQ>;  // (RSUM: the total's blocks -- q's columns are v's here, dO's are q's)
    constexpr bool SCALED = walk_fwd_scaled<T, NORM, FM>;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)smem;
    unsigned char *tl = smem + SETS * TPS * W::TILE;
    unsigned char *xv = tl + W::STATE;  // NORM 2: per set: zc, (unused), dn of the chunk
    float *zv = reinterpret_cast<float *>(xv), *zpart = zv + 256;  // NORM 1: zc; the waves' column sums
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rb = W::NCH == 1 ? wave : wave % W::NRB, db0 = OB::db0(wave);
    const WalkSlice sl = walk_slice(p);
    if (!sl.valid) return;
    const int fmap = FM ? p.fmap : 0;
    const void *slope_y = FM ? p.slope_y : nullptr;
    const int b = sl.bh / p.H, h = sl.bh - b * p.H, N = p.N;
    const T *Q = static_cast<const T *>(p.q) + b * p.qs_b + h * p.qs_h;
    const T *K = static_cast<const T *>(p.k) + b * p.ks_b + h * p.ks_h;
    const int col0 = COLS ? 64 * (int)blockIdx.y : 0;
    const int wv = !COLS ? p.wv : p.wv - col0 < 64 ? p.wv - col0 : 64;
    const T *V = static_cast<const T *>(p.v) + b * p.vs_b + h * p.vs_h + col0;
    const int qs2 = (int)p.qs_n * 2, ks2 = (int)p.ks_n * 2, vs2 = (int)p.vs_n * 2;
    const u32x4 rq = make_rsrc(Q, (uint32_t)((N - 1) * qs2 + p.wqk * 2));
    const u32x4 rk = make_rsrc(K, (uint32_t)((N - 1) * ks2 + p.wqk * 2));
    const u32x4 rv = make_rsrc(V, (uint32_t)((N - 1) * vs2 + wv * 2));
    const WalkResult ro(p.o, b * p.os_b + h * p.os_h + col0, p.os_n, wv, N, WIDE);
    const WalkAnyRows<T> ao(p.rows_o, b, h, col0, !COLS ? p.rows_o.width : p.rows_o.width - col0 < 64 ? p.rows_o.width - col0 : 64, N);

    // (RSUM: the first segment's total is under no sum of the reverse walk)
    const bool rsum = RSUM && sl.seg > 0;
    const int rs2 = RSUM ? (int)p.rs_n * 2 : 0;
    const u32x4 rr = RSUM ? make_rsrc(static_cast<const T *>(p.r_q) + b * p.rs_b + h * p.rs_h, (uint32_t)((N - 1) * rs2 + p.wv * 2)) : rq;
    f32x16 rt[W::NBW];
    if constexpr (RSUM) {
#pragma unroll
        for (int i = 0; i < W::NBW; ++i)
#pragma unroll
            for (int v = 0; v < 16; ++v) rt[i][v] = 0.f;
    }

    f32x16 st[W::NBW];
    walk_load_init<D, B>(p, sl, wave, lane, st, false);
    if constexpr (DOUBLE && NORM <= 1) {  // (the entry state this walk formed from the segments' totals, for backward)
        // (Through a descriptor.  By walk_write_state, with a scalar address per store, scalar registers ran out: the loop below held the
        // result's descriptor in vector registers, with a loop over the lanes around each of its stores -- in every plan, entry states
        // or not.  Forward that way -> this: normalised, B H 300, N 600 66.9 -> 64.1 us (two rounds of one segment), B H 100, N 1000 45.3 -> 43.6
        // (two), B H 16, N 20000 110.9 -> 107.5; plain, B H 300, N 600 51.7 -> 49.1)
        if (p.init_is_totals && p.entry_out && sl.seg > 0) {
            const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
                p.entry_out + ((int64_t)sl.bh * p.n_seg + sl.seg) * (D * D), 0, D * D * 4, 0x00020000);
#pragma unroll
            for (int i = 0; i < B::SLOTS; ++i)
                if (B::valid(wave, i)) {
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        const float x = st[i][v];  // (of an element itself the cast takes the vector's first)
                        const int at = (32 * B::dbk(wave, i) + 8 * (v / 4) + 4 * g + (v % 4)) * D + 32 * B::eb(wave) + l32;
                        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, x), rs, (uint32_t)(at * 4), 0, 0);
                    }
                }
        }
    }
    // the state's copy in LDS for the next chunk (SCALED: every wave has passed a barrier since its walk_state_max)
    float sback = 1.f, *smax = reinterpret_cast<float *>(xv);
    auto publish_state = [&]() {
        if constexpr (SCALED) {
            const float scale = walk_state_scale(smax, sback);
            walk_state_to_lds<T, D, B>(tl, wave, lane, st, scale);
        } else {
            walk_state_to_lds<T, D, B>(tl, wave, lane, st);
        }
    };
    if constexpr (SCALED) {
        walk_state_max<D, B>(smax, wave, lane, st);
        __syncthreads();
    }
    publish_state();
    // NORM 1: zc at the segment's entry from the segments' totals, thread groups of D taking every (256 / D)-th segment
    float zrun = 0.f;  // (of column tid, tid < D)
    auto zc_publish = [&](int c) {
        zv[tid] = zrun;
        if (p.zc_out) p.zc_out[((int64_t)sl.bh * p.n_chunks + c) * D + tid] = zrun;
    };
    if constexpr (NORM == 1) {
        constexpr int G = 256 / D;
        float t = 0.f;
        if (p.vsum) {
            const float *vs = p.vsum + (int64_t)sl.bh * p.n_seg * D + tid % D;
            const int before = p.n_seg == 2 ? (sl.seg ? 2 : 0) : sl.seg;
#pragma unroll 8
            for (int f = tid / D; f < before; f += G) t += vs[(int64_t)f * D];
        }
        zpart[tid] = t;
        __syncthreads();
        if (tid < D) {
#pragma unroll
            for (int u = 0; u < G; ++u) zrun += zpart[u * D + tid];
            zc_publish(sl.c_lo);
        }
    }

    auto load_chunk = [&](int c, int buf) {
        const uint32_t base = lds0 + buf * TPS * W::TILE;
        walk_load_tile<D>(rq, base, c * W::C, qs2, p.wqk, wave, lane);
        walk_load_tile<D>(rk, base + W::TILE, c * W::C, ks2, p.wqk, wave, lane);
        walk_load_tile<D>(rv, base + 2 * W::TILE, c * W::C, vs2, wv, wave, lane);
        if constexpr (RSUM)
            if (rsum) walk_load_tile<D>(rr, base + 3 * W::TILE, c * W::C, rs2, p.wv, wave, lane);
        const uint32_t xbase = lds0 + SETS * 3 * W::TILE + W::STATE + buf * W::VEC;
        if constexpr (NORM == 2) {
            walk_load_vec<D>(p.zc + ((int64_t)sl.bh * p.n_chunks + c) * D, xbase, lane);
            walk_load_rows<D>(p.dn + (int64_t)sl.bh * N, c * W::C, N, xbase + 2048, lane);
        }
    };
    constexpr int n_extra = NORM == 2 ? 1 + W::NID : 0;  // loads per chunk and wave beyond the tiles
    if constexpr (DOUBLE) load_chunk(sl.c_lo, 0);
#pragma unroll 1
    for (int c = sl.c_lo; c < sl.c_hi; ++c) {
        const int row0 = c * W::C, buf = DOUBLE ? (c - sl.c_lo) & 1 : 0;
        unsigned char *tq = smem + buf * TPS * W::TILE, *tk = tq + W::TILE, *tv = tq + 2 * W::TILE;
        const int row = row0 + 32 * rb + l32;
        // dQ walk with a feature map: this lane's values of phi(xq) under its accumulator registers,
        // requested before the tiles so that they have arrived with them
        V8 ys[W::DBW][2];
        if (slope_y) {
            const T *yrow = static_cast<const T *>(slope_y) + b * p.sy_b + h * p.sy_h + (int64_t)(row < N ? row : 0) * p.sy_n;
#pragma unroll
            for (int i = 0; i < W::DBW; ++i)
#pragma unroll
                for (int hq = 0; hq < 2; ++hq) {
                    const int col = 32 * (db0 + i) + 16 * g + 8 * hq;
                    u32x4 raw = {0u, 0u, 0u, 0u};
                    if (col < p.wv) raw = *reinterpret_cast<const u32x4 *>(yrow + col);
                    ys[i][hq] = __builtin_bit_cast(V8, raw);
                }
        }
        if constexpr (DOUBLE) {
            const bool more = c + 1 < sl.c_hi;
            if (more) load_chunk(c + 1, buf ^ 1);  // (every wave has left the barrier that ended the reads of that set)
            // this wave's loads of chunk c have landed when at most the loads issued after them are
            // outstanding (the stores of the previous chunk were issued before those)
            if (more && rsum)
                wait_vm<4 * W::NI>();
            else if (more)
                wait_vm<3 * W::NI + n_extra>();
            else
                wait_vm<0>();
            __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's part of the state is in LDS
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            if (fmap && p.qmap_out) {
                walk_map_tile<T, D>(tq, fmap, row0, N, p.wqk, static_cast<T *>(p.qmap_out) + b * p.qo_b + h * p.qo_h,
                                    p.qo_n, tid);
                __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the rewritten tile is in LDS
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
            }
        } else {
            load_chunk(c, 0);
            wait_vm<0>();
            __syncthreads();  // the tiles have landed; the state written by the previous iteration is visible
            if (fmap && p.qmap_out) {
                walk_map_tile<T, D>(tq, fmap, row0, N, p.wqk, static_cast<T *>(p.qmap_out) + b * p.qo_b + h * p.qo_h,
                                    p.qo_n, tid);
                __syncthreads();
            }
        }
        if constexpr (!DOUBLE && NORM <= 1) {
            if (p.saved && c > 0) {  // the state's copy for backward's dQ (at the first chunk it is zero and not read)
                unsigned char *sv = static_cast<unsigned char *>(p.saved) + ((int64_t)sl.bh * p.n_chunks + c) * W::STATE;
                for (int i = tid * 16; i < W::STATE; i += 4096) {
                    V8 copy = __builtin_bit_cast(V8, *reinterpret_cast<const u32x4 *>(tl + i));
                    if (SCALED && !p.saved_scale) {
#pragma unroll
                        for (int e = 0; e < 8; ++e) copy[e] = static_cast<T>(static_cast<float>(copy[e]) * sback);
                    }
                    *reinterpret_cast<u32x4 *>(sv + i) = __builtin_bit_cast(u32x4, copy);
                }
                if constexpr (std::is_same<T, _Float16>::value && NORM == 0)  // (1 where the copy is not scaled)
                    if (p.saved_scale && tid == 0) p.saved_scale[(int64_t)sl.bh * p.n_chunks + c] = sback;
            }
        }
        f32x16 acc[W::DBW];
        const float *vz = reinterpret_cast<const float *>(xv + (NORM == 1 ? 0 : buf * W::VEC));
        const float *vd = reinterpret_cast<const float *>(xv + buf * W::VEC + 2048);
        auto sfrag = [&](int db, int kc) -> V8 { return walk_row_frag<T, D>(tl, 32 * db + walk_e_lane(l32), kc, g); };
        if constexpr (NORM == 1) {  // forward with the normaliser: n = masked row sum + q . zc + eps
            float tot;
            walk_product<T, D, false, 1, B::KQ, NV>(tq, tk, tv, wave, lane, c > 0, sfrag, acc, &tot, vz);
            const float n = tot + p.eps, inv = 1.0f / n;
#pragma unroll
            for (int i = 0; i < W::DBW; ++i)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[i][v] *= inv;
            if (db0 == 0 && g == 0 && row < N) p.denom[(int64_t)sl.bh * N + row] = n;
        } else if constexpr (NORM == 2) {  // dQ with the normaliser's term: scores + dn_i, result + dn_i zc
            float ax = vd[32 * rb + l32];
            walk_product<T, D, false, 2, B::KQ, NV>(tq, tk, tv, wave, lane, c > 0, sfrag, acc, &ax);
            walk_add_vec<D>(acc, ax, vz, db0, g);
        } else {
            walk_product<T, D, false, 0, B::KQ, NV, false, SCALED>(tq, tk, tv, wave, lane, c > 0, sfrag, acc, nullptr, nullptr,
                                                                   WalkNoRows{}, sback);
        }
        if (slope_y) {
            feature_dispatch(fmap, [&](auto map) {
#pragma unroll
                for (int i = 0; i < W::DBW; ++i)
#pragma unroll
                    for (int v = 0; v < 16; ++v)
                        acc[i][v] *= feature_slope_c<decltype(map)::value>(static_cast<float>(ys[i][v / 8][v % 8]));
            });
        }
        if constexpr (ROWS)
            ao.template store<D, OB::PER>(row, g, db0, acc);
        else
            walk_store<T, D, OB::PER>(ro.rs, ro.stride, wv, row, g, db0, acc, 0, nullptr, 0, WIDE);
        walk_update<T, D, B>(tk, tv, wave, lane, st);
        if constexpr (COLS) {
            if (p.mid_out && c + 1 == p.mid_chunk) {  // (as the partial sums of two segments: this, and zeros)
                const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
                    p.mid_out + (int64_t)sl.bh * 2 * (D * D), 0, 2 * D * D * 4, 0x00020000);
#pragma unroll
                for (int i = 0; i < B::SLOTS; ++i)
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        const float x = st[i][v];
                        const int at = (32 * B::dbk(wave, i) + 8 * (v / 4) + 4 * g + (v % 4)) * D + col0 + 32 * B::eb(wave) + l32;
                        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, x), rs, (uint32_t)(at * 4), 0, 0);
                        __builtin_amdgcn_raw_buffer_store_b32(0u, rs, (uint32_t)(at * 4), D * D * 4, 0);
                    }
            }
        }
        if constexpr (RSUM)
            if (rsum) walk_update<T, D, RB>(tv + W::TILE, tq, wave, lane, rt);
        if constexpr (SCALED) walk_state_max<D, B>(smax, wave, lane, st);
        if constexpr (NORM == 1) {
            f32x16 zs;
#pragma unroll
            for (int v = 0; v < 16; ++v) zs[v] = 0.f;
            walk_col_sums<T, D>(tk, wave, lane, zs);
            walk_col_sums_to_lds<D>(zpart, wave, lane, zs);
        }
        if constexpr (DOUBLE) {
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(0xc07f);  // this wave's LDS reads of the tiles and of the state are done
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        } else {
            __syncthreads();  // every wave is done with the tiles and with the old state
        }
        publish_state();
        if constexpr (NORM == 1) {
            if (tid < D && c + 1 < sl.c_hi) {
                zrun += walk_col_sum_of<D>(zpart, tid);
                zc_publish(c + 1);
            }
        }
    }
    if constexpr (RSUM) {
        float *out = p.r_totals + ((int64_t)sl.bh * p.n_seg + sl.seg) * (D * D);
        if (rsum && p.r_frags)
            walk_write_frags<D, RB>(out, wave, lane, rt);
        else if (rsum)
            walk_write_state<D, RB>(out, wave, lane, rt);
        return;
    }
    if (p.total_out && sl.c_hi == p.n_chunks) {  // the state after the last chunk, for the backward walks
        float *out = p.total_out + (int64_t)sl.bh * (D * D) + col0;
#pragma unroll
        for (int i = 0; i < B::SLOTS; ++i)
            if (B::valid(wave, i)) {
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    out[(32 * B::dbk(wave, i) + 8 * (v / 4) + 4 * g + (v % 4)) * D + 32 * B::eb(wave) + l32] = st[i][v];
            }
        // (built for a narrow q / k side: walk_bwd_rev_kernel has no such variant and reads every block)
        if constexpr (NQ < W::DB) {
            for (int e = tid; e < D * D; e += 256)
                if (e / D >= 32 * NQ || e % D >= 32 * NV) out[e] = 0.f;
        }
    }
#else
    (void)p;
#endif
}

// ---- forward for q and k of 129 .. 256 columns (v of at most 128), one walk over both 128-column halves:
//   O_c = sum over the halves h of lower(Q_h,c K_h,c^T) V_c + Q_h,c S_h,   then S_h += K_h,c^T V_c
// Each half is the D = 128 product of walk_fwd_kernel with a state of its own; the chunk's result stays in
// its fp32 accumulators from the first half to the second and is rounded and stored once, and V is loaded
// once per chunk -- where two walks of walk_fwd_kernel, the second adding to the first one's result, load V
// twice, write O twice and read it back once.
// LDS: a set of (Q_h, K_h) tiles per half -- while half h of a chunk is multiplied, the loads of the next
// half-chunk go to the other set -- two V tiles (chunk parity), and ONE 16-bit state: a half's state is
// needed in LDS only for that half's product, so at the end of a half-chunk the other half's state (in
// registers throughout, updated one half-chunk earlier) is rounded into the buffer.
// NV: the state's v blocks that hold anything (2: v of at most 64 columns).  N2: those of the second half of the contraction (4, 2: at most
// 64 columns, 1: 32), whose state, scores and updates leave the padding's MFMAs and states out.
// A v of 129 .. 256 columns as well (WalkParams::quad): every gradient is a sum over the two halves of one operand pair against a
// half of a third, as O is, and takes this walk too: dQ in its halves ascending, with (dO, V, K) for (Q, K, V); REV, chunks descending:
// dV in its halves from (K, Q, dO) and dK from (V, dO, Q).
template <typename T, int NV, bool REV, int N2, bool QUAD>
__device__ __forceinline__ void walk_wide_body(const WalkParams &p) {
    constexpr int D = 128;
    using W = WalkCfg<D>;
    using V8 = typename Mma<T>::V8;
    using B = WalkExt<D, D / 32, NV>;
    using B2 = WalkExt<D, N2, NV>;
    using OB = WalkOut<D, NV>;  // the result is as wide as v
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)smem;
    unsigned char *tl = smem + 6 * W::TILE;
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rb = wave % W::NRB, db0 = OB::db0(wave);
    const WalkSlice sl = walk_slice(p);
    if (!sl.valid) return;
    // quad: grid y is the half of v (of the third operand) that this workgroup takes; REV: 0, 1 dV's halves, 2, 3 dK's
    const int part = QUAD ? (int)blockIdx.y : 0, vh = part & 1;
    const bool dk = REV && part >= 2;
    const int wx2 = dk ? p.wv2 : p.wqk2, wv = vh ? (dk ? p.wqk2 : p.wv2) : p.wv;
    // (the states of dQ and dK are the transposed ones of O's and dV's)
    const bool transposed = REV ? dk : QUAD && p.init_transposed != 0;
    WalkSlice ss = sl;  // (as sl, for the states)
    ss.bh += (transposed ? 1 : 2) * vh * p.BH;
    const int64_t to_second = (int64_t)(transposed ? 2 : 1) * p.BH * p.n_seg * (D * D);
    const float *const init2 = QUAD && p.init ? p.init + to_second : p.init2;
    const int b = sl.bh / p.H, h = sl.bh - b * p.H, N = p.N;
    // X, Y, Z and the result: Q, K, V and O (REV: K, Q, dO and dV; V, dO, Q and dK)
    const T *tensor[4] = {static_cast<const T *>(p.q) + b * p.qs_b + h * p.qs_h, static_cast<const T *>(p.k) + b * p.ks_b + h * p.ks_h,
                          static_cast<const T *>(p.v) + b * p.vs_b + h * p.vs_h,
                          REV ? static_cast<const T *>(p.go) + b * p.gs_b + h * p.gs_h : nullptr};
    const int row_bytes[4] = {(int)p.qs_n * 2, (int)p.ks_n * 2, (int)p.vs_n * 2, (int)p.gs_n * 2};
    const T *Q = !REV ? tensor[0] : dk ? tensor[2] : tensor[1], *K = !REV ? tensor[1] : dk ? tensor[3] : tensor[0];
    const T *V = (!REV ? tensor[2] : dk ? tensor[0] : tensor[3]) + vh * D;
    const int qs2 = !REV ? row_bytes[0] : dk ? row_bytes[2] : row_bytes[1], ks2 = !REV ? row_bytes[1] : dk ? row_bytes[3] : row_bytes[0];
    const int vs2 = !REV ? row_bytes[2] : dk ? row_bytes[0] : row_bytes[3];
    T *O = (!REV ? static_cast<T *>(p.o) + b * p.os_b + h * p.os_h
                 : dk ? static_cast<T *>(p.dk) + b * p.dks_b + h * p.dks_h : static_cast<T *>(p.dv) + b * p.dvs_b + h * p.dvs_h) + vh * D;
    const int os2 = (int)(!REV ? p.os_n : dk ? p.dks_n : p.dvs_n) * 2;
    const u32x4 rq0 = make_rsrc(Q, (uint32_t)((N - 1) * qs2 + p.wqk * 2));
    const u32x4 rk0 = make_rsrc(K, (uint32_t)((N - 1) * ks2 + p.wqk * 2));
    const u32x4 rq1 = make_rsrc(Q + D, (uint32_t)((N - 1) * qs2 + wx2 * 2));
    const u32x4 rk1 = make_rsrc(K + D, (uint32_t)((N - 1) * ks2 + wx2 * 2));
    const u32x4 rv = make_rsrc(V, (uint32_t)((N - 1) * vs2 + wv * 2));
    const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(O, 0, (N - 1) * os2 + wv * 2, 0x00020000);

    // (rows of the second half's state that are padding: the readers take all of them)
    auto zero_rest = [&](float *out) {
        if constexpr (N2 < 4)
            for (int e = 32 * N2 * D + 4 * tid; e < D * D; e += 1024) *reinterpret_cast<u32x4 *>(out + e) = u32x4{0u, 0u, 0u, 0u};
    };
    f32x16 st0[W::NBW], st1[W::NBW];
    if (p.init_is_totals) {
        const int64_t at = (int64_t)ss.bh * p.n_seg * (D * D);
        const int f_lo = REV ? sl.seg + 1 : 0, f_hi = REV ? p.n_seg : sl.seg;
        if constexpr (NV == 2) {  // (both halves' loads in flight together; with four blocks per wave and state, one half's)
            walk_sum_two<D, B, B2>(p.init + at, init2 + at, f_lo, f_hi, wave, lane, st0, st1);
        } else {
            walk_sum_states<D, B, false>(p.init + at, f_lo, f_hi, wave, lane, st0);
            walk_sum_states<D, B2, false>(init2 + at, f_lo, f_hi, wave, lane, st1);
        }
        if constexpr (REV) {
            // (dK's totals are [q/k][v] too: a second half of v that is narrow is so in their columns, and in rows once they are turned.  One
            // map of blocks to waves for both, as B2 would be, leaves rows unsummed and turns what the LDS held there)
            static_assert(NV == 4 && N2 == 4, "whole states are turned");
            if (dk) {
                float *const turn = reinterpret_cast<float *>(smem);
                walk_transpose_state<D, B>(turn, wave, lane, st0);
                walk_transpose_state<D, B>(turn, wave, lane, st1);
            }
        }
        if (!REV && p.entry_out && sl.seg > 0) {  // (the first segment's entry state, zero, is read by nobody)
            walk_write_state<D, B>(p.entry_out + at + (int64_t)sl.seg * (D * D), wave, lane, st0);
            walk_write_state<D, B2>(p.entry_out2 + at + (int64_t)sl.seg * (D * D), wave, lane, st1);
            zero_rest(p.entry_out2 + at + (int64_t)sl.seg * (D * D));
        }
    } else {
        walk_load_init_from<D, B>(p.init, p, ss, wave, lane, st0, REV, transposed);
        walk_load_init_from<D, B2>(init2, p, ss, wave, lane, st1, REV, transposed);
    }
    walk_state_to_lds<T, D, B>(tl, wave, lane, st0);

    auto load_half = [&](int c, auto half) {  // Q_h, K_h of chunk c to set h
        constexpr int HF = decltype(half)::value;
        const uint32_t base = lds0 + HF * 2 * W::TILE;
        walk_load_tile<D>(HF ? rq1 : rq0, base, c * W::C, qs2, HF ? wx2 : p.wqk, wave, lane);
        walk_load_tile<D>(HF ? rk1 : rk0, base + W::TILE, c * W::C, ks2, HF ? wx2 : p.wqk, wave, lane);
    };
    const int c_first = REV ? sl.c_hi - 1 : sl.c_lo;
    auto v_slot = [&](int c) { return 4 + ((c - c_first) & 1); };
    auto load_v = [&](int c) { walk_load_tile<D>(rv, lds0 + v_slot(c) * W::TILE, c * W::C, vs2, wv, wave, lane); };
    auto sync = [&]() {  // this wave's LDS accesses are done; then every wave's
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0xc07f);
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    auto sfrag = [&](int db, int kc) -> V8 { return walk_row_frag<T, D>(tl, 32 * db + walk_e_lane(l32), kc, g); };
    load_half(c_first, std::integral_constant<int, 0>{});
    load_v(c_first);
#pragma unroll 1
    for (int i = 0; i < sl.c_hi - sl.c_lo; ++i) {
        const int c = REV ? c_first - i : c_first + i, c_next = REV ? c - 1 : c + 1;
        const bool others = REV ? c + 1 < p.n_chunks : c > 0;  // chunks under the state exist: it is not identically zero
        unsigned char *tq0 = smem, *tk0 = smem + W::TILE, *tq1 = smem + 2 * W::TILE, *tk1 = smem + 3 * W::TILE;
        unsigned char *tv = smem + v_slot(c) * W::TILE;
        const int row = c * W::C + 32 * rb + l32;
        f32x16 acc[W::DBW];
        // first half.  (Every wave has left the barrier that ended the reads of the set loaded next, one
        // half-chunk ago.)  This wave's loads of the half-chunk have landed when at most the loads issued
        // after them are outstanding; the stores of the chunk before were issued before those.
        load_half(c, std::integral_constant<int, 1>{});
        wait_vm<2 * W::NI>();
        sync();  // the tiles have landed, S_0 is in LDS
        walk_product<T, D, REV, 0, B::KQ, NV>(tq0, tk0, tv, wave, lane, others, sfrag, acc);
        walk_update<T, D, B>(tk0, tv, wave, lane, st0);
        sync();  // every wave has read S_0 and this half's tiles
        walk_state_to_lds<T, D, B2>(tl, wave, lane, st1);
        // second half
        const bool more = i + 1 < sl.c_hi - sl.c_lo;
        if (more) {
            load_half(c_next, std::integral_constant<int, 0>{});
            load_v(c_next);  // (to the slot of the chunk before this one)
            wait_vm<3 * W::NI>();
        } else {
            wait_vm<0>();
        }
        sync();  // the tiles have landed, S_1 is in LDS
        walk_product<T, D, REV, 0, B2::KQ, NV, true>(tq1, tk1, tv, wave, lane, others, sfrag, acc);
        walk_store<T, D, OB::PER>(ro, os2, wv, row, g, db0, acc);
        walk_update<T, D, B2>(tk1, tv, wave, lane, st1);
        sync();  // every wave has read S_1, this half's tiles and V
        walk_state_to_lds<T, D, B>(tl, wave, lane, st0);
    }
    if (!REV && p.total_out && sl.c_hi == p.n_chunks) {  // the states after the last chunk, for the backward walk
        walk_write_state<D, B>(p.total_out + (int64_t)ss.bh * (D * D), wave, lane, st0);
        walk_write_state<D, B2>(p.total_out2 + (int64_t)ss.bh * (D * D), wave, lane, st1);
        zero_rest(p.total_out2 + (int64_t)ss.bh * (D * D));
        // (NV = 2: the v blocks beyond stay unwritten -- walk_bwd_rev_wide_kernel, the reader, is built for the same extent)
    }
}

// (QUAD: a q / k and a v that are both wider than 128 columns, by at most 32 N2: the second half of the result is as narrow.  Looked up in
// the other launches, the halves of v cost 256 / 64, B H 64, N 4096 up to 2 % of a step.  Second halves of one and two blocks, forward +
// backward, all four -> this: 160 / 160, B H 32, N 3968 313 -> 267 us, B H 8, N 28156 552 -> 488, B H 260, N 192 157 -> 137; 160 / 128, B H 32,
// N 4096 207 -> 199; 160 / 64 133.5 -> 130; 192 / 128 206 -> 200)
template <typename T, int NV, int N2 = 4, bool QUAD = false>
__global__ __launch_bounds__(256, 1) void walk_fwd_wide_kernel(const WalkParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (QUAD && N2 < 4) {
        if (blockIdx.y == 1) {
            walk_wide_body<T, 2, false, N2, QUAD>(p);
            return;
        }
    }
    walk_wide_body<T, NV, false, N2, QUAD>(p);
#else
    (void)p;
#endif
}
// dV and dK of a q / k and a v that are both wider than 128 columns
template <typename T>
__global__ __launch_bounds__(256, 1) void walk_rev_wide_kernel(const WalkParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
    walk_wide_body<T, 4, true, 4, true>(p);
#else
    (void)p;
#endif
}

// ---- backward: dQ, dV, dK of a chunk from one set of tiles; R += Q_c^T dO_c, chunks descending.
// dQ's state, the sum of K^T V over the chunks before: the 16-bit copy forward saved at the entry of every chunk
// (WalkParams::saved), brought to LDS with the chunk's tiles.  With the normaliser's terms (NORM), whose vectors leave room for
// one state: dQ first, then R in its place, for two barriers more.  (dQ's state as fragments straight from memory, which
// forward then wrote element by element, spilled 64 bytes a lane: B H 64, N 4096, D 64 71 us, this way 59.)
// (Obtained backwards instead -- from the state at the segment's end, subtracting every chunk's K^T V when the walk reaches
// it -- one late row that is infinite, NaN or merely huge spoiled the dQ of every chunk before it.  Forward + backward
// at B H 16, N 32768, D 64 that way 222 us, this way 234 at the time, 222 with totals added up by fragments.)
// fp16, plain: R's copy is scaled, as forward's (walk_state_scale); the waves exchange their largest elements through a tile that has been
// multiplied, between two barriers more per chunk -- tiles and states fill half of a CU's LDS.  fp16 calls that took this walk unscaled before
// (LinearAttentionChunked, feature maps) pay 2 to 3 % at 64 columns: B H 64, N 4000 100 -> 102 us, with a feature map 119 -> 122; 32 columns and those
// of walk_dkdv_kernel 0 to 1 %.
template <typename T, int D, bool NORM, bool WIDE = false, bool GN = false>
__global__ __launch_bounds__(256, 2) void walk_bwd_kernel(const WalkParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
    using W = WalkCfg<D>;
    using V8 = typename Mma<T>::V8;
    static_assert(W::NCH == 1, "the fused backward keeps dQ's state fragments of all output blocks in registers");
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)smem;
    unsigned char *tq = smem, *tk = smem + W::TILE, *tv = smem + 2 * W::TILE, *tg = smem + 3 * W::TILE,
                  *tl = smem + 4 * W::TILE;
    unsigned char *tx = tl + W::STATE;  // (!NORM) dQ's state; (NORM) the chunk's vectors
    // (NORM: zc, rc, dn of the chunk, and the waves' parts of rc's next term)
    const float *vz = reinterpret_cast<const float *>(tl + W::STATE), *vd = vz + 512;
    float *vr = reinterpret_cast<float *>(tl + W::STATE) + 256, *rpart = vr + 512;
    const uint32_t xbase = lds0 + 4 * W::TILE + W::STATE;
    const int tid = threadIdx.x;
    int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const WalkSlice sl = walk_slice(p);
    if (!sl.valid) return;
    const int b = sl.bh / p.H, h = sl.bh - b * p.H, N = p.N;
    const T *Q = static_cast<const T *>(p.q) + b * p.qs_b + h * p.qs_h;
    const T *K = static_cast<const T *>(p.k) + b * p.ks_b + h * p.ks_h;
    const T *V = static_cast<const T *>(p.v) + b * p.vs_b + h * p.vs_h;
    const T *G = static_cast<const T *>(p.go) + b * p.gs_b + h * p.gs_h;
    const int qs2 = (int)p.qs_n * 2, ks2 = (int)p.ks_n * 2, vs2 = (int)p.vs_n * 2, gs2 = (int)p.gs_n * 2;
    const u32x4 rq = make_rsrc(Q, (uint32_t)((N - 1) * qs2 + p.wqk * 2));
    const u32x4 rk = make_rsrc(K, (uint32_t)((N - 1) * ks2 + p.wqk * 2));
    const u32x4 rv = make_rsrc(V, (uint32_t)((N - 1) * vs2 + p.wv * 2));
    const u32x4 rg = make_rsrc(G, (uint32_t)((N - 1) * gs2 + p.wv * 2));
    const WalkResult rdq(p.dq, b * p.dqs_b + h * p.dqs_h, p.dqs_n, p.wqk, N, WIDE);
    const WalkResult rdk(p.dk, b * p.dks_b + h * p.dks_h, p.dks_n, p.wqk, N, WIDE);
    const WalkResult rdv(p.dv, b * p.dvs_b + h * p.dvs_h, p.dvs_n, p.wv, N, WIDE);

    f32x16 st[W::NBW];  // R[q/k index][v index]
    walk_load_init<D>(p, sl, wave, lane, st, true);
    constexpr bool SCALED = walk_fwd_scaled<T, NORM, false>;
    float sback = 1.f;
    auto publish_state = [&]() {  // (no wave reads the tiles, and no load is on its way to them)
        if constexpr (SCALED) {
            float *smax = reinterpret_cast<float *>(tq);
            walk_state_max<D, WalkExt<D>>(smax, wave, lane, st);
            __syncthreads();
            const float scale = walk_state_scale(smax, sback);
            walk_state_to_lds<T, D>(tl, wave, lane, st, scale);
            __syncthreads();
        } else {
            walk_state_to_lds<T, D>(tl, wave, lane, st);
        }
    };
    if constexpr (!NORM) publish_state();
    float rrun = 0.f;  // NORM: rc (of column tid, tid < D); at the segment's entry from the segments' totals, as zc in forward
    if constexpr (NORM) {
        constexpr int G = 256 / D;
        float t = 0.f;
        if (p.rc) {
            const float *rs = p.rc + (int64_t)sl.bh * p.n_seg * D + tid % D;
            const int lo = p.n_seg == 2 ? (sl.seg ? 2 : 0) : sl.seg + 1;
#pragma unroll 8
            for (int f = lo + tid / D; f < p.n_seg; f += G) t += rs[(int64_t)f * D];
        }
        rpart[tid] = t;
        __syncthreads();
        if (tid < D) {
#pragma unroll
            for (int u = 0; u < G; ++u) rrun += rpart[u * D + tid];
            vr[tid] = rrun;
        }
    }

#pragma unroll 1
    for (int c = sl.c_hi - 1; c >= sl.c_lo; --c) {
        // (NORM, WIDE: LDS addresses that depend on the lane alone would be computed ahead of the loop and held in registers, to the
        // point of spilling)
        if constexpr (NORM && WIDE) asm volatile("" : "+v"(lane));
        const int l32 = lane & 31, g = lane >> 5;
        const int row0 = c * W::C;
        const int64_t at = (int64_t)sl.bh * p.n_chunks + c;
        walk_load_tile<D>(rq, lds0, row0, qs2, p.wqk, wave, lane);
        walk_load_tile<D>(rk, lds0 + W::TILE, row0, ks2, p.wqk, wave, lane);
        walk_load_tile<D>(rv, lds0 + 2 * W::TILE, row0, vs2, p.wv, wave, lane);
        walk_load_tile<D>(rg, lds0 + 3 * W::TILE, row0, gs2, p.wv, wave, lane);
        if constexpr (NORM) {  // the normaliser's terms: zc of this chunk and its rows of dn
            walk_load_vec<D>(p.zc + ((int64_t)sl.bh * p.n_chunks + c) * D, xbase, lane);
            walk_load_rows<D>(p.dn + (int64_t)sl.bh * N, row0, N, xbase + 2048, lane);
            if constexpr (GN) walk_load_rows<D>(p.gn + (int64_t)sl.bh * N, row0, N, xbase + 2560, lane);
        }
        if (c > 0)
            walk_load_state_copy<D>(static_cast<const unsigned char *>(p.saved) + at * W::STATE, NORM ? lds0 + 4 * W::TILE : xbase, wave,
                                    lane);
        wait_vm<0>();
        __syncthreads();
        if constexpr (NORM) {
            if constexpr (GN) {  // dO = g / n, as walk_grad_totals_kernel rounds it
                const float *vn = vd + 128;
#pragma unroll
                for (int v = 0; v < W::C * W::CR / 256; ++v) {
                    const int u = tid + 256 * v, r = u / W::CR, pos = u % W::CR;
                    if (row0 + r < N && (pos ^ walk_swizzle<W::CR>(r)) * 8 < p.wv) {
                        u32x4 *ptr = reinterpret_cast<u32x4 *>(tg + r * W::RB + (pos << 4));
                        V8 x = __builtin_bit_cast(V8, *ptr);
                        const float inv = 1.0f / vn[r];
#pragma unroll
                        for (int e = 0; e < 8; ++e) x[e] = static_cast<T>(static_cast<float>(x[e]) * inv);
                        *ptr = __builtin_bit_cast(u32x4, x);
                    }
                }
                __syncthreads();
            }
        }
        const int row = row0 + 32 * wave + l32;
        const bool later = c + 1 < p.n_chunks;  // chunks after this one exist: R is not identically zero
        const float sx = SCALED && p.saved_scale && c > 0 ? p.saved_scale[at] : 1.f;
        f32x16 acc[W::DBW];
        if constexpr (NORM) {
            // dQ = lower(dO V^T) K + dO S_c^T  (normaliser: scores + dn_i, result + dn_i zc)
            float ax = vd[32 * wave + l32];
            walk_product<T, D, false, 2>(tg, tv, tk, wave, lane, c > 0, [&](int db, int kc) -> V8 {
                return walk_col_frag_perm<T, D>(tl, 16 * kc, db, lane, true);
            }, acc, &ax);
            walk_add_vec<D>(acc, ax, vz, 0, g);
            walk_store<T, D>(rdq.rs, rdq.stride, p.wqk, row, g, 0, acc, p.fmap, tq, 32 * wave + l32, WIDE);
            __syncthreads();  // every wave has read dQ's state
            walk_state_to_lds<T, D>(tl, wave, lane, st);
            __syncthreads();
        }
        // dV = upper(K Q^T) dO + K R: A operand R^T[v index][q/k index] = the LDS copy as it is
        walk_product<T, D, true, 0, W::KC, W::DB, false, SCALED>(tk, tq, tg, wave, lane, later, [&](int db, int kc) -> V8 {
            return walk_row_frag<T, D>(tl, 32 * db + walk_e_lane(l32), kc, g);
        }, acc, nullptr, nullptr, WalkNoRows{}, sback);
        walk_store<T, D>(rdv.rs, rdv.stride, p.wv, row, g, 0, acc, 0, nullptr, 0, WIDE);
        // dK = upper(V dO^T) Q + V R^T: A operand R[q/k index][v index] = the LDS copy read transposed
        // (normaliser: scores + dn_i with i the dO row, result + rc)
        if constexpr (NORM) {
            walk_product<T, D, true, 3>(tv, tg, tq, wave, lane, later, [&](int db, int kc) -> V8 {
                return walk_col_frag_perm<T, D>(tl, 16 * kc, db, lane, true);
            }, acc, nullptr, nullptr, [&](int s, int a) -> f32x4 {
                return *reinterpret_cast<const f32x4 *>(vd + 32 * s + 8 * a + 4 * g);
            });
            walk_add_vec<D>(acc, 1.0f, vr, 0, g);
        } else {
            walk_product<T, D, true, 0, W::KC, W::DB, false, SCALED>(tv, tg, tq, wave, lane, later, [&](int db, int kc) -> V8 {
                return walk_col_frag_perm<T, D>(tl, 16 * kc, db, lane, true);
            }, acc, nullptr, nullptr, WalkNoRows{}, sback);
        }
        walk_store<T, D>(rdk.rs, rdk.stride, p.wqk, row, g, 0, acc, p.fmap, tk, 32 * wave + l32, WIDE);
        if constexpr (!NORM) {
            // dQ = lower(dO V^T) K + dO S_c^T: A operand S_c[q/k index][v index], its LDS copy read transposed
            walk_product<T, D, false, 0, W::KC, W::DB, false, SCALED>(tg, tv, tk, wave, lane, c > 0, [&](int db, int kc) -> V8 {
                return walk_col_frag_perm<T, D>(tx, 16 * kc, db, lane, true);
            }, acc, nullptr, nullptr, WalkNoRows{}, sx);
            walk_store<T, D>(rdq.rs, rdq.stride, p.wqk, row, g, 0, acc, p.fmap, tq, 32 * wave + l32, WIDE);
        }
        walk_update<T, D>(tq, tg, wave, lane, st);
        if constexpr (NORM) walk_weighted_sums_to_lds<D>(rpart, wave, lane, walk_weighted_sums<T, D>(tq, vd, wave, lane));
        __syncthreads();
        if constexpr (!NORM) {
            publish_state();
        } else {
            if (tid < D) {
                rrun += walk_col_sum_of<D>(rpart, tid);
                vr[tid] = rrun;
            }
        }
    }
#else
    (void)p;
#endif
}

// ---- backward without saved per-chunk states, dV and dK: chunks descending, R += Q_c^T dO_c.  One
// workgroup per CU with two sets of tiles: the loads of the next chunk are in flight while this
// one is multiplied.  (dQ is a walk_fwd_kernel launch over dO, V, K.)
// NORM: dK with the normaliser's terms (scores + dn_i, i the dO row; result + rc).  Tiles and state fill the LDS at
// D = 128, so the chunk's dn comes as ordinary loads, a chunk ahead, in the order in which the scores' registers take it, and
// rc is carried in registers: a wave adds up its own output columns, in the order of an MFMA's A rows, and one MFMA
// per 32 columns adds rc to the result (walk_split3).
// fp16, plain: R's copy is scaled, as forward's (walk_state_scale).  With two sets of tiles and the state the LDS is full at D = 128: the waves
// exchange their largest elements through the set of tiles that has just been multiplied, behind a barrier more per chunk, and the next
// loads into that set go out behind the barrier that follows.
template <typename T, int D, bool NORM, int NQ = D / 32, int NV = D / 32, bool WIDE = false, bool ROWS = false, bool ROLES = false>
__global__ __launch_bounds__(256, 1) void walk_dkdv_kernel(const WalkParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
    using W = WalkCfg<D>;
    using V8 = typename Mma<T>::V8;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)smem;
    unsigned char *tl = smem + 8 * W::TILE;
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    using B = WalkExt<D, NQ, NV>;   // R [q/k index][v index]
    using OV = WalkOut<D, NV>;      // dV is as wide as v,
    using OQ = WalkOut<D, NQ>;      // dK as q and k
    static_assert(!NORM || (NQ == W::DB && NV == W::DB), "the normaliser's variant is built for full widths");
    const int rb = W::NCH == 1 ? wave : wave % W::NRB, db0 = OQ::db0(wave);  // (db0: dK's, and rc's columns)
    static_assert(!ROLES || !NORM, "one result of a plain walk");
    const WalkSlice sl = walk_slice(p);
    if (!sl.valid) return;
    constexpr bool SCALED = walk_fwd_scaled<T, NORM, false>;
    const bool with_dv = !ROLES || blockIdx.y == 0, with_dk = !ROLES || blockIdx.y != 0;
    constexpr int n_tiles = ROLES ? 3 : 4;
    const int b = sl.bh / p.H, h = sl.bh - b * p.H, N = p.N;
    const T *Q = static_cast<const T *>(p.q) + b * p.qs_b + h * p.qs_h;
    const T *K = static_cast<const T *>(p.k) + b * p.ks_b + h * p.ks_h;
    const T *V = static_cast<const T *>(p.v) + b * p.vs_b + h * p.vs_h;
    const T *G = static_cast<const T *>(p.go) + b * p.gs_b + h * p.gs_h;
    const int qs2 = (int)p.qs_n * 2, ks2 = (int)p.ks_n * 2, vs2 = (int)p.vs_n * 2, gs2 = (int)p.gs_n * 2;
    const u32x4 rq = make_rsrc(Q, (uint32_t)((N - 1) * qs2 + p.wqk * 2));
    const u32x4 rk = make_rsrc(K, (uint32_t)((N - 1) * ks2 + p.wqk * 2));
    const u32x4 rv = make_rsrc(V, (uint32_t)((N - 1) * vs2 + p.wv * 2));
    const u32x4 rg = make_rsrc(G, (uint32_t)((N - 1) * gs2 + p.wv * 2));
    const WalkResult rdk(p.dk, b * p.dks_b + h * p.dks_h, p.dks_n, p.wqk, N, WIDE);
    const WalkResult rdv(p.dv, b * p.dvs_b + h * p.dvs_h, p.dvs_n, p.wv, N, WIDE);
    const WalkAnyRows<T> adk(p.rows_dk, b, h, 0, p.rows_dk.width, N), adv(p.rows_dv, b, h, 0, p.rows_dv.width, N);

    f32x16 st[W::NBW];  // R[q/k index][v index]
    walk_load_init<D, B>(p, sl, wave, lane, st, true);
    float sback = 1.f;
    // (`dead`: tiles that nobody reads and no load is on its way to)
    auto publish_state = [&](unsigned char *dead) {
        if constexpr (SCALED) {
            float *smax = reinterpret_cast<float *>(dead);
            walk_state_max<D, B>(smax, wave, lane, st);
            __builtin_amdgcn_s_waitcnt(0xc07f);
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            const float scale = walk_state_scale(smax, sback);
            walk_state_to_lds<T, D, B>(tl, wave, lane, st, scale);
        } else {
            walk_state_to_lds<T, D, B>(tl, wave, lane, st);
        }
    };
    publish_state(smem + 4 * W::TILE);

    auto load_chunk = [&](int c, int buf) {
        const uint32_t base = lds0 + buf * 4 * W::TILE;
        const int row0 = c * W::C;
        walk_load_tile<D>(rq, base, row0, qs2, p.wqk, wave, lane);
        if (with_dv) walk_load_tile<D>(rk, base + W::TILE, row0, ks2, p.wqk, wave, lane);
        if (with_dk) walk_load_tile<D>(rv, base + 2 * W::TILE, row0, vs2, p.wv, wave, lane);
        walk_load_tile<D>(rg, base + 3 * W::TILE, row0, gs2, p.wv, wave, lane);
    };
    static_assert(!NORM || W::C == 64, "eight groups of four dn values are a chunk of 64 rows");
    // Ordinary loads, requested a chunk ahead (once the tiles of the chunk before have been awaited) and
    // read at the top of their chunk, BEFORE the next tile loads go out: the wait the compiler puts
    // in front of the first use is one for every outstanding load and store (it cannot count past
    // stores), and at that point nothing is in flight that the walk would not wait for anyway but the
    // previous chunk's stores, issued two products earlier.
    f32x4 nxt_dn[8];
    // (whole groups of four rows: up to three values past the sequence's end, of the next head or of the scratch behind dn, are
    // read and dropped below; groups past the end read as zero.  Without the normaliser the descriptor is never used)
    const __amdgpu_buffer_rsrc_t rs_dn = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(NORM ? p.dn + (int64_t)sl.bh * N : nullptr), 0, NORM ? (N + 3) / 4 * 16 : 0, 0x00020000);
    auto load_vecs = [&](int c) {  // dn of rows 8 a + 4 g .. of chunk c
        if constexpr (NORM) {
#pragma unroll
            for (int a = 0; a < 8; ++a)
                nxt_dn[a] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs_dn, (c * W::C + 8 * a + 4 * g) * 4, 0, 0));
        }
    };
    // rc of column 32 (db0 + i) + walk_e_lane(l32), at the segment's entry from the segments' totals: the part of every other
    // row (g) or segment that this lane adds up -- the lane of the other g holds the rest
    float rrun[W::DBW];
#pragma unroll
    for (int i = 0; i < W::DBW; ++i) rrun[i] = 0.f;
    if constexpr (NORM) {
        if (p.rc) {
            const float *rs = p.rc + (int64_t)sl.bh * p.n_seg * D + 32 * db0 + walk_e_lane(l32);
            const int lo = p.n_seg == 2 ? (sl.seg ? 2 : 0) : sl.seg + 1;
#pragma unroll 4
            for (int f = lo + g; f < p.n_seg; f += 2)
#pragma unroll
                for (int i = 0; i < W::DBW; ++i) rrun[i] += rs[(int64_t)f * D + 32 * i];
        }
    }
    load_chunk(sl.c_hi - 1, 0);
    load_vecs(sl.c_hi - 1);
#pragma unroll 1
    for (int c = sl.c_hi - 1; c >= sl.c_lo; --c) {
        const int buf = (sl.c_hi - 1 - c) & 1;
        unsigned char *tq = smem + buf * 4 * W::TILE, *tk = tq + W::TILE, *tv = tq + 2 * W::TILE, *tg = tq + 3 * W::TILE;
        const bool more = c > sl.c_lo;
        f32x4 dnv[8];  // dn of tile rows 8 a + 4 g ..
        if constexpr (NORM) {
#pragma unroll
            for (int a = 0; a < 8; ++a) {
                dnv[a] = nxt_dn[a];
                asm volatile("" : "+v"(dnv[a])::"memory");  // (awaited before the tile loads below)
            }
            if ((c + 1) * W::C > N) {
#pragma unroll
                for (int a = 0; a < 8; ++a)
#pragma unroll
                    for (int b4 = 0; b4 < 4; ++b4) dnv[a][b4] = c * W::C + 8 * a + 4 * g + b4 < N ? dnv[a][b4] : 0.f;
            }
        }
        if (!SCALED && more) load_chunk(c - 1, buf ^ 1);  // (every wave has left the barrier that ended the reads of that set)
        // this wave's loads of chunk c have landed when at most the loads issued after them are
        // outstanding (the stores of the previous chunk were issued before those)
        if (!SCALED && more)
            wait_vm<n_tiles * W::NI>();
        else
            wait_vm<0>();
        if constexpr (NORM) {
            if (more) load_vecs(c - 1);
        }
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's part of the state is in LDS
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (SCALED && more) load_chunk(c - 1, buf ^ 1);  // (every wave has read the largest elements there)
        const int row = c * W::C + 32 * rb + l32;
        const bool later = c + 1 < p.n_chunks;  // chunks after this one exist: R is not identically zero
        f32x16 acc[W::DBW];
        if (with_dv) {
            // dV = upper(K Q^T) dO + K R: A operand R^T[v index][q/k index] = the LDS copy as it is
            walk_product<T, D, true, 0, B::KQ, NV, false, SCALED>(tk, tq, tg, wave, lane, later, [&](int db, int kc) -> V8 {
                return walk_row_frag<T, D>(tl, 32 * db + walk_e_lane(l32), kc, g);
            }, acc, nullptr, nullptr, WalkNoRows{}, sback);
            if constexpr (ROWS)
                adv.template store<D, OV::PER>(row, g, OV::db0(wave), acc);
            else
                walk_store<T, D, OV::PER>(rdv.rs, rdv.stride, p.wv, row, g, OV::db0(wave), acc, 0, nullptr, 0, WIDE);
        }
        if (with_dk) {
            // dK = upper(V dO^T) Q + V R^T: A operand R[q/k index][v index] = the LDS copy read transposed
            if constexpr (NORM) {
                walk_product<T, D, true, 3>(tv, tg, tq, wave, lane, later, [&](int db, int kc) -> V8 {
                    return walk_col_frag_perm<T, D>(tl, 16 * kc, db, lane, true);
                }, acc, nullptr, nullptr, [&](int s, int a4) -> f32x4 { return s == 0 ? dnv[a4] : dnv[4 + a4]; });
                const Mma<__bf16>::V8 ones = walk_ones3(g);
#pragma unroll
                for (int i = 0; i < W::DBW; ++i)
                    acc[i] = Mma<__bf16>::mma(walk_split3(rrun[i] + __shfl_xor(rrun[i], 32, 64), g), ones, acc[i]);
            } else {
                walk_product<T, D, true, 0, B::KV, NQ, false, SCALED>(tv, tg, tq, wave, lane, later, [&](int db, int kc) -> V8 {
                    return walk_col_frag_perm<T, D>(tl, 16 * kc, db, lane, true);
                }, acc, nullptr, nullptr, WalkNoRows{}, sback);
            }
            if constexpr (ROWS)
                adk.template store<D, OQ::PER>(row, g, db0, acc);
            else
                walk_store<T, D, OQ::PER>(rdk.rs, rdk.stride, p.wqk, row, g, db0, acc, p.fmap, tk, 32 * rb + l32, WIDE);
        }
        walk_update<T, D, B>(tq, tg, wave, lane, st);
        if constexpr (NORM) {  // rc += this chunk's dn_i q_i
            static_for<0, W::C / 16>([&](auto j) {
                constexpr int ks = decltype(j)::value;
#pragma unroll
                for (int i = 0; i < W::DBW; ++i) {
                    const V8 y = walk_col_frag_perm<T, D>(tq, 16 * ks, db0 + i, lane, false);
#pragma unroll
                    for (int e = 0; e < 8; ++e) rrun[i] += dnv[2 * ks + e / 4][e % 4] * static_cast<float>(y[e]);
                }
            });
        }
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0xc07f);  // this wave's LDS reads of the tiles and of the state are done
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        publish_state(tq);
    }
#else
    (void)p;
#endif
}

// ---- backward at D = 128 in one reverse walk: dV, dK and dQ of a chunk from one set of tiles.
//   R = sum of Q^T dO over the chunks after this one, as in walk_dkdv_kernel;
//   X = sum of K^T V over the chunks before it, obtained backwards: X starts as the forward state at
//   the end of the segment (the next segment's entry state, or the state after the last chunk) and
//   every chunk's K^T V is subtracted when the walk reaches it.  (In fp32: the difference carries
//   the rounding of the sums it is taken from, about 1e-7 of the segment's largest state -- below the
//   16-bit rounding the state gets before it multiplies dO unless the rows so far are some 1e4 times smaller
//   than later ones; and a late row that is infinite or NaN leaves nothing of it.)
// The one 16-bit state in LDS holds R for dV and dK, then X for dQ.  q, k, v, dO are read once and
// nothing but the results is written, where the walk for dQ followed by walk_dkdv_kernel reads
// dO, v, k twice.
template <typename T, int D, int NQ = D / 32, int NV = D / 32, bool FM = false, bool WIDE = false, bool ROWS = false>
__global__ __launch_bounds__(256, 1) void walk_bwd_rev_kernel(const WalkParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
    using W = WalkCfg<D>;
    using V8 = typename Mma<T>::V8;
    using B = WalkExt<D, NQ, NV>;   // R, X [q/k index][v index]
    using OV = WalkOut<D, NV>;      // dV is as wide as v,
    using OQ = WalkOut<D, NQ>;      // dK and dQ as q and k
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)smem;
    unsigned char *tl = smem + 8 * W::TILE;
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rb = W::NCH == 1 ? wave : wave % W::NRB;
    const WalkSlice sl = walk_slice(p);
    if (!sl.valid) return;
    const int wqk = p.wqk, wv = p.wv;
    // FM: q and k hold y = phi(x); dQ and dK leave multiplied by the slope of phi, computed from the tiles
    const int fmap = FM ? p.fmap : 0;
    const int b = sl.bh / p.H, h = sl.bh - b * p.H, N = p.N;
    const T *Q = static_cast<const T *>(p.q) + b * p.qs_b + h * p.qs_h;
    const T *K = static_cast<const T *>(p.k) + b * p.ks_b + h * p.ks_h;
    const T *V = static_cast<const T *>(p.v) + b * p.vs_b + h * p.vs_h;
    const T *G = static_cast<const T *>(p.go) + b * p.gs_b + h * p.gs_h;
    const int qs2 = (int)p.qs_n * 2, ks2 = (int)p.ks_n * 2, vs2 = (int)p.vs_n * 2, gs2 = (int)p.gs_n * 2;
    const u32x4 rq = make_rsrc(Q, (uint32_t)((N - 1) * qs2 + wqk * 2));
    const u32x4 rk = make_rsrc(K, (uint32_t)((N - 1) * ks2 + wqk * 2));
    const u32x4 rv = make_rsrc(V, (uint32_t)((N - 1) * vs2 + wv * 2));
    const u32x4 rg = make_rsrc(G, (uint32_t)((N - 1) * gs2 + wv * 2));
    const WalkResult rdq(p.dq, b * p.dqs_b + h * p.dqs_h, p.dqs_n, wqk, N, WIDE);
    const WalkResult rdk(p.dk, b * p.dks_b + h * p.dks_h, p.dks_n, wqk, N, WIDE);
    const WalkResult rdv(p.dv, b * p.dvs_b + h * p.dvs_h, p.dvs_n, wv, N, WIDE);
    const WalkAnyRows<T> adq(p.rows_dq, b, h, 0, p.rows_dq.width, N), adk(p.rows_dk, b, h, 0, p.rows_dk.width, N),
        adv(p.rows_dv, b, h, 0, p.rows_dv.width, N);

    f32x16 st[W::NBW];  // R [q/k index][v index]
    f32x16 xs[W::NBW];  // X [q/k index][v index]
    walk_load_init<D, B>(p, sl, wave, lane, st, true);
    walk_load_end_state<D, B>(p, sl, wave, lane, xs);
    walk_state_to_lds<T, D, B>(tl, wave, lane, st);

    auto load_chunk = [&](int c, int buf) {
        const uint32_t base = lds0 + buf * 4 * W::TILE;
        const int row0 = c * W::C;
        walk_load_tile<D>(rq, base, row0, qs2, wqk, wave, lane);
        walk_load_tile<D>(rk, base + W::TILE, row0, ks2, wqk, wave, lane);
        walk_load_tile<D>(rv, base + 2 * W::TILE, row0, vs2, wv, wave, lane);
        walk_load_tile<D>(rg, base + 3 * W::TILE, row0, gs2, wv, wave, lane);
    };
    auto sync = [&]() {  // this wave's LDS accesses are done; then every wave's
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0xc07f);
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    load_chunk(sl.c_hi - 1, 0);
#pragma unroll 1
    for (int c = sl.c_hi - 1; c >= sl.c_lo; --c) {
        const int buf = (sl.c_hi - 1 - c) & 1;
        unsigned char *tq = smem + buf * 4 * W::TILE, *tk = tq + W::TILE, *tv = tq + 2 * W::TILE, *tg = tq + 3 * W::TILE;
        const bool more = c > sl.c_lo;
        if (more) load_chunk(c - 1, buf ^ 1);  // (every wave has left the barrier that ended the reads of that set)
        // this wave's loads of chunk c have landed when at most the loads issued after them are
        // outstanding (the stores of the previous chunk were issued before those)
        if (more)
            wait_vm<4 * W::NI>();
        else
            wait_vm<0>();
        sync();  // the tiles have landed, R is in LDS
        const int row = c * W::C + 32 * rb + l32;
        const bool later = c + 1 < p.n_chunks;  // chunks after this one exist: R is not identically zero
        walk_update<T, D, B, true, true>(tk, tv, wave, lane, xs);  // X: now the sum over the chunks before this one
        f32x16 acc[W::DBW];
        // dV = upper(K Q^T) dO + K R: A operand R^T[v index][q/k index] = the LDS copy as it is
        walk_product<T, D, true, 0, B::KQ, NV>(tk, tq, tg, wave, lane, later, [&](int db, int kc) -> V8 {
            return walk_row_frag<T, D>(tl, 32 * db + walk_e_lane(l32), kc, g);
        }, acc);
        if constexpr (ROWS)
            adv.template store<D, OV::PER>(row, g, OV::db0(wave), acc);
        else
            walk_store<T, D, OV::PER>(rdv.rs, rdv.stride, wv, row, g, OV::db0(wave), acc, 0, nullptr, 0, WIDE);
        // dK = upper(V dO^T) Q + V R^T: A operand R[q/k index][v index] = the LDS copy read transposed
        walk_product<T, D, true, 0, B::KV, NQ>(tv, tg, tq, wave, lane, later, [&](int db, int kc) -> V8 {
            return walk_col_frag_perm<T, D>(tl, 16 * kc, db, lane, true);
        }, acc);
        if constexpr (ROWS)
            adk.template store<D, OQ::PER>(row, g, OQ::db0(wave), acc);
        else
            walk_store<T, D, OQ::PER>(rdk.rs, rdk.stride, wqk, row, g, OQ::db0(wave), acc, fmap, tk, 32 * rb + l32, WIDE);
        // R += Q^T dO touches registers and tiles only, so it can sit on either side of the barriers: the waves of
        // the last row block, with one score block in dV and dK against two, take it here, the others after dQ,
        // where they have one score block against two
        // (full widths only: with a narrow v side the balance is the other way round, measured)
        constexpr bool kSplitUpdate = W::NRB == 2 && NQ == W::DB && NV == W::DB;
        if (kSplitUpdate && rb == 1) walk_update<T, D, B, false, true>(tq, tg, wave, lane, st);
        sync();  // every wave has read R
        // (X stays in its accumulation registers up to here: without this the copies that the rounding
        // below reads are made right after the update and occupy 64 registers through both products)
        if constexpr (B::SLOTS == 4)
            asm volatile("" : "+a"(xs[0]), "+a"(xs[1]), "+a"(xs[2]), "+a"(xs[3]));
        else
            asm volatile("" : "+a"(xs[0]), "+a"(xs[1]));
        walk_state_to_lds<T, D, B>(tl, wave, lane, xs);
        sync();  // X is in LDS
        // dQ = lower(dO V^T) K + dO X^T: A operand X[q/k index][v index], read transposed like R for dK
        walk_product<T, D, false, 0, B::KV, NQ>(tg, tv, tk, wave, lane, c > 0, [&](int db, int kc) -> V8 {
            return walk_col_frag_perm<T, D>(tl, 16 * kc, db, lane, true);
        }, acc);
        if constexpr (ROWS)
            adq.template store<D, OQ::PER>(row, g, OQ::db0(wave), acc);
        else
            walk_store<T, D, OQ::PER>(rdq.rs, rdq.stride, wqk, row, g, OQ::db0(wave), acc, fmap, tq, 32 * rb + l32, WIDE);
        if (!(kSplitUpdate && rb == 1)) walk_update<T, D, B, false, true>(tq, tg, wave, lane, st);
        sync();  // every wave has read X and is done with the tiles
        walk_state_to_lds<T, D, B>(tl, wave, lane, st);
    }
#else
    (void)p;
#endif
}

// ---- the reverse walk for q and k of 129 .. 256 columns against a v of at most 128: one walk over
// both 128-column halves.  Per chunk and half h, with R_h and X_h the states of walk_bwd_rev_kernel for the half:
//   dV  += upper(K_h Q_h^T) dO + K_h R_h        (fp32 accumulators from the first half to the second, stored once)
//   dK_h = upper(V dO^T) Q_h + V R_h^T
//   WITH_DQ: dQ_h = lower(dO V^T) K_h + dO X_h^T     (otherwise dQ_h is a walk_fwd_kernel launch of its own)
// V and dO are loaded once per chunk.  (A walk per half, the second adding its part of dV to the first one's in memory,
// loaded them twice and rounded that part of dV once more.)
// LDS as in walk_fwd_wide_kernel: a set of (Q_h, K_h) tiles per half, two (V, dO) pairs by chunk parity, and ONE
// 16-bit state that holds R_h, then X_h, of the half at work; at the end of a half-chunk the other half's R (in
// registers throughout) is rounded into it.  With dQ four states in registers: built for v blocks NV = 2 only.
template <typename T, int NV, bool WITH_DQ, bool WIDE = false, bool ROWS = false>
__global__ __launch_bounds__(256, 1) void walk_bwd_rev_wide_kernel(const WalkParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int D = 128, NQ = D / 32;
    static_assert(!WITH_DQ || NV == 2, "R and X of both halves live in registers: two blocks per wave and state");
    using W = WalkCfg<D>;
    using V8 = typename Mma<T>::V8;
    using B = WalkExt<D, NQ, NV>;   // R, X [q/k index][v index]
    using OV = WalkOut<D, NV>;      // dV is as wide as v,
    using OQ = WalkOut<D, NQ>;      // dK and dQ as q and k
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)smem;
    unsigned char *tl = smem + 8 * W::TILE;
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rb = wave % W::NRB;
    const WalkSlice sl = walk_slice(p);
    if (!sl.valid) return;
    const int b = sl.bh / p.H, h = sl.bh - b * p.H, N = p.N;
    const T *Q = static_cast<const T *>(p.q) + b * p.qs_b + h * p.qs_h;
    const T *K = static_cast<const T *>(p.k) + b * p.ks_b + h * p.ks_h;
    const T *V = static_cast<const T *>(p.v) + b * p.vs_b + h * p.vs_h;
    const T *G = static_cast<const T *>(p.go) + b * p.gs_b + h * p.gs_h;
    const int qs2 = (int)p.qs_n * 2, ks2 = (int)p.ks_n * 2, vs2 = (int)p.vs_n * 2, gs2 = (int)p.gs_n * 2;
    const u32x4 rq0 = make_rsrc(Q, (uint32_t)((N - 1) * qs2 + p.wqk * 2));
    const u32x4 rk0 = make_rsrc(K, (uint32_t)((N - 1) * ks2 + p.wqk * 2));
    const u32x4 rq1 = make_rsrc(Q + D, (uint32_t)((N - 1) * qs2 + p.wqk2 * 2));
    const u32x4 rk1 = make_rsrc(K + D, (uint32_t)((N - 1) * ks2 + p.wqk2 * 2));
    const u32x4 rv = make_rsrc(V, (uint32_t)((N - 1) * vs2 + p.wv * 2));
    const u32x4 rg = make_rsrc(G, (uint32_t)((N - 1) * gs2 + p.wv * 2));
    const int64_t dq_at = b * p.dqs_b + h * p.dqs_h, dk_at = b * p.dks_b + h * p.dks_h;
    const WalkResult rdq0(p.dq, dq_at, p.dqs_n, p.wqk, N, WIDE), rdq1(p.dq, dq_at + D, p.dqs_n, p.wqk2, N, WIDE);
    const WalkResult rdk0(p.dk, dk_at, p.dks_n, p.wqk, N, WIDE), rdk1(p.dk, dk_at + D, p.dks_n, p.wqk2, N, WIDE);
    const WalkAnyRows<T> adk0(p.rows_dk, b, h, 0, D, N), adk1(p.rows_dk, b, h, D, p.rows_dk.width - D, N);
    const WalkResult rdv(p.dv, b * p.dvs_b + h * p.dvs_h, p.dvs_n, p.wv, N, WIDE);

    f32x16 st0[W::NBW], st1[W::NBW];  // R_0, R_1
    f32x16 xs0[W::NBW], xs1[W::NBW];  // X_0, X_1
    if (p.init_is_totals) {
        const int64_t at = (int64_t)sl.bh * p.n_seg * (D * D);
        if constexpr (NV == 2) {
            walk_sum_two<D, B>(p.init + at, p.init2 + at, sl.seg + 1, p.n_seg, wave, lane, st0, st1);
        } else {
            walk_sum_states<D, B>(p.init + at, sl.seg + 1, p.n_seg, wave, lane, st0);
            walk_sum_states<D, B>(p.init2 + at, sl.seg + 1, p.n_seg, wave, lane, st1);
        }
    } else {
        walk_load_init_from<D, B>(p.init, p, sl, wave, lane, st0, true, p.init_transposed != 0);
        walk_load_init_from<D, B>(p.init2, p, sl, wave, lane, st1, true, p.init_transposed != 0);
    }
    if constexpr (WITH_DQ) {
        walk_load_end_state_from<D, B>(p.xinit, p.xtotal, p, sl, wave, lane, xs0);
        walk_load_end_state_from<D, B>(p.xinit2, p.xtotal2, p, sl, wave, lane, xs1);
    }
    walk_state_to_lds<T, D, B>(tl, wave, lane, st0);

    auto load_half = [&](int c, auto half) {  // Q_h, K_h of chunk c to set h
        constexpr int HF = decltype(half)::value;
        const uint32_t base = lds0 + HF * 2 * W::TILE;
        walk_load_tile<D>(HF ? rq1 : rq0, base, c * W::C, qs2, HF ? p.wqk2 : p.wqk, wave, lane);
        walk_load_tile<D>(HF ? rk1 : rk0, base + W::TILE, c * W::C, ks2, HF ? p.wqk2 : p.wqk, wave, lane);
    };
    auto vg_slot = [&](int c) { return 4 + 2 * ((sl.c_hi - 1 - c) & 1); };
    auto load_vg = [&](int c) {
        const uint32_t base = lds0 + vg_slot(c) * W::TILE;
        walk_load_tile<D>(rv, base, c * W::C, vs2, p.wv, wave, lane);
        walk_load_tile<D>(rg, base + W::TILE, c * W::C, gs2, p.wv, wave, lane);
    };
    auto sync = [&]() {  // this wave's LDS accesses are done; then every wave's
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0xc07f);
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    // A operands of the state products: R^T[v index][q/k index] is the LDS copy as it is (dV); R and X
    // [q/k index][v index] are the copy read transposed (dK, dQ)
    auto rows_of_state = [&](int db, int kc) -> V8 { return walk_row_frag<T, D>(tl, 32 * db + walk_e_lane(l32), kc, g); };
    auto cols_of_state = [&](int db, int kc) -> V8 { return walk_col_frag_perm<T, D>(tl, 16 * kc, db, lane, true); };
    load_half(sl.c_hi - 1, std::integral_constant<int, 0>{});
    load_vg(sl.c_hi - 1);
#pragma unroll 1
    for (int c = sl.c_hi - 1; c >= sl.c_lo; --c) {
        unsigned char *tv = smem + vg_slot(c) * W::TILE, *tg = tv + W::TILE;
        const int row = c * W::C + 32 * rb + l32;
        const bool later = c + 1 < p.n_chunks;  // chunks after this one exist: R is not identically zero
        f32x16 dvacc[W::DBW];
        auto half_chunk = [&](auto half, f32x16 (&st)[W::NBW], f32x16 (&xs)[W::NBW], f32x16 (&st_next)[W::NBW]) {
            constexpr int HF = decltype(half)::value;
            unsigned char *tq = smem + HF * 2 * W::TILE, *tk = tq + W::TILE;
            // (every wave has left the barrier that ended the reads of the set loaded next, one half-chunk ago.)
            // This wave's loads of the half-chunk have landed when at most the loads issued after them are
            // outstanding; the stores of the half-chunk before were issued before those.
            if constexpr (HF == 0) {
                load_half(c, std::integral_constant<int, 1>{});
                wait_vm<2 * W::NI>();
            } else {
                if (c > sl.c_lo) {
                    load_half(c - 1, std::integral_constant<int, 0>{});
                    load_vg(c - 1);  // (to the slots of the chunk after this one)
                    wait_vm<4 * W::NI>();
                } else {
                    wait_vm<0>();
                }
            }
            sync();  // the tiles have landed, R_h is in LDS
            if constexpr (WITH_DQ) walk_update<T, D, B, true, true>(tk, tv, wave, lane, xs);  // X_h: now the sum over the chunks before this one
            walk_product<T, D, true, 0, B::KQ, NV, HF != 0>(tk, tq, tg, wave, lane, later, rows_of_state, dvacc);
            f32x16 acc[W::DBW];
            walk_product<T, D, true, 0, B::KV, NQ>(tv, tg, tq, wave, lane, later, cols_of_state, acc);
            if constexpr (ROWS)
                (HF ? adk1 : adk0).template store<D, OQ::PER>(row, g, OQ::db0(wave), acc);
            else
                walk_store<T, D, OQ::PER>((HF ? rdk1 : rdk0).rs, rdk0.stride, HF ? p.wqk2 : p.wqk, row, g, OQ::db0(wave), acc, 0, nullptr, 0, WIDE);
            if constexpr (WITH_DQ) {
                sync();  // every wave has read R_h
                // (X stays in its accumulation registers up to here: without this the copies that the rounding
                // below reads are made right after the update and occupy registers through both products)
                asm volatile("" : "+a"(xs[0]), "+a"(xs[1]));
                walk_state_to_lds<T, D, B>(tl, wave, lane, xs);
                sync();  // X_h is in LDS
                walk_product<T, D, false, 0, B::KV, NQ>(tg, tv, tk, wave, lane, c > 0, cols_of_state, acc);
                walk_store<T, D, OQ::PER>((HF ? rdq1 : rdq0).rs, rdq0.stride, HF ? p.wqk2 : p.wqk, row, g, OQ::db0(wave), acc, 0, nullptr, 0, WIDE);
            }
            if constexpr (HF != 0) walk_store<T, D, OV::PER>(rdv.rs, rdv.stride, p.wv, row, g, OV::db0(wave), dvacc, 0, nullptr, 0, WIDE);
            walk_update<T, D, B, false, true>(tq, tg, wave, lane, st);  // R_h += Q_h^T dO
            sync();  // every wave has read the state's copy and is done with this half's tiles
            walk_state_to_lds<T, D, B>(tl, wave, lane, st_next);
        };
        half_chunk(std::integral_constant<int, 0>{}, st0, xs0, st1);
        half_chunk(std::integral_constant<int, 1>{}, st1, xs1, st0);
    }
#else
    (void)p;
#endif
}

// ---- segment totals: totals[bh][seg] = sum over the segment's rows of Y^T Z, fp32 [D][D]
struct WalkTotalsParams {
    const void *y, *z;
    int64_t ys_b, ys_h, ys_n, zs_b, zs_h, zs_n;
    int32_t H, N, BH, dy, dz;
    int32_t n_chunks, seg_chunks, n_seg;
    int32_t seg_lo, seg_hi;  // only segments seg_lo .. seg_hi - 1 are needed (the others' totals stay unwritten)
    float *totals;
    // two segments: only the total of segment seg_lo is needed, as the other segment's entry state.
    // The kernel writes it in the layout the walks read (see walk_load_init) -- `totals` is where
    // the entry states go -- and no scan follows.
    int32_t direct;
    // feature map on load: Y holds the argument of the map; every Y tile is mapped in LDS as it lands
    // and the mapped rows are written to ymap_out (Y's shape, element strides yo_*).  0: none.
    int32_t map_y;
    void *ymap_out;
    int64_t yo_b, yo_h, yo_n;
    // A second Y operand of the same layout against the same Z, in the same launch: the other 128-column half
    // of a wide q / k, whose totals go to `totals2`.  Null: none.  (Without a feature map.)  Every workgroup takes both.
    const void *y2;
    int32_t dy2;
    float *totals2;
    int32_t pairs;  // with dz2: walk_totals_pairs_kernel
    // walk_totals_quad_kernel: true width of Z's second half (its columns 128 ..), 0: Z has one half.  The totals of
    // (Y half i, Z half j) are matrices (2 j + i) BH n_seg .. of `totals` (totals2 = totals + BH n_seg D D).
    int32_t dz2;
    // The totals of Y's rows, fp32 [BH][n_seg][D], in the slots of `totals` -- the normaliser's running sum of k at the
    // segments' entries (WalkParams::vsum); null: not formed.  One operand only.
    float *vsum;
    // the totals are written by fragments (walk_write_frags): the walks add them up as they start
    int32_t frags;
    int32_t alone;  // of a forward that hands no states over (walk_whole_parts)
    // nobody reads the totals' columns 64 .. (every walk behind them leaves a narrow z's padding out): they may stay
    // unwritten for a narrow y as well
    int32_t z_narrow;
    int32_t place;  // (as in WalkParams; at the far end, where they bring in the rest of the parameters' lines together with n_seg)
    uint32_t n_seg_inv;
};

constexpr int walk_totals_sets(int D) { return D == 128 ? 4 : 2; }  // sets of (Y, Z) tiles in LDS

// BOTH (D = 128): the launch's two Y operands (WalkTotalsParams::y2) in ONE workgroup -- three sets of (Y, Y2, Z) tiles, a
// state per operand -- so that Z is loaded once for the two.  256 / 128, forward + backward, a workgroup per operand -> this:
// B H 64, N 4096 430 -> 420 us; B H 32, N 2048 178 -> 168 us.
template <typename T, int D, int NQ, int NV, bool BOTH, bool PAIRS = false>
__device__ __forceinline__ void walk_totals_body(const WalkTotalsParams &p) {
    using W = WalkCfg<D>;
    static_assert(!BOTH || D == 128, "halves of 128 columns");
    // (the halves of Z and of Y: walk_totals_quad_kernel, walk_totals_pairs_kernel -- grid y there is 2 (half of Y) + half of Z; elsewhere & ~0, no
    // instruction)
    const int zh = (BOTH || PAIRS) && p.dz2 ? (int)blockIdx.y & (PAIRS ? 1 : ~0) : 0, dz = zh ? p.dz2 : p.dz;
    const bool yh = PAIRS && blockIdx.y >= 2;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)smem;
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const XcdItem item = xcd_item(blockIdx.x, p.BH, p.n_seg, p.place, p.n_seg_inv);
    const int bh = item.bh, seg = item.part;
    if (bh < 0) return;
    const int dy = yh ? p.dy2 : p.dy;
    int64_t out_at;
    int c_lo, c_hi;
    if (p.direct) {
        // both workgroups of a (b, h) at work: half of the needed segment's chunks each (with a feature map
        // every row has to be visited: the needed segment's workgroup forms its total alone, the other one
        // maps its own segment's rows and hands in zeros)
        const int needed = p.seg_lo, part = seg != needed;
        out_at = ((int64_t)bh * 2 + part) * (D * D);
        c_lo = seg * p.seg_chunks;
        c_hi = c_lo + p.seg_chunks < p.n_chunks ? c_lo + p.seg_chunks : p.n_chunks;
        if (!p.map_y) {
            const int n_lo = needed * p.seg_chunks;
            const int n_hi = n_lo + p.seg_chunks < p.n_chunks ? n_lo + p.seg_chunks : p.n_chunks;
            const int mid = n_lo + (n_hi - n_lo + 1) / 2;
            c_lo = part ? mid : n_lo, c_hi = part ? n_hi : mid;
        }
    } else {
        if (seg < p.seg_lo || seg >= p.seg_hi) return;
        out_at = ((int64_t)bh * p.n_seg + seg) * (D * D);
        c_lo = seg * p.seg_chunks;
        c_hi = c_lo + p.seg_chunks < p.n_chunks ? c_lo + p.seg_chunks : p.n_chunks;
    }
    out_at += (int64_t)2 * zh * p.BH * p.n_seg * (D * D);
    float *const out = (yh ? p.totals2 : p.totals) + out_at;
    float *const out2 = BOTH ? p.totals2 + out_at : nullptr;
    if (c_lo >= c_hi) {  // nothing to add up (a segment beyond the end of the sequence, the second half of one chunk)
        for (int i = tid; i < D * D; i += 256) {
            out[i] = 0.f;
            if constexpr (BOTH) out2[i] = 0.f;
        }
        if (p.vsum && tid < D) p.vsum[out_at / D + tid] = 0.f;
        return;
    }
    const bool discard = p.direct && p.map_y && seg != p.seg_lo;  // (visited for the map only)
    const int b = bh / p.H, h = bh - b * p.H, N = p.N;
    const T *Y = static_cast<const T *>(yh ? p.y2 : p.y) + b * p.ys_b + h * p.ys_h;
    const T *Y2 = static_cast<const T *>(BOTH ? p.y2 : p.y) + b * p.ys_b + h * p.ys_h;
    const T *Z = static_cast<const T *>(p.z) + b * p.zs_b + h * p.zs_h + zh * D;
    const int ys2 = (int)p.ys_n * 2, zs2 = (int)p.zs_n * 2;
    const u32x4 ry = make_rsrc(Y, (uint32_t)((N - 1) * ys2 + dy * 2));
    const u32x4 ry2 = make_rsrc(Y2, (uint32_t)((N - 1) * ys2 + (BOTH ? p.dy2 : dy) * 2));
    const u32x4 rz = make_rsrc(Z, (uint32_t)((N - 1) * zs2 + dz * 2));
    using B = WalkExt<D, NQ, NV>;  // (blocks outside it stay unwritten: no walk of the same extent reads them)
    f32x16 st[W::NBW], st2[W::NBW], zs;  // (zs: the column sums of Y, with vsum)
#pragma unroll
    for (int v = 0; v < 16; ++v) zs[v] = 0.f;
#pragma unroll
    for (int i = 0; i < W::NBW; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) st[i][v] = 0.f, st2[i][v] = 0.f;
    // SETS sets of tiles.  Two (two workgroups per CU): the loads of chunk c + 1 are in flight while
    // chunk c is multiplied.  More (D = 128, where the grid has at most one workgroup per CU and a
    // workgroup's own chain load -> barrier -> product bounds its rate): SETS - 1 chunks in flight.
    constexpr int SETS = BOTH ? 3 : walk_totals_sets(D), TPS = BOTH ? 3 : 2;  // tiles per set: Y, (Y2,) Z
    auto load_chunk = [&](int c, int set) {
        const uint32_t base = lds0 + set * TPS * W::TILE;
        walk_load_tile<D>(ry, base, c * W::C, ys2, dy, wave, lane);
        if constexpr (BOTH) walk_load_tile<D>(ry2, base + W::TILE, c * W::C, ys2, p.dy2, wave, lane);
        walk_load_tile<D>(rz, base + (TPS - 1) * W::TILE, c * W::C, zs2, dz, wave, lane);
    };
    auto map_tile = [&](unsigned char *ty, int c) {
        walk_map_tile<T, D>(ty, p.map_y, c * W::C, N, dy, static_cast<T *>(p.ymap_out) + b * p.yo_b + h * p.yo_h,
                            p.yo_n, tid);
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the rewritten tile is in LDS
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    if constexpr (SETS == 2) {
        load_chunk(c_lo, 0);
#pragma unroll 1
        for (int c = c_lo; c < c_hi; ++c) {
            const int buf = (c - c_lo) & 1;
            unsigned char *ty = smem + buf * 2 * W::TILE, *tz = ty + W::TILE;
            const bool more = c + 1 < c_hi;
            if (more) load_chunk(c + 1, buf ^ 1);  // (every wave has left the barrier that ended the reads of that set)
            // this wave's loads of chunk c have landed: only those of chunk c + 1 may still be in flight
            // (the mapped rows' stores of a feature map share the counter: then everything is awaited)
            if (more && !p.map_y)
                wait_vm<2 * W::NI>();
            else
                wait_vm<0>();
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            if (p.map_y) map_tile(ty, c);
            walk_update<T, D, B>(ty, tz, wave, lane, st);
            if (p.vsum) walk_col_sums<T, D>(ty, wave, lane, zs);
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(0xc07f);  // this wave's LDS reads of the set are done
            __builtin_amdgcn_s_barrier();
        }
    } else {
        static_assert(SETS == 3 || SETS == 4, "the waits below count up to two chunks behind the awaited one");
#pragma unroll
        for (int i = 0; i < SETS - 1; ++i)
            if (c_lo + i < c_hi) load_chunk(c_lo + i, i);
        int set = 0;
#pragma unroll 1
        for (int c = c_lo; c < c_hi; ++c) {
            unsigned char *ty = smem + set * TPS * W::TILE, *tz = ty + (TPS - 1) * W::TILE;
            // this wave's loads of chunk c have landed: those of up to SETS - 2 later chunks may still be in
            // flight (the mapped rows' stores of a feature map share the counter: then everything is awaited)
            const int behind = c_hi - 1 - c;
            if (p.map_y || behind == 0)
                wait_vm<0>();
            else if (behind == 1 || SETS == 3)
                wait_vm<TPS * W::NI>();
            else
                wait_vm<2 * TPS * W::NI>();
            __builtin_amdgcn_s_waitcnt(0xc07f);  // this wave's LDS reads of the chunk before are done
            __builtin_amdgcn_s_barrier();        // ... and so are every wave's: its set can be loaded over
            asm volatile("" ::: "memory");
            if (c + SETS - 1 < c_hi) load_chunk(c + SETS - 1, (set + SETS - 1) % SETS);
            if (p.map_y) map_tile(ty, c);
            walk_update<T, D, B>(ty, tz, wave, lane, st);
            if constexpr (BOTH) walk_update<T, D, B>(ty + W::TILE, tz, wave, lane, st2);
            if constexpr (!BOTH && NV == W::DB)
                if (p.vsum) walk_col_sums<T, D>(ty, wave, lane, zs);
            asm volatile("" ::: "memory");
            set = (set + 1) % SETS;
        }
    }
    if (p.frags) {
        walk_write_frags<D, B>(out, wave, lane, st);
        if constexpr (BOTH) walk_write_frags<D, B>(out2, wave, lane, st2);
    } else
#pragma unroll
    for (int i = 0; i < B::SLOTS; ++i)
        if (B::valid(wave, i)) {
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int at = (32 * B::dbk(wave, i) + 8 * (v / 4) + 4 * g + (v % 4)) * D + 32 * B::eb(wave) + l32;
                out[at] = discard ? 0.f : st[i][v];
                if constexpr (BOTH) out2[at] = st2[i][v];
            }
        }
    if (p.vsum) {  // (no loads into LDS are in flight any more)
        float *part = reinterpret_cast<float *>(smem);
        __syncthreads();
        walk_col_sums_to_lds<D>(part, wave, lane, zs);
        __syncthreads();
        if (tid < D) p.vsum[out_at / D + tid] = discard ? 0.f : walk_col_sum_of<D>(part, tid);
    }
}

template <typename T, int D, int NQ = D / 32, int NV = D / 32, bool BOTH = false>
__global__ __launch_bounds__(256, BOTH ? 1 : 2) void walk_totals_kernel(const WalkTotalsParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
    walk_totals_body<T, D, NQ, NV, BOTH>(p);
#else
    (void)p;
#endif
}

// Both 128-column halves of Y against a Z of more than 64 columns: a workgroup takes both halves of Y; of a Z wider than 128
// columns grid y picks the half (all four pairs in one launch).
template <typename T>
__global__ __launch_bounds__(256, 1) void walk_totals_quad_kernel(const WalkTotalsParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
    walk_totals_body<T, 128, 4, 4, true>(p);
#else
    (void)p;
#endif
}

// ... one of the four pairs (grid y), for plans of half as many segments: four workgroups to a segment
template <typename T>
__global__ __launch_bounds__(256, 1) void walk_totals_pairs_kernel(const WalkTotalsParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
    walk_totals_body<T, 128, 4, 4, false, true>(p);
#else
    (void)p;
#endif
}

// Entry states of the walk's segments from the segments' totals: entry[bh][s][e] = sum of
// totals[bh][f][e] over f < s (reverse == 0) or f > s (reverse != 0).  Only the totals under those
// sums are read.  entry may be totals (a thread reads an element before it writes it).  One thread
// per pair of elements; the loads of up to sixteen segments are issued together (a chain of
// dependent loads would cost a memory latency each).
// `cols`: only the first `cols` columns of every row of the D-wide states are summed (the totals
// kernel built for a narrow v side writes no others, and no walk of that extent reads them).
// (a template only so that the header can be included by several translation units)
// grid y = 1 scans a second pair of buffers of the same shape (totals_b, entry_b; the other half of a wide q / k).
template <int kUnused = 0>
__global__ __launch_bounds__(256) void walk_scan_kernel(const float *totals, float *entry, int n_seg, int E,
                                                        int64_t total2, int reverse, int D, int cols,
                                                        const float *totals_b, float *entry_b) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    const int64_t i2 = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i2 >= total2) return;
    if (blockIdx.y != 0) totals = totals_b, entry = entry_b;
    const int half = cols / 2;
    const int64_t per_bh = (int64_t)(E / D) * half, bh = i2 / per_bh, r = i2 - bh * per_bh;
    const int64_t e = (r / half) * D + 2 * (r % half);
    const float *pt = totals + bh * n_seg * E + e;
    float *pe = entry + bh * n_seg * E + e;
    const int64_t step = reverse ? -(int64_t)E : (int64_t)E;
    if (reverse) pt += (int64_t)(n_seg - 1) * E, pe += (int64_t)(n_seg - 1) * E;
    f32x2 run = {0.f, 0.f};
    int s = 0;
    auto batch = [&](auto nn) {
        constexpr int NB = decltype(nn)::value;
        for (; s + NB <= n_seg - 1; s += NB) {
            f32x2 t[NB];
#pragma unroll
            for (int u = 0; u < NB; ++u) t[u] = *reinterpret_cast<const f32x2 *>(pt + u * step);
#pragma unroll
            for (int u = 0; u < NB; ++u) {
                *reinterpret_cast<f32x2 *>(pe + u * step) = run;
                run += t[u];
            }
            pt += NB * step, pe += NB * step;
        }
    };
    batch(std::integral_constant<int, 16>{});
    batch(std::integral_constant<int, 4>{});
    batch(std::integral_constant<int, 1>{});
    *reinterpret_cast<f32x2 *>(pe) = run;  // the last segment in walking order: its own total is not needed
}

// ---- per-chunk column sums: out[bh][c][col] = sum over the rows of chunk c of y[row][col]; fp32.  A scan over the chunks
// (walk_vec_scan_kernel) then gives zc where forward's is not at hand (a backward at D = 128 without forward's state).
struct WalkVecParams {
    const void *y;
    int64_t ys_b, ys_h, ys_n;
    int32_t H, N, width, n_chunks;
    float *out;      // [BH][n_chunks][D]
};

template <typename T, int D>
__global__ __launch_bounds__(256) void walk_vec_sums_kernel(const WalkVecParams p) {
    using W = WalkCfg<D>;
    using V8 = typename Mma<T>::V8;
    constexpr int SLOTS = 256 / W::CR;  // rows visited at a time
    __shared__ float part[SLOTS][D];
    const int tid = threadIdx.x, pos = tid % W::CR, slot = tid / W::CR;
    const int c = blockIdx.x, bh = blockIdx.y, b = bh / p.H, h = bh - b * p.H;
    const T *Y = static_cast<const T *>(p.y) + b * p.ys_b + h * p.ys_h;
    float acc[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = 0.f;
    if (pos * 8 < p.width) {
#pragma unroll 4
        for (int r = slot; r < W::C; r += SLOTS) {
            const int row = c * W::C + r;
            if (row < p.N) {
                const V8 y = __builtin_bit_cast(V8, *reinterpret_cast<const u32x4 *>(Y + (int64_t)row * p.ys_n + pos * 8));
#pragma unroll
                for (int e = 0; e < 8; ++e) acc[e] += static_cast<float>(y[e]);
            }
        }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) part[slot][pos * 8 + e] = acc[e];
    __syncthreads();
    if (tid < D) {
        float t = 0.f;
#pragma unroll
        for (int u = 0; u < SLOTS; ++u) t += part[u][tid];
        p.out[((int64_t)bh * p.n_chunks + c) * D + tid] = t;
    }
}

// ---- exclusive prefix sums over the chunks of the vectors above, in place: v[bh][c][col] <- sum of v[bh][c'][col] over
// c' < c.  There are few columns and many
// chunks, so the chunks of a (b, h) are split over sixteen thread groups: each adds up its range,
// the ranges' sums are scanned in LDS, and each group writes its range's running sums.
// (a template only so that the header can be included by several translation units)
template <int kUnused = 0>
__global__ __launch_bounds__(256) void walk_vec_scan_kernel(float *v, int n_chunks, int D) {
    __shared__ float part[16][16];
    const int j = threadIdx.x & 15, grp = threadIdx.x >> 4;  // column within the block's 16, range of chunks
    const int bh = blockIdx.y, col = blockIdx.x * 16 + j;
    const int per = (n_chunks + 15) / 16;
    float *base = v + (int64_t)bh * n_chunks * D + col;
    const int t0 = grp * per, t1 = t0 + per < n_chunks ? t0 + per : n_chunks;
    float sum = 0.f;
    for (int t = t0; t < t1; t += 8) {
        float x[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) x[u] = t + u < t1 ? base[(int64_t)(t + u) * D] : 0.f;
#pragma unroll
        for (int u = 0; u < 8; ++u) sum += x[u];
    }
    part[grp][j] = sum;
    __syncthreads();
    float run = 0.f;
    for (int g2 = 0; g2 < grp; ++g2) run += part[g2][j];
    for (int t = t0; t < t1; t += 8) {
        float x[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) x[u] = t + u < t1 ? base[(int64_t)(t + u) * D] : 0.f;
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (t + u < t1) {
                base[(int64_t)(t + u) * D] = run;
                run += x[u];
            }
    }
}

inline hipError_t launch_walk_vec_scan(float *v, int64_t BH, int n_chunks, int D, hipStream_t stream) {
    if (BH > 65535 || D % 16 != 0) return hipErrorInvalidConfiguration;
    return launch_kernel<walk_vec_scan_kernel<0>>(dim3((unsigned)(D / 16), (unsigned)BH), dim3(256), 0, stream, v, n_chunks,
                         D);
}

template <typename T, int D>
hipError_t launch_walk_vec_sums(const WalkVecParams &p, int64_t BH, hipStream_t stream) {
    if (BH > 65535) return hipErrorInvalidConfiguration;
    return launch_kernel<walk_vec_sums_kernel<T, D>>(dim3((unsigned)p.n_chunks, (unsigned)BH), dim3(256), 0, stream, p);
}

// ---- the normalised backward's first pass: dO = g / n and dn = -(g . out) / n (contiguous, for the walks behind it), and from
// them, while they are in LDS, every segment's totals of Q^T dO -- walk_totals_kernel's -- and of dn_i q_i.
// Bound by memory: g, out and dO once each and the needed segments' q.  As passes of their own (dO and dn, totals, per-chunk
// vectors and their scan, each reading q or dO again) B H 64, N 4096, D 64 took 42 us, this way 25 (134 MB: 5.4 TB/s); B H 16,
// N 8192, D 128 48 -> 33 us.
struct WalkGradParams {
    const void *q, *go, *o;
    int64_t qs_b, qs_h, qs_n, gs_b, gs_h, gs_n, os_b, os_h, os_n;
    const float *denom;        // n, fp32 [BH][N]
    void *dout;                // dO: contiguous rows of wv elements
    float *dn;                 // fp32 [BH][N]
    int32_t H, N, BH, wqk, wv;
    int32_t vec;               // g and out allow 16-byte loads
    int32_t n_chunks, seg_chunks, n_seg;
    float *totals, *rsum;      // [BH][n_seg] states and vectors in the slots the walks read (two segments: partial sums of the
                               // second one's in both; the first one's stay unwritten otherwise); null with a single segment
    int32_t frags;             // WalkTotalsParams::frags
    int32_t keep_g;            // dO is formed again by the walk behind (WalkParams::gn) and not written
    int32_t place;             // (as in WalkTotalsParams)
    uint32_t n_seg_inv;
};

// Steps on their way: what a step needs is requested DEPTH steps ahead -- one where two workgroups share a CU, two at D = 128,
// where one workgroup has it (one there: 36 us in place of 33 at B H 16, N 8192).
// VEC: g and out allow 16-byte loads.
constexpr int walk_grad_depth(int D) { return D == 128 ? 2 : 1; }

template <typename T, int D, bool VEC>
__global__ __launch_bounds__(256, D == 128 ? 1 : 2) void walk_grad_totals_kernel(const WalkGradParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
    using W = WalkCfg<D>;
    using V8 = typename Mma<T>::V8;
    constexpr int PIECES = W::C * W::CR / 256;  // 16-byte pieces of a tile per thread
    constexpr int DEPTH = walk_grad_depth(D), QT = DEPTH + 1;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)smem;
    float *vd = reinterpret_cast<float *>(smem + (QT + 2) * W::TILE);  // QT tiles of Q, two of dO, two of dn
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const XcdItem item = xcd_item(blockIdx.x, p.BH, p.n_seg, p.place, p.n_seg_inv);
    const int bh = item.bh, seg = item.part;
    if (bh < 0) return;
    // the chunks whose sums are wanted, [a_lo, a_hi), and those that are visited for dO and dn alone, from b_lo on.  Two
    // segments: both workgroups of a (b, h) take one half of either segment
    int a_lo = seg * p.seg_chunks, a_hi = a_lo + p.seg_chunks < p.n_chunks ? a_lo + p.seg_chunks : p.n_chunks;
    int b_lo = a_lo, b_hi = a_lo;
    if (p.n_seg == 2) {
        const int first = p.seg_chunks, mid = first + (p.n_chunks - first + 1) / 2;
        a_lo = seg ? mid : first, a_hi = seg ? p.n_chunks : mid;
        b_lo = seg ? (first + 1) / 2 : 0, b_hi = seg ? first : (first + 1) / 2;
    } else if (seg == 0) {
        b_hi = a_hi, a_hi = a_lo;
    }
    const int n_a = a_hi - a_lo, n_all = n_a + b_hi - b_lo;
    auto chunk_of = [&](int i) { return i < n_a ? a_lo + i : b_lo + i - n_a; };
    const int b = bh / p.H, h = bh - b * p.H, N = p.N;
    const T *Q = static_cast<const T *>(p.q) + b * p.qs_b + h * p.qs_h;
    const T *G = static_cast<const T *>(p.go) + b * p.gs_b + h * p.gs_h;
    const T *O = static_cast<const T *>(p.o) + b * p.os_b + h * p.os_h;
    const float *den = p.denom + (int64_t)bh * N;
    T *dO = static_cast<T *>(p.dout) + (int64_t)bh * N * p.wv;
    float *dn = p.dn + (int64_t)bh * N;
    const int qs2 = (int)p.qs_n * 2;
    const u32x4 rq = make_rsrc(Q, (uint32_t)((N - 1) * qs2 + p.wqk * 2));
    f32x16 st[W::NBW];
    float zs = 0.f;
#pragma unroll
    for (int i = 0; i < W::NBW; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) st[i][v] = 0.f;
    const int col = 8 * (tid % W::CR), r0 = tid / W::CR;  // of piece u: row r0 + u 256 / CR of the chunk
    u32x4 gw[DEPTH][PIECES], ow[DEPTH][PIECES];
    float nw[DEPTH][PIECES];
    int q_next = 0;  // the Q tile of the next request
    auto request = [&](int i, auto set) {  // step i: q to its tile, the other operands to registers (rows past the end: the last one)
        constexpr int S = decltype(set)::value;
        const int row0 = chunk_of(i) * W::C;
        if (i < n_a) walk_load_tile<D>(rq, lds0 + q_next * W::TILE, row0, qs2, p.wqk, wave, lane);
        q_next = q_next + 1 == QT ? 0 : q_next + 1;
#pragma unroll
        for (int u = 0; u < PIECES; ++u) {
            const int row = row0 + r0 + u * (256 / W::CR), at = row < N ? row : N - 1;
            gw[S][u] = load8(G + (int64_t)at * p.gs_n, true, col, p.wv, VEC);
            ow[S][u] = load8(O + (int64_t)at * p.os_n, true, col, p.wv, VEC);
            nw[S][u] = den[at];
        }
    };
    static_for<0, DEPTH>([&](auto set) {
        if (decltype(set)::value < n_all) request(decltype(set)::value, set);
    });
    int q_at = 0;
    auto step = [&](int i, auto set) {
        constexpr int S = decltype(set)::value;
        const int row0 = chunk_of(i) * W::C;
        unsigned char *tq = smem + q_at * W::TILE, *tg = smem + (QT + (i & 1)) * W::TILE;
        q_at = q_at + 1 == QT ? 0 : q_at + 1;
        float *vdn = vd + (i & 1) * W::C;
        // what was requested for this step has arrived: at most the next step's requests, which follow the stores of the step
        // before, are out
        if constexpr (DEPTH == 1) {
            wait_vm<0>();
        } else {
            if (i + 1 < n_a)
                wait_vm<W::NI + 3 * PIECES>();
            else if (i + 1 < n_all)
                wait_vm<3 * PIECES>();
            else
                wait_vm<0>();
        }
#pragma unroll
        for (int u = 0; u < PIECES; ++u) {
            const int r = r0 + u * (256 / W::CR), row = row0 + r;
            const bool ok = row < N;
            const V8 a = __builtin_bit_cast(V8, gw[S][u]), o8 = __builtin_bit_cast(V8, ow[S][u]);
            const float inv = 1.0f / nw[S][u];
            float dot = 0.f;
            V8 d8;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                dot += static_cast<float>(a[e]) * static_cast<float>(o8[e]);
                d8[e] = static_cast<T>(static_cast<float>(a[e]) * inv);
            }
#pragma unroll
            for (int d = 1; d < W::CR; d <<= 1) dot += __shfl_xor(dot, d, 64);
            u32x4 w = __builtin_bit_cast(u32x4, d8);
#pragma unroll
            for (int e = 0; e < 4; ++e) w[e] = ok ? w[e] : 0u;
            *reinterpret_cast<u32x4 *>(tg + r * W::RB + (((tid % W::CR) ^ walk_swizzle<W::CR>(r)) << 4)) = w;
            if (tid % W::CR == 0) vdn[r] = ok ? -dot * inv : 0.f;
            if (ok) {
                if (col < p.wv && !p.keep_g) *reinterpret_cast<u32x4 *>(dO + (int64_t)row * p.wv + col) = w;
                if (tid % W::CR == 0) dn[row] = -dot * inv;
            }
        }
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's part of dO and dn is in LDS, its reads of the step before are done
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (i + DEPTH < n_all) request(i + DEPTH, set);
        if (i < n_a) {
            walk_update<T, D>(tq, tg, wave, lane, st);
            zs += walk_weighted_sums<T, D>(tq, vdn, wave, lane);
        }
    };
#pragma unroll 1
    for (int i = 0; i < n_all; i += DEPTH)
        static_for<0, DEPTH>([&](auto set) {
            if (i + decltype(set)::value < n_all) step(i + decltype(set)::value, set);
        });
    if (p.n_seg == 1 || (p.n_seg > 2 && seg == 0)) return;
    const int64_t at = (int64_t)bh * p.n_seg + seg;
    if (p.frags)
        walk_write_frags<D, WalkExt<D>>(p.totals + at * (D * D), wave, lane, st);
    else
        walk_write_state<D, WalkExt<D>>(p.totals + at * (D * D), wave, lane, st);
    float *part = reinterpret_cast<float *>(smem);
    __syncthreads();
    walk_weighted_sums_to_lds<D>(part, wave, lane, zs);
    __syncthreads();
    if (tid < D) p.rsum[at * D + tid] = walk_col_sum_of<D>(part, tid);
#else
    (void)p;
#endif
}

template <typename T, int D>
hipError_t launch_walk_grad_totals(const WalkGradParams &p, hipStream_t stream) {
    const int64_t grid = (int64_t)8 * ((p.BH + 7) / 8) * p.n_seg;
    if (grid > 0x7fffffffLL) return hipErrorInvalidConfiguration;
    if (p.n_seg > 1 && (!p.totals || !p.rsum)) return hipErrorInvalidValue;
    constexpr int smem = (walk_grad_depth(D) + 3) * WalkCfg<D>::TILE + 2 * WalkCfg<D>::C * 4;
    if (p.vec) {
        constexpr auto kern = walk_grad_totals_kernel<T, D, true>;
        if (hipError_t e = ensure_dynamic_lds<kern>(smem)) return e;
        return launch_kernel<kern>(dim3((unsigned)grid), dim3(256), smem, stream, p);
    }
    constexpr auto kern = walk_grad_totals_kernel<T, D, false>;
    if (hipError_t e = ensure_dynamic_lds<kern>(smem)) return e;
    return launch_kernel<kern>(dim3((unsigned)grid), dim3(256), smem, stream, p);
}

// columns of the D x D totals that walk_totals_kernel writes for operands of true widths dy, dz (the
// variant without the padding blocks of a narrow z leaves the others unwritten)
inline int walk_totals_cols(int D, int dy, int dz) { return D == 128 && dy > 64 && dz <= 64 ? 64 : D; }

template <typename T, int D>
hipError_t launch_walk_totals(const WalkTotalsParams &p, hipStream_t stream) {
    const int64_t grid = (int64_t)8 * ((p.BH + 7) / 8) * p.n_seg;
    if (grid > 0x7fffffffLL) return hipErrorInvalidConfiguration;
    constexpr int smem = walk_totals_sets(D) * 2 * WalkCfg<D>::TILE;
    if (p.direct && (p.n_seg != 2 || p.seg_lo < 0 || p.seg_lo > 1 || p.frags)) return hipErrorInvalidValue;
    // (a second operand runs the same kernel variant: the caller pairs operands of one kind only)
    if (p.y2 && (p.map_y || !p.totals2 ||
                 (!p.z_narrow && walk_totals_cols(D, p.dy2, p.dz) != walk_totals_cols(D, p.dy, p.dz))))
        return hipErrorInvalidValue;
    if (p.vsum && (p.y2 || p.dz2 || (D == 128 && walk_totals_cols(D, p.dy, p.dz) == 64))) return hipErrorInvalidValue;
    if (p.y2 || p.dz2 || p.z_narrow) {
        if (D != 128 || (p.dz2 && (!p.y2 || p.dy != 128 || p.dz != 128 || p.dz2 < 1 || p.dz2 > 128 || p.z_narrow)) ||
            (p.z_narrow && p.dz > 64))
            return hipErrorInvalidValue;
    }
    const dim3 g((unsigned)grid);
    if constexpr (D == 128) {
        constexpr int smem_both = 3 * 3 * WalkCfg<D>::TILE;
        const bool narrow = p.z_narrow || walk_totals_cols(D, p.dy, p.dz) == 64;
        if (p.dz2 && p.pairs) {
            constexpr auto kern = walk_totals_pairs_kernel<T>;
            if (hipError_t e = ensure_dynamic_lds<kern>(smem)) return e;
            return launch_kernel<kern>(dim3((unsigned)grid, 4u), dim3(256), smem, stream, p);
        }
        if (p.dz2 || (p.y2 && !narrow)) {
            constexpr auto kern = walk_totals_quad_kernel<T>;
            if (hipError_t e = ensure_dynamic_lds<kern>(smem_both)) return e;
            return launch_kernel<kern>(dim3((unsigned)grid, p.dz2 ? 2u : 1u), dim3(256), smem_both, stream, p);
        }
        if (p.y2 && narrow) {  // ... and both operands in one workgroup: z loaded once
            constexpr auto kern = walk_totals_kernel<T, D, 4, 2, true>;
            if (hipError_t e = ensure_dynamic_lds<kern>(smem_both)) return e;
            return launch_kernel<kern>(dim3((unsigned)grid), dim3(256), smem_both, stream, p);
        }
        if (narrow) {  // z of at most 64 true columns: the state's other v blocks hold zeros
            constexpr auto kern = walk_totals_kernel<T, D, 4, 2>;
            if (hipError_t e = ensure_dynamic_lds<kern>(smem)) return e;
            return launch_kernel<kern>(g, dim3(256), smem, stream, p);
        }
    }
    constexpr auto kern = walk_totals_kernel<T, D>;
    if (hipError_t e = ensure_dynamic_lds<kern>(smem)) return e;
    return launch_kernel<kern>(g, dim3(256), smem, stream, p);
}

inline hipError_t launch_walk_scan(const float *totals, float *entry, int64_t BH, int n_seg, int D, int cols,
                                   int reverse, hipStream_t stream, const float *totals_b = nullptr,
                                   float *entry_b = nullptr) {
    const int E = D * D;
    const int64_t total2 = BH * D * (cols / 2);
    if (n_seg < 1 || cols < 2 || cols > D || cols % 2 || (totals_b != nullptr) != (entry_b != nullptr))
        return hipErrorInvalidValue;
    return launch_kernel<walk_scan_kernel<0>>(dim3((unsigned)((total2 + 255) / 256), totals_b ? 2u : 1u), dim3(256), 0,
                                              stream, totals, entry, n_seg, E, total2, reverse, D, cols, totals_b, entry_b);
}

template <auto kern>
hipError_t launch_walk_kernel(int64_t grid, int smem, const WalkParams &p, hipStream_t stream, int parts = 1) {
    if (hipError_t e = ensure_dynamic_lds<kern>(smem)) return e;
    return launch_kernel<kern>(dim3((unsigned)grid, (unsigned)parts), dim3(256), smem, stream, p);
}

inline bool walk_rows_ok(const WalkRowsOut &o, int most) { return o.ptr && o.width >= 1 && o.width <= most; }

template <typename T, int D, bool WIDE = false, bool ROWS = false>
hipError_t launch_walk_fwd(const WalkParams &p, hipStream_t stream) {
    if constexpr (!ROWS) {
        if (p.any_rows) {
            if constexpr (D == 128 && !WIDE) return launch_walk_fwd<T, D, false, true>(p, stream);
            return hipErrorNotSupported;
        }
    }
    if constexpr (!WIDE) {
        if (p.wide_out) {  // (dQ's walk)
            if constexpr (D == 128 && !ROWS && std::is_same<T, __bf16>::value) return launch_walk_fwd<T, D, true>(p, stream);
            return hipErrorNotSupported;
        }
    }
    constexpr int NB = D / 32;
    const int64_t grid = (int64_t)8 * ((p.BH + 7) / 8) * p.n_seg;
    if (grid > 0x7fffffffLL) return hipErrorInvalidConfiguration;
    constexpr bool kDouble = D > 64;  // (the plan's workgroup count must match: one per CU when double)
    // (walk_fwd_scaled: the waves' largest elements behind the state)
    constexpr int smem = (kDouble ? 6 : 3) * WalkCfg<D>::TILE + WalkCfg<D>::STATE + (walk_fwd_scaled<T, 0, false> ? 16 : 0);
    const bool fm = p.fmap || p.slope_y;
    // (segment totals in place of entry states: the D = 128 walks, by the flag; below that by the number of segments)
    if (p.init_is_totals && (D != 128 || p.n_seg < 3 || !p.init)) return hipErrorInvalidValue;
    if (p.entry_out && (!p.init_is_totals || p.dn || p.slope_y)) return hipErrorInvalidValue;
    if (WIDE && p.denom) return hipErrorInvalidValue;
    if constexpr (ROWS) {
        if (p.denom || p.dn || fm || !walk_rows_ok(p.rows_o, p.wv)) return hipErrorInvalidValue;
    } else if (p.denom || p.dn) {  // the normaliser's terms: its vectors live behind the state
        if ((p.dn && !p.zc) || (p.denom && p.n_seg > 1 && !p.vsum)) return hipErrorInvalidValue;
        constexpr int smem_n = smem + (kDouble ? 2 : 1) * WalkCfg<D>::VEC;
        if constexpr (!WIDE)
            if (p.denom)
                return fm ? launch_walk_kernel<walk_fwd_kernel<T, D, kDouble, 1, true>>(grid, smem_n, p, stream)
                          : launch_walk_kernel<walk_fwd_kernel<T, D, kDouble, 1, false>>(grid, smem_n, p, stream);
        return fm ? launch_walk_kernel<walk_fwd_kernel<T, D, kDouble, 2, true, NB, NB, WIDE>>(grid, smem_n, p, stream)
                  : launch_walk_kernel<walk_fwd_kernel<T, D, kDouble, 2, false, NB, NB, WIDE>>(grid, smem_n, p, stream);
    }
    if constexpr (!ROWS)
        if (fm) return launch_walk_kernel<walk_fwd_kernel<T, D, kDouble, 0, true, NB, NB, WIDE>>(grid, smem, p, stream);
    if (p.cols) {
        if constexpr (D == 128) {
            if (p.denom || p.dn || fm || p.r_totals || p.n_seg != 1 || p.init || p.wqk <= 64 || p.wv <= 64) return hipErrorInvalidValue;
            return launch_walk_kernel<walk_fwd_kernel<T, D, kDouble, 0, false, 4, 2, WIDE, ROWS, false, true>>(grid, smem, p, stream, 2);
        }
        return hipErrorNotSupported;
    }
    if (p.r_totals) {
        if constexpr (D == 128 && std::is_same<T, __bf16>::value) {
            constexpr int smem_r = 8 * WalkCfg<D>::TILE + WalkCfg<D>::STATE;
            static_assert(smem_r <= 160 * 1024, "two sets of four tiles and the state must fit the LDS of a CU");
            if (!p.r_q || p.n_seg < 3 || p.total_out || p.entry_out || p.denom || p.dn || fm) return hipErrorInvalidValue;
            if (p.wqk <= 64 && p.wv > 64) return launch_walk_kernel<walk_fwd_kernel<T, D, kDouble, 0, false, 2, 4, WIDE, ROWS, true>>(grid, smem_r, p, stream);
            if (p.wqk <= 64) return launch_walk_kernel<walk_fwd_kernel<T, D, kDouble, 0, false, 2, 2, WIDE, ROWS, true>>(grid, smem_r, p, stream);
            if (p.wv > 64) return launch_walk_kernel<walk_fwd_kernel<T, D, kDouble, 0, false, 4, 4, WIDE, ROWS, true>>(grid, smem_r, p, stream);
        }
        return hipErrorNotSupported;
    }
    if constexpr (D == 128) {
        // operands of at most 64 true columns on a side (the halves of a wide q / k, a narrow v): the kernels that
        // leave out the blocks of padding, which the states in memory may not hold either
        if (p.wqk > 64 && p.wv <= 64) return launch_walk_kernel<walk_fwd_kernel<T, D, kDouble, 0, false, 4, 2, WIDE, ROWS>>(grid, smem, p, stream);
        if (p.wqk <= 64 && p.wv > 64) return launch_walk_kernel<walk_fwd_kernel<T, D, kDouble, 0, false, 2, 4, WIDE, ROWS>>(grid, smem, p, stream);
        if (p.wqk <= 64 && p.wv <= 64) return launch_walk_kernel<walk_fwd_kernel<T, D, kDouble, 0, false, 2, 2, WIDE, ROWS>>(grid, smem, p, stream);
    }
    return launch_walk_kernel<walk_fwd_kernel<T, D, kDouble, 0, false, NB, NB, WIDE, ROWS>>(grid, smem, p, stream);
}

template <typename T>
hipError_t launch_walk_fwd_wide(const WalkParams &p, hipStream_t stream) {
    if (p.any_rows) return hipErrorNotSupported;
    using W = WalkCfg<128>;
    const int64_t grid = (int64_t)8 * ((p.BH + 7) / 8) * p.n_seg;
    if (grid > 0x7fffffffLL) return hipErrorInvalidConfiguration;
    if (p.wqk != 128 || p.wqk2 < 1 || p.wqk2 > 128 || p.wv < 1 || p.wv > 128 || p.fmap || p.slope_y || p.denom || p.dn ||
        (p.init_transposed && !p.quad) || (p.n_seg > 1 && (!p.init || (!p.quad && !p.init2))) || (p.total_out && !p.total_out2) ||
        (p.init_is_totals && (p.n_seg < 3 || !p.init || (!p.quad && !p.init2) || p.init_transposed)) ||
        (p.entry_out != nullptr) != (p.entry_out2 != nullptr) || (p.entry_out && !p.init_is_totals))
        return hipErrorInvalidValue;
    constexpr int smem = 6 * W::TILE + W::STATE;  // two sets of (Q_h, K_h), two V tiles, one state
    if (p.quad) {
        if (p.quad != 1 || p.wv != 128 || p.wv2 < 1 || p.wv2 > 128) return hipErrorInvalidValue;
        const int wider = p.wqk2 > p.wv2 ? p.wqk2 : p.wv2;
        return wider <= 32   ? launch_walk_kernel<walk_fwd_wide_kernel<T, 4, 1, true>>(grid, smem, p, stream, 2)
               : wider <= 64 ? launch_walk_kernel<walk_fwd_wide_kernel<T, 4, 2, true>>(grid, smem, p, stream, 2)
                             : launch_walk_kernel<walk_fwd_wide_kernel<T, 4, 4, true>>(grid, smem, p, stream, 2);
    }
    if (p.wv <= 64)
        return p.wqk2 <= 32   ? launch_walk_kernel<walk_fwd_wide_kernel<T, 2, 1>>(grid, smem, p, stream)
               : p.wqk2 <= 64 ? launch_walk_kernel<walk_fwd_wide_kernel<T, 2, 2>>(grid, smem, p, stream)
                              : launch_walk_kernel<walk_fwd_wide_kernel<T, 2>>(grid, smem, p, stream);
    return p.wqk2 <= 32   ? launch_walk_kernel<walk_fwd_wide_kernel<T, 4, 1>>(grid, smem, p, stream)
           : p.wqk2 <= 64 ? launch_walk_kernel<walk_fwd_wide_kernel<T, 4, 2>>(grid, smem, p, stream)
                          : launch_walk_kernel<walk_fwd_wide_kernel<T, 4>>(grid, smem, p, stream);
}

template <typename T>
hipError_t launch_walk_rev_wide(const WalkParams &p, hipStream_t stream) {
    using W = WalkCfg<128>;
    const int64_t grid = (int64_t)8 * ((p.BH + 7) / 8) * p.n_seg;
    if (grid > 0x7fffffffLL) return hipErrorInvalidConfiguration;
    if (p.quad != 1 || p.wqk != 128 || p.wqk2 < 1 || p.wqk2 > 128 || p.wv != 128 || p.wv2 < 1 || p.wv2 > 128 || p.fmap || p.dn || p.any_rows ||
        p.wide_out || p.init_transposed || (p.n_seg > 1 && !p.init) || (p.init_is_totals && p.n_seg < 3))
        return hipErrorInvalidValue;
    constexpr int smem = 6 * W::TILE + W::STATE;
    static_assert(smem >= 128 * (128 + 4) * 4, "a state is turned in the tiles' place");
    return launch_walk_kernel<walk_rev_wide_kernel<T>>(grid, smem, p, stream, 4);
}

template <typename T, int D, bool WIDE = false>
hipError_t launch_walk_bwd(const WalkParams &p, hipStream_t stream) {
    if (p.any_rows) return hipErrorNotSupported;
    if constexpr (!WIDE) {
        if (p.wide_out) {
            if constexpr (std::is_same<T, __bf16>::value) return launch_walk_bwd<T, D, true>(p, stream);
            return hipErrorNotSupported;
        }
    }
    const int64_t grid = (int64_t)8 * ((p.BH + 7) / 8) * p.n_seg;
    if (grid > 0x7fffffffLL) return hipErrorInvalidConfiguration;
    constexpr int smem = 4 * WalkCfg<D>::TILE + WalkCfg<D>::STATE;
    if (p.gn && !p.dn) return hipErrorInvalidValue;
    if (p.dn) {
        if (!p.zc || !p.saved || (p.n_seg > 1 && !p.rc)) return hipErrorInvalidValue;
        constexpr int smem_n = smem + WalkCfg<D>::VEC + 1024;
        return p.gn ? launch_walk_kernel<walk_bwd_kernel<T, D, true, WIDE, true>>(grid, smem_n, p, stream)
                    : launch_walk_kernel<walk_bwd_kernel<T, D, true, WIDE>>(grid, smem_n, p, stream);
    }
    if (!p.saved) return hipErrorInvalidValue;
    constexpr auto kern = walk_bwd_kernel<T, D, false, WIDE>;
    constexpr int smem_x = smem + WalkCfg<D>::STATE;  // dQ's state beside R
    if (hipError_t e = ensure_dynamic_lds<kern>(smem_x)) return e;
    return launch_kernel<kern>(dim3((unsigned)grid), dim3(256), smem_x, stream, p);
}

template <typename T, int D, bool WIDE = false, bool ROWS = false>
hipError_t launch_walk_dkdv(const WalkParams &p, hipStream_t stream) {
    if constexpr (!ROWS) {
        if (p.any_rows) {
            if constexpr (!WIDE) return launch_walk_dkdv<T, D, false, true>(p, stream);
            return hipErrorNotSupported;
        }
    }
    if constexpr (!WIDE) {
        if (p.wide_out) {
            if constexpr (!ROWS && std::is_same<T, __bf16>::value) return launch_walk_dkdv<T, D, true>(p, stream);
            return hipErrorNotSupported;
        }
    }
    constexpr int NB = D / 32;
    const int64_t grid = (int64_t)8 * ((p.BH + 7) / 8) * p.n_seg;
    if (grid > 0x7fffffffLL) return hipErrorInvalidConfiguration;
    constexpr int smem = 8 * WalkCfg<D>::TILE + WalkCfg<D>::STATE;
    static_assert(smem <= 160 * 1024, "two sets of tiles and the state must fit the LDS of a CU");
    if constexpr (ROWS) {
        if (p.dn || p.fmap || !walk_rows_ok(p.rows_dk, p.wqk) || !walk_rows_ok(p.rows_dv, p.wv)) return hipErrorInvalidValue;
    } else if (p.dn) {
        if (p.n_seg > 1 && !p.rc) return hipErrorInvalidValue;
        if (p.roles) return hipErrorInvalidValue;
        constexpr auto kern = walk_dkdv_kernel<T, D, true, NB, NB, WIDE>;
        if (hipError_t e = ensure_dynamic_lds<kern>(smem)) return e;
        return launch_kernel<kern>(dim3((unsigned)grid), dim3(256), smem, stream, p);
    }
    if constexpr (D == 128) {
        if (p.roles) {
            if (p.fmap || p.n_seg != 1 || p.init || p.wqk <= 64 || p.wv <= 64) return hipErrorInvalidValue;
            return launch_walk_kernel<walk_dkdv_kernel<T, D, false, NB, NB, WIDE, ROWS, true>>(grid, smem, p, stream, 2);
        }
        if (!p.fmap && p.wqk > 64 && p.wv <= 64) {
            constexpr auto kern = walk_dkdv_kernel<T, D, false, 4, 2, WIDE, ROWS>;
            if (hipError_t e = ensure_dynamic_lds<kern>(smem)) return e;
            return launch_kernel<kern>(dim3((unsigned)grid), dim3(256), smem, stream, p);
        }
    }
    constexpr auto kern = walk_dkdv_kernel<T, D, false, NB, NB, WIDE, ROWS>;
    if (hipError_t e = ensure_dynamic_lds<kern>(smem)) return e;
    return launch_kernel<kern>(dim3((unsigned)grid), dim3(256), smem, stream, p);
}

template <typename T, int D, bool WIDE = false, bool ROWS = false>
hipError_t launch_walk_bwd_rev(const WalkParams &p, hipStream_t stream) {
    if constexpr (!ROWS) {
        if (p.any_rows) {
            if constexpr (!WIDE) return launch_walk_bwd_rev<T, D, false, true>(p, stream);
            return hipErrorNotSupported;
        }
    } else if (p.fmap || !walk_rows_ok(p.rows_dq, p.wqk) || !walk_rows_ok(p.rows_dk, p.wqk) || !walk_rows_ok(p.rows_dv, p.wv)) {
        return hipErrorInvalidValue;
    }
    if constexpr (!WIDE && !ROWS) {
        if (p.wide_out) {
            if constexpr (std::is_same<T, __bf16>::value) return launch_walk_bwd_rev<T, D, true>(p, stream);
            return hipErrorNotSupported;
        }
    }
    const int64_t grid = (int64_t)8 * ((p.BH + 7) / 8) * p.n_seg;
    if (grid > 0x7fffffffLL) return hipErrorInvalidConfiguration;
    if (!p.xtotal || (p.n_seg > 1 && !p.xinit)) return hipErrorInvalidValue;
    if (p.entry_out || (p.init_is_totals && (p.n_seg < 3 || !p.init))) return hipErrorInvalidValue;
    constexpr int smem = 8 * WalkCfg<D>::TILE + WalkCfg<D>::STATE;
    static_assert(smem <= 160 * 1024, "two sets of tiles and the state must fit the LDS of a CU");
    constexpr int NB = D / 32;
    if constexpr (D == 128) {  // a half of a wide q / k against a narrow v: without the blocks of padding
        if (!p.fmap && p.wqk > 64 && p.wv <= 64) return launch_walk_kernel<walk_bwd_rev_kernel<T, D, 4, 2, false, WIDE, ROWS>>(grid, smem, p, stream);
    }
    if constexpr (!ROWS)
        if (p.fmap) return launch_walk_kernel<walk_bwd_rev_kernel<T, D, NB, NB, true, WIDE>>(grid, smem, p, stream);
    return launch_walk_kernel<walk_bwd_rev_kernel<T, D, NB, NB, false, WIDE, ROWS>>(grid, smem, p, stream);
}

template <typename T, bool WIDE = false>
hipError_t launch_walk_bwd_rev_wide(const WalkParams &p, hipStream_t stream) {
    if constexpr (!WIDE) {
        if (p.wide_out) {
            if constexpr (std::is_same<T, __bf16>::value) return launch_walk_bwd_rev_wide<T, true>(p, stream);
            return hipErrorNotSupported;
        }
    }
    using W = WalkCfg<128>;
    const int64_t grid = (int64_t)8 * ((p.BH + 7) / 8) * p.n_seg;
    if (grid > 0x7fffffffLL) return hipErrorInvalidConfiguration;
    if (p.wqk != 128 || p.wqk2 < 1 || p.wqk2 > 128 || p.wv < 1 || p.wv > (p.dq ? 64 : 128)) return hipErrorNotSupported;
    if (p.fmap || p.dn || p.init_transposed || p.entry_out || p.entry_out2 ||
        (p.n_seg > 1 && (!p.init || !p.init2)) || (p.init_is_totals && p.n_seg < 3))
        return hipErrorInvalidValue;
    constexpr int smem = 8 * W::TILE + W::STATE;  // two sets of (Q_h, K_h), two of (V, dO), one state
    static_assert(smem <= 160 * 1024, "the tiles and the state must fit the LDS of a CU");
    if (p.dq) {
        if (p.any_rows) return hipErrorNotSupported;
        if (!p.xtotal || !p.xtotal2 || (p.n_seg > 1 && (!p.xinit || !p.xinit2))) return hipErrorInvalidValue;
        return launch_walk_kernel<walk_bwd_rev_wide_kernel<T, 2, true, WIDE>>(grid, smem, p, stream);
    }
    if (p.any_rows) {
        if (WIDE || p.wv > 64 || p.rows_dk.width <= 128 || !walk_rows_ok(p.rows_dk, 128 + p.wqk2)) return hipErrorInvalidValue;
        return launch_walk_kernel<walk_bwd_rev_wide_kernel<T, 2, false, false, true>>(grid, smem, p, stream);
    }
    if (p.wv <= 64) return launch_walk_kernel<walk_bwd_rev_wide_kernel<T, 2, false, WIDE>>(grid, smem, p, stream);
    if constexpr (WIDE)  // (40 bytes of spills, which this kernel may not have)
        return hipErrorNotSupported;
    else
        return launch_walk_kernel<walk_bwd_rev_wide_kernel<T, 4, false>>(grid, smem, p, stream);
}

// xcd_place's line for a launch of walks or of their totals, D <= 64: whole heads up to twice as many parts, as many as an XCD has CUs (two
// workgroups share a CU), for the normalised operator and where a forward walk without a backward adds up its head's totals as it
// starts; at D = 32 in both passes.  Passes that hand states over go by the same line: a plain forward with whole heads in front of
// a backward in runs, D = 64, took up to 10 % longer than both in runs (B H 15 N 2048 29.4 us, 26.8; both with whole heads 26.8).
// Runs -> whole heads, 17 to 32 parts on the fullest XCD, N 1100 to 4083, device time: normalised forward B H 1 N 4083 15.6 -> 13.7,
// B H 7 N 3500 16.1 -> 13.8, B H 9 N 2048 12.9 -> 11.8, D = 32 B H 9 N 2048 10.1 -> 9.1; with backward B H 15 N 2048 38.0 -> 33.8, D = 32
// 27.1 -> 23.4.  Plain forward B H 7 N 4083 13.9 -> 12.7, B H 12 N 2048 10.7 -> 10.8, D = 32 B H 9 N 2048 8.6 -> 8.0; D = 32 from 17 segments
// on, whose totals another kernel adds up, B H 4 N 4083 11.2 -> 11.8.  Plain, with backward: B H 4 N 4083 27.7 -> 30.4, B H 7 N 3000 27.9
// -> 27.0, B H 12 N 2048 25.0 -> 26.4, but D = 32 B H 9 N 1500 17.2 -> 16.5, B H 12 N 2048 18.5 -> 18.8.
inline int walk_whole_parts(int D, int n_seg, bool norm, bool alone) {
    return D <= 64 && (norm || (n_seg <= walk_sum_on_load_max(D) && (alone || D == 32))) ? 2 * kWholeHeadParts : kWholeHeadParts;
}
// ... and the workgroups that an XCD holds, where the totals are added up as the walks start (D = 128: kSumOnLoadMost)
inline int walk_resident(int D, int n_seg) { return n_seg > (D <= 64 ? walk_sum_on_load_max(D) : 20) ? 0 : D <= 64 ? 64 : 32; }
template <typename P>
void walk_place(int D, P &p, int64_t stride_h, bool norm, bool alone) {
    p.place = xcd_place(p.BH, p.n_seg, stride_h, walk_whole_parts(D, p.n_seg, norm, alone), walk_resident(D, p.n_seg));
    p.n_seg_inv = xcd_inverse(p.n_seg);
}
inline void walk_place(int D, WalkParams &p) { walk_place(D, p, p.ks_h, p.denom || p.dn, !p.saved); }
inline void walk_place(int D, WalkTotalsParams &p) { walk_place(D, p, p.ys_h, p.vsum != nullptr, p.alone); }
inline void walk_place(int D, WalkGradParams &p) { walk_place(D, p, p.qs_h, true, false); }

}  // namespace fla
