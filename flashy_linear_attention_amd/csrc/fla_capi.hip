// C ABI of libfla_gfx950.so (declared in include/fla.h): argument checks,
// mapping of forward / gradients onto the one masked-product kernel, launch.
#include "fla.h"

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>

#include "fla_dispatch.h"
#include "fla_convert.h"
#include "fla_norm.h"
#include "fla_pack.h"
#include "fla_poly_walk.h"

// Scratch of fla_linear_attn_chunked_fwd_static: one copy per GPU, at its own address on each.
// Host code never uses the array's name as an address; it asks the runtime for the device
// address once per device (static_scratch below) and passes that pointer on.  (No `used`
// attribute: it would pin the device symbol to local binding, where the runtime's lookup by
// name cannot find it; the reference from host code below is what keeps the array and makes
// the compiler give it global binding.)
static __device__ __align__(256) unsigned char scratch[FLA_STATIC_SCRATCH_BYTES];

namespace {

constexpr int kMaxDevices = 64;
std::atomic<void *> g_scratch_ptr[kMaxDevices];

// Device address of `scratch` on the current device (looked up on the first call per device).
int static_scratch(void **out) {
#if defined(FLA_TRACE_LAUNCHES)
    *out = reinterpret_cast<void *>((uintptr_t)0x700000000000ull);  // (no device: a made-up, aligned address)
    return FLA_OK;
#endif
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return FLA_ERR_LAUNCH;
    void *ptr = g_scratch_ptr[dev].load(std::memory_order_acquire);
    if (!ptr) {
        if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) return FLA_ERR_LAUNCH;
        g_scratch_ptr[dev].store(ptr, std::memory_order_release);
    }
    *out = ptr;
    return FLA_OK;
}

using fla::TriParams;
typedef hipError_t (*launch_fn)(const TriParams &, hipStream_t);

int pad_index(int64_t d) { return d <= 32 ? 0 : d <= 64 ? 1 : d <= 128 ? 2 : 3; }

launch_fn lookup(int dtype, int64_t dc, int64_t dout) {
#define FLA_ENTRY(c, o) {fla::FLA_LAUNCH_NAME(0, c, o), fla::FLA_LAUNCH_NAME(1, c, o)},
    static const launch_fn table[16][2] = {FLA_FOR_EACH_DIM_PAIR(FLA_ENTRY)};
#undef FLA_ENTRY
    return table[pad_index(dc) * 4 + pad_index(dout)][dtype];
}

typedef hipError_t (*state_fn)(const fla::ChunkStateParams &, hipStream_t);

state_fn lookup_state(int dtype, int64_t dc, int64_t dout) {
#define FLA_ENTRY(c, o) {fla::FLA_STATE_NAME(0, c, o), fla::FLA_STATE_NAME(1, c, o)},
    static const state_fn table[16][2] = {FLA_FOR_EACH_DIM_PAIR(FLA_ENTRY)};
#undef FLA_ENTRY
    return table[pad_index(dc) * 4 + pad_index(dout)][dtype];
}

// rows per chunk of the chunked evaluation for this pair of widths (0: none available)
int chunk_rows(int64_t dc, int64_t dout) {
#define FLA_ENTRY(c, o) fla::fla_chunk_rows_c##c##_o##o,
    static int (*const table[16])() = {FLA_FOR_EACH_DIM_PAIR(FLA_ENTRY)};
#undef FLA_ENTRY
    return table[pad_index(dc) * 4 + pad_index(dout)]();
}

int64_t padded(int64_t d) { return d <= 32 ? 32 : d <= 64 ? 64 : d <= 128 ? 128 : 256; }

int64_t next_pow2(int64_t x) {
    int64_t p = 1;
    while (p < x) p <<= 1;
    return p;
}

struct View {
    const void *ptr;
    const int64_t *strides;
};

int check_view(const View &t) {
    if (!t.ptr) return FLA_ERR_NULL_POINTER;
    if (!t.strides) return FLA_ERR_STRIDE;
    if (t.strides[3] != 1) return FLA_ERR_STRIDE;
    if (t.strides[0] < 0 || t.strides[1] < 0 || t.strides[2] < 0) return FLA_ERR_STRIDE;
    return FLA_OK;
}

// 16-byte vector loads are legal when every row starts 16-byte aligned and the
// width is a whole number of 8-element chunks.
int vec_ok(const View &t, int64_t width) {
    return width % 8 == 0 && reinterpret_cast<uintptr_t>(t.ptr) % 16 == 0 && t.strides[0] % 8 == 0 &&
           t.strides[1] % 8 == 0 && t.strides[2] % 8 == 0;
}

// The kernels read tiles of the inputs while other workgroups already write results: an output
// that shares memory with an input (or with another output) would be read half-updated.  The
// test is on the byte ranges [first element, one past the last addressed element).
struct Span {
    uintptr_t lo, hi;
};

Span span_of(const View &t, int64_t B, int64_t H, int64_t N, int64_t width, int size = 2) {
    if (B <= 0 || H <= 0 || N <= 0 || !t.ptr || !t.strides) return {0, 0};
    const int64_t last = (B - 1) * t.strides[0] + (H - 1) * t.strides[1] + (N - 1) * t.strides[2] + width;
    const uintptr_t lo = reinterpret_cast<uintptr_t>(t.ptr);
    return {lo, lo + (uintptr_t)last * size};
}

bool overlap(const Span &a, const Span &b) { return a.lo < b.hi && b.lo < a.hi; }

int check_alias(const Span *ins, int n_in, const Span *outs, int n_out) {
    for (int o = 0; o < n_out; ++o) {
        for (int i = 0; i < n_in; ++i)
            if (overlap(outs[o], ins[i])) return FLA_ERR_ALIAS;
        for (int o2 = o + 1; o2 < n_out; ++o2)
            if (overlap(outs[o], outs[o2])) return FLA_ERR_ALIAS;
    }
    return FLA_OK;
}

int check_common(int64_t B, int64_t H, int64_t N, int dtype) {
    if (dtype != FLA_DTYPE_BF16 && dtype != FLA_DTYPE_F16) return FLA_ERR_DTYPE;
    if (B < 0 || H < 0 || N < 0) return FLA_ERR_SHAPE;
    if (N > (int64_t)1 << 30) return FLA_ERR_SHAPE;
    if (H > 0 && B > ((int64_t)1 << 30) / H) return FLA_ERR_SHAPE;
    return FLA_OK;
}

// forward-shaped call: two operands of width dc and one of width dout in, one of width dout out
int check_alias_fwd(const View &x, const View &y, const View &z, const View &out, int64_t B, int64_t H, int64_t N,
                    int64_t dc, int64_t dout) {
    const Span ins[] = {span_of(x, B, H, N, dc), span_of(y, B, H, N, dc), span_of(z, B, H, N, dout)};
    const Span outs[] = {span_of(out, B, H, N, dout)};
    return check_alias(ins, 3, outs, 1);
}

// backward-shaped call: go, v (and the forward's output `o`, when given) of width dv, q, k of width
// dqk in; dq, dk of width dqk and dv of width dv out
int check_alias_bwd(const View &go, const View &q, const View &k, const View &v, const View *o, const View &dq,
                    const View &dk, const View &dvv, int64_t B, int64_t H, int64_t N, int64_t dqk, int64_t dv,
                    bool wide = false) {
    const int size = wide ? 4 : 2;  // (FLA_GRADS_F32)
    const Span ins[] = {span_of(go, B, H, N, dv), span_of(q, B, H, N, dqk), span_of(k, B, H, N, dqk),
                        span_of(v, B, H, N, dv), o ? span_of(*o, B, H, N, dv) : Span{0, 0}};
    const Span outs[] = {span_of(dq, B, H, N, dqk, size), span_of(dk, B, H, N, dqk, size), span_of(dvv, B, H, N, dv, size)};
    return check_alias(ins, 5, outs, 3);
}

TriParams make_params(const View &x, const View &y, const View &z, const View &out, int64_t B, int64_t H, int64_t N,
                      int64_t dc, int64_t dout, int upper) {
    TriParams p;
    p.x = x.ptr, p.y = y.ptr, p.z = z.ptr, p.out = const_cast<void *>(out.ptr);
    p.xs_b = x.strides[0], p.xs_h = x.strides[1], p.xs_n = x.strides[2];
    p.ys_b = y.strides[0], p.ys_h = y.strides[1], p.ys_n = y.strides[2];
    p.zs_b = z.strides[0], p.zs_h = z.strides[1], p.zs_n = z.strides[2];
    p.os_b = out.strides[0], p.os_h = out.strides[1], p.os_n = out.strides[2];
    p.H = (int32_t)H, p.N = (int32_t)N, p.BH = (int32_t)(B * H);
    p.dc = (int32_t)dc, p.dout = (int32_t)dout;
    p.upper = upper ? 1 : 0;
    p.n_tiles = 0;
    p.single = 0;
    p.state = nullptr;
    p.state_transposed = 0;
    p.denom = nullptr;
    p.eps = 0.f;
    p.poly[0] = p.poly[1] = p.poly[2] = 0.f;
    p.poly_on = 0;
    p.map_x = p.map_out = 0;
    p.xmap_out = nullptr, p.omap = nullptr;
    p.xo_b = p.xo_h = p.xo_n = 0;
    p.ms_b = p.ms_h = p.ms_n = 0;
    p.vec_x = vec_ok(x, dc), p.vec_y = vec_ok(y, dc), p.vec_z = vec_ok(z, dout), p.vec_out = vec_ok(out, dout);
    return p;
}

typedef hipError_t (*batch_fn)(const fla::TriBatch &, int, hipStream_t);

batch_fn lookup_batch(int dtype, int64_t d) {
    static const batch_fn table[4][2] = {{fla::FLA_BATCH_NAME(0, 32), fla::FLA_BATCH_NAME(1, 32)},
                                         {fla::FLA_BATCH_NAME(0, 64), fla::FLA_BATCH_NAME(1, 64)},
                                         {fla::FLA_BATCH_NAME(0, 128), fla::FLA_BATCH_NAME(1, 128)},
                                         {fla::FLA_BATCH_NAME(0, 256), fla::FLA_BATCH_NAME(1, 256)}};
    return table[pad_index(d)][dtype];
}

batch_fn lookup_chunked_batch(int dtype, int64_t d) {
    static const batch_fn table[4][2] = {{fla::FLA_CBATCH_NAME(0, 32), fla::FLA_CBATCH_NAME(1, 32)},
                                         {fla::FLA_CBATCH_NAME(0, 64), fla::FLA_CBATCH_NAME(1, 64)},
                                         {fla::FLA_CBATCH_NAME(0, 128), fla::FLA_CBATCH_NAME(1, 128)},
                                         {fla::FLA_CBATCH_NAME(0, 256), fla::FLA_CBATCH_NAME(1, 256)}};
    return table[pad_index(d)][dtype];
}

// Out = mask(X Y^T) Z; all arguments already validated.
int run_tri(const View &x, const View &y, const View &z, const View &out, int64_t B, int64_t H, int64_t N,
            int64_t dc, int64_t dout, int upper, int dtype, void *stream) {
    if (B == 0 || H == 0 || N == 0) return FLA_OK;
    // Output wider than 128 columns with a narrow (<= 64) or a 256-wide contraction: run the two
    // 128-column halves of Z / Out as separate launches.  The 64-rows-per-wave kernels that
    // this selects beat the single 256-wide launch (which needs the 32-row layout, or the
    // generic kernel for 256 x 256) although S is formed twice; results are bit-identical
    // because every output column is an independent sum.
    if (dout > 128 && (dc <= 64 || dc > 128)) {
        const View z_hi{static_cast<const char *>(z.ptr) + 128 * 2, z.strides};
        const View out_hi{static_cast<const char *>(out.ptr) + 128 * 2, out.strides};
        if (int rc = run_tri(x, y, z, out, B, H, N, dc, 128, upper, dtype, stream)) return rc;
        return run_tri(x, y, z_hi, out_hi, B, H, N, dc, dout - 128, upper, dtype, stream);
    }
    const TriParams p = make_params(x, y, z, out, B, H, N, dc, dout, upper);
    launch_fn fn = lookup(dtype, dc, dout);
    if (!fn) return FLA_ERR_UNSUPPORTED;
    return fn(p, static_cast<hipStream_t>(stream)) == hipSuccess ? FLA_OK : FLA_ERR_LAUNCH;
}

// bytes of workspace the chunked evaluation of one product needs: fp32 chunk states plus
// their 16-bit running sums, [BH][chunks][DO][DC] each with padded widths
int64_t chunked_bytes(int64_t B, int64_t H, int64_t N, int64_t dc, int64_t dout) {
    if (dout > 128 && (dc <= 64 || dc > 128)) dout = 128;  // evaluated as two 128-column halves
    const int rows = chunk_rows(dc, dout);
    if (rows == 0 || N <= rows) return 0;
    const int64_t chunks = (N + rows - 1) / rows;
    return B * H * chunks * padded(dc) * padded(dout) * 6;
}

// ---- element-wise feature passes, for the shapes and layouts the kernels' own map-on-load does
// not cover: mode 1 writes dst = phi(src); mode 2 multiplies dst in place by phi'(x) computed from
// src = phi(x); mode 3 adds src to dst in place (fp32 sum, one rounding).  Any strides; eight elements per thread where both tensors allow 16-byte accesses.
template <typename T, bool VEC>
__global__ __launch_bounds__(256) void feature_pass_kernel(int mode, int fmap, const T *src, int64_t ss_b, int64_t ss_h,
                                                           int64_t ss_n, T *dst, int64_t ds_b, int64_t ds_h,
                                                           int64_t ds_n, int H, int64_t N, int D, int64_t total) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= total) return;
    constexpr int E = VEC ? 8 : 1;
    const int per_row = D / E;
    const int64_t row = t / per_row;
    const int col = (int)(t - row * per_row) * E;
    const int64_t bh = row / N, n = row - bh * N;
    const int64_t b = bh / H, h = bh - b * H;
    const T *sp = src + b * ss_b + h * ss_h + n * ss_n + col;
    T *dp = dst + b * ds_b + h * ds_h + n * ds_n + col;
    if constexpr (VEC) {
        typedef T v8 __attribute__((ext_vector_type(8)));
        v8 s = *reinterpret_cast<const v8 *>(sp), d;
        if (mode != 1) d = *reinterpret_cast<const v8 *>(dp);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float x = static_cast<float>(s[e]);
            d[e] = static_cast<T>(mode == 1   ? fla::feature_value(fmap, x)
                                  : mode == 2 ? static_cast<float>(d[e]) * fla::feature_slope_from_value(fmap, x)
                                              : static_cast<float>(d[e]) + x);
        }
        *reinterpret_cast<v8 *>(dp) = d;
    } else {
        const float x = static_cast<float>(*sp);
        *dp = static_cast<T>(mode == 1   ? fla::feature_value(fmap, x)
                             : mode == 2 ? static_cast<float>(*dp) * fla::feature_slope_from_value(fmap, x)
                                         : static_cast<float>(*dp) + x);
    }
}

int launch_feature_pass(int mode, int fmap, const View &src, const View &dst, int64_t B, int64_t H, int64_t N,
                        int64_t D, int dtype, void *stream) {
    if (B == 0 || H == 0 || N == 0) return FLA_OK;
    const bool vec = vec_ok(src, D) && vec_ok(dst, D);
    const int64_t total = B * H * N * (vec ? D / 8 : D);
    const int64_t grid = (total + 255) / 256;
    if (grid > 0x7fffffffLL) return FLA_ERR_SHAPE;
    hipStream_t s = static_cast<hipStream_t>(stream);
    hipError_t e;
#define FLA_FEATURE_PASS(T, V)                                                                                      \
    fla::launch_kernel<feature_pass_kernel<T, V>>(dim3((unsigned)grid), dim3(256), 0, s, mode, fmap,                \
                       static_cast<const T *>(src.ptr), src.strides[0], src.strides[1], src.strides[2],            \
                       static_cast<T *>(const_cast<void *>(dst.ptr)), dst.strides[0], dst.strides[1], dst.strides[2], \
                       (int)H, N, (int)D, total)
    if (dtype == FLA_DTYPE_BF16)
        e = vec ? FLA_FEATURE_PASS(__bf16, true) : FLA_FEATURE_PASS(__bf16, false);
    else
        e = vec ? FLA_FEATURE_PASS(_Float16, true) : FLA_FEATURE_PASS(_Float16, false);
#undef FLA_FEATURE_PASS
    return e == hipSuccess ? FLA_OK : FLA_ERR_LAUNCH;
}

// ---- chunk-wise evaluation, in three steps per product:
//   chunk_states: per-chunk Y_c^T Z_c in fp32, then the exclusive running sum over the chunks
//                 before (lower) / after (upper) each chunk, rounded to the storage dtype;
//   chunk_main:   diagonal blocks plus X_c . S_c, S_c taken as stored or transposed.

// true when (x, y, z, out) of these widths can be evaluated chunk-wise: a fast kernel exists,
// the operands qualify for it, and there is more than one chunk
bool chunkable(const TriParams &p, int64_t dc, int64_t dout, int64_t N) {
    const int rows = chunk_rows(dc, dout);
    return rows != 0 && N > rows && fla::fast_path_ok(p);
}

int chunk_states(const View &y, const View &z, int64_t B, int64_t H, int64_t N, int64_t dc, int64_t dout, int upper,
                 int dtype, float *w, void *state, void *stream, int map_y = 0, const View *ymap_out = nullptr) {
    const int64_t rows = chunk_rows(dc, dout), chunks = (N + rows - 1) / rows, E = padded(dc) * padded(dout);
    hipStream_t s = static_cast<hipStream_t>(stream);
    fla::ChunkStateParams cp;
    cp.y = y.ptr, cp.z = z.ptr, cp.w = w;
    cp.ys_b = y.strides[0], cp.ys_h = y.strides[1], cp.ys_n = y.strides[2];
    cp.zs_b = z.strides[0], cp.zs_h = z.strides[1], cp.zs_n = z.strides[2];
    cp.H = (int32_t)H, cp.N = (int32_t)N, cp.BH = (int32_t)(B * H), cp.dc = (int32_t)dc, cp.dout = (int32_t)dout;
    cp.n_chunks = (int32_t)chunks;
    cp.map_y = map_y, cp.ymap_out = nullptr;
    cp.yo_b = cp.yo_h = cp.yo_n = 0;
    if (map_y) {
        cp.ymap_out = const_cast<void *>(ymap_out->ptr);
        cp.yo_b = ymap_out->strides[0], cp.yo_h = ymap_out->strides[1], cp.yo_n = ymap_out->strides[2];
    }
    if (lookup_state(dtype, dc, dout)(cp, s) != hipSuccess) return FLA_ERR_LAUNCH;
    const hipError_t e = dtype == FLA_DTYPE_BF16
                             ? fla::launch_chunk_scan<__bf16>(w, state, B * H, (int)chunks, E, upper ? 1 : 0, s)
                             : fla::launch_chunk_scan<_Float16>(w, state, B * H, (int)chunks, E, upper ? 1 : 0, s);
    return e == hipSuccess ? FLA_OK : FLA_ERR_LAUNCH;
}

int chunk_main(TriParams p, int64_t dc, int64_t dout, int dtype, const void *state, int transposed, void *stream) {
    p.state = state;
    p.state_transposed = transposed;
    const hipError_t e = lookup(dtype, dc, dout)(p, static_cast<hipStream_t>(stream));
    return e == hipSuccess ? FLA_OK : e == hipErrorNotSupported ? FLA_ERR_UNSUPPORTED : FLA_ERR_LAUNCH;
}

// Out *= phi'(x) from y = phi(x) held in `y` (Out's shape): the chain rule in the kernel's epilogue
void set_output_slope(TriParams &p, int fmap, const View &y) {
    p.map_out = fmap, p.omap = y.ptr;
    p.ms_b = y.strides[0], p.ms_h = y.strides[1], p.ms_n = y.strides[2];
}

// Out = mask(X Y^T) Z evaluated chunk-wise; same arguments as run_tri plus the workspace.
// Falls back to the quadratic kernels when the operands do not qualify for the fast path
// or the sequence is a single chunk.
int run_tri_chunked(const View &x, const View &y, const View &z, const View &out, int64_t B, int64_t H, int64_t N,
                    int64_t dc, int64_t dout, int upper, int dtype, void *workspace, int64_t workspace_bytes,
                    void *stream) {
    if (B == 0 || H == 0 || N == 0) return FLA_OK;
    if (dout > 128 && (dc <= 64 || dc > 128)) {
        const View z_hi{static_cast<const char *>(z.ptr) + 128 * 2, z.strides};
        const View out_hi{static_cast<const char *>(out.ptr) + 128 * 2, out.strides};
        if (int rc = run_tri_chunked(x, y, z, out, B, H, N, dc, 128, upper, dtype, workspace, workspace_bytes, stream))
            return rc;
        return run_tri_chunked(x, y, z_hi, out_hi, B, H, N, dc, dout - 128, upper, dtype, workspace, workspace_bytes,
                               stream);
    }
    const TriParams p = make_params(x, y, z, out, B, H, N, dc, dout, upper);
    if (!chunkable(p, dc, dout, N)) return run_tri(x, y, z, out, B, H, N, dc, dout, upper, dtype, stream);
    const int64_t rows = chunk_rows(dc, dout), chunks = (N + rows - 1) / rows, E = padded(dc) * padded(dout);
    const int64_t BH = B * H;
    if (!workspace || reinterpret_cast<uintptr_t>(workspace) % 16 != 0 || workspace_bytes < BH * chunks * E * 6)
        return FLA_ERR_WORKSPACE;
    float *w = static_cast<float *>(workspace);
    void *state = static_cast<char *>(workspace) + BH * chunks * E * 4;
    if (int rc = chunk_states(y, z, B, H, N, dc, dout, upper, dtype, w, state, stream)) return rc;
    return chunk_main(p, dc, dout, dtype, state, 0, stream);
}

// ---- the whole operator chunk-wise, with running states shared between products.  With equal
// padded head dims up to 128 all four products run the same square kernel, and
//     state(dQ) = state(O)^T   (sum of K_c^T V_c over the chunks before)
//     state(dK) = state(dV)^T  (sum of Q_c^T dO_c over the chunks after)
// so forward can hand its state to backward, and backward computes one new state instead of
// three.  Any other shape evaluates each product on its own.

// ---- equal padded head dims up to 128: the walk kernels (fla_chunk_walk.h).  A workgroup walks a
// segment of chunks (128 rows, 64 at D = 128) with the running state in registers; segment entry
// states come from a totals kernel and a scan over the segments.
//   D <= 64: two workgroups per CU; forward saves the 16-bit state at the entry of every chunk, and
//            one backward kernel computes dQ, dV and dK of a chunk from one set of tiles;
//   D = 128 (`split`): one workgroup per CU with two sets of tiles.  A per-chunk state would cost as
//            much traffic as an operand, so forward hands over its segments' fp32 entry states
//            only (backward: chunked_backward).  The totals kernel visits a part of the
//            sequence only (the last segment's total is never needed).
struct WalkPlan {
    bool ok, split;
    int D, rows;
    int64_t n_chunks, seg_chunks, n_seg;  // the walks' segments
    int64_t entry_bytes;                  // fp32 entry states of the walk segments (formed in place over their totals)
    int64_t work_bytes;                   // workspace of one direction: the same
    int64_t saved_bytes;                  // what forward hands to backward -- D = 128: the entry states and, behind them, the
                                          // state after the last chunk of every (b, h); up to 64: the 16-bit state at the
                                          // entry of every chunk
};

// `mixed`: also for head dims whose padded widths differ (128 / 64, 64 / 32, 64 / 128 ...), at the larger one: the tiles
// are padded with zeros as they land in LDS, and at D = 128 the kernels built for at most 64 true columns on one side
// leave the padding's MFMAs out.  The plain operator only (the normaliser's and the feature maps' variants of the
// kernels are built for equal padded widths).
// From three segments per (b, h) up to this many the walks add up the segments' totals themselves, beyond it a scan kernel
// does (padded head dims up to 64: fla::walk_sum_on_load_max, which the kernels know).
//   D = 128.  Forward + backward, scan against sums on load: B H 24, N 1500 (8 segments) 66.8 / 62.4 us; B H 20, N 2048 (11)
//   89.6 / 83.6; B H 16, N 4096 (16) 92.0 / 87.5; B H 12, N 4096 (16) 83.8 / 82.0; B H 10, N 4096 (22) 106.0 / 107.6; B H 9
//   (22) 101.9 / 105.7; B H 10, N 16384 (24) 248 / 251; B H 8, N 8192 (32) 91.4 / 99.4.  Four pairs of column
//   halves at a time (256 / 256) the same: B H 8, N 4096 (16) 154.4 / 141.7; B H 6, N 8192 (19) 313 / 304; B H 5, N 4096 (22)
//   182.9 / 190.1.
//   A wide q / k against a v of up to 128: two states to add up.  256 / 64, B H 64, N 4096 (4) 320 / 313 (kernels); through the
//   operator, v of 64: 153 / 64, B H 32, N 2048 (8) 121.6 / 117.0; 256 / 64, B H 32, N 2048 (8) 99.6 / 98.7, B H 24, N 8192 (10)
//   226.0 / 219.9, B H 16, N 4096 (16) 103.6 / 104.8.  v of 128: 192 / 128, B H 32, N 2048 (8) 148 / 130, B H 24, N 4096 (10)
//   191 / 176, 256 / 128, B H 16, N 4096 (16) 151.8 / 146.0, N 2048 111.2 / 108.6, forward alone 192 / 128, B H 16, N 4096 51.2 / 48.6.
//   kSumOnLoadWorkspace: a plain forward with a state buffer and no workspace is refused up to this many segments and taken beyond,
//   by a scan in the state buffer.  The scan could do the fewer segments as well; twelve is where the walks' sums ended before the
//   loads of several states were in flight together, and it stays so that every call keeps its answer.
//   The polynomial map, 41 KiB a state, forward + backward (forward alone): B H 20, N 4096 (11 segments) 136.1 / 129.9 us (47.1 /
//   43.7); B H 16, N 4096 (16) 84.1 / 83.3 (32.5 / 27.2); B H 10, N 2000 (16) 59.2 / 53.4; B H 8, N 8192 (32) 83.8 / 94.6.
constexpr int kSumOnLoadMost = 20, kSumOnLoadWide = 15, kSumOnLoadPoly = 20, kSumOnLoadWorkspace = 12;

// `parts`: workgroups per segment (a launch that does several column halves at a time).
// `halves`: a 128-column half of wider operands.  Up to 256 rows there, and with padded widths that differ, the products would be a launch
// for each and for each half of a result (sixteen, with chunk states 24, at 256 / 256); equal widths of 128 are one diagonal block for the quadratic kernel.
WalkPlan walk_plan(int64_t B, int64_t H, int64_t N, int64_t dqk, int64_t dv, bool mixed = false, int64_t parts = 1, bool halves = false) {
    WalkPlan w{};
    if (B <= 0 || H <= 0 || N <= 0) return w;  // (an empty problem has no plan; the callers return before any launch)
    const int64_t wider = padded(dqk) > padded(dv) ? padded(dqk) : padded(dv);
    if (wider > 128 || (!mixed && pad_index(dqk) != pad_index(dv))) return w;
    w.D = (int)wider;
    w.rows = fla::walk_rows(w.D);
    w.split = w.D > 64;
    w.ok = N > (w.split && !halves && pad_index(dqk) == pad_index(dv) ? 256 : w.rows);
    if (!w.ok) return w;
    w.n_chunks = (N + w.rows - 1) / w.rows;
    // Segments per (b, h): the largest number that keeps B H n_seg within the workgroups that run at once (one per
    // CU at D = 128, two below; measured at B H = 16, N = 32768, D = 64: 256 / 512 / 1024 / 2048 workgroups give
    // 0.265 / 0.231 / 0.243 / 0.268 ms per forward + backward).  Workgroups beyond those wait for a free CU and run
    // as a second round: B H = 192, N = 4096, D = 128 takes 0.87 ms with two unequal segments in 384 workgroups
    // and 0.53 ms with one segment each; plans of several rounds of shorter segments, chosen by a cost model of
    // rounds x segment length, measured 5 to 35 % slower than this rule over B H = 65 ... 300.
    // (totals over finer segments than the walk's, 2 or 4 per walk segment, would put more workgroups on the
    // totals kernel; measured at D = 128 over B H = 8 ... 256, N = 1024 ... 32768, one total per walk segment
    // is the fastest everywhere, by 3 to 27 % of a forward + backward step)
    const int64_t resident = (w.split ? 256 : 512) / parts;
    int64_t segs = resident / (B * H) > 1 ? resident / (B * H) : 1;
    if (segs > w.n_chunks) segs = w.n_chunks;
    if (w.split && N <= 256) segs = 1;  // (four chunks at most: less than a totals kernel takes)
    w.seg_chunks = (w.n_chunks + segs - 1) / segs;
    w.n_seg = (w.n_chunks + w.seg_chunks - 1) / w.seg_chunks;
    w.entry_bytes = B * H * w.n_seg * w.D * w.D * 4;
    w.work_bytes = w.entry_bytes;  // (a single segment needs them only with a feature map)
    // (up to 64 with few chunks per segment: the size that held the segments' fp32 states, which callers of the C ABI may
    // have set aside, stays the larger)
    const int64_t states = w.entry_bytes + B * H * w.D * w.D * 4;
    const int64_t per_chunk = B * H * w.n_chunks * w.D * w.D * 2;
    w.saved_bytes = w.split || states > per_chunk ? states : per_chunk;
    return w;
}

bool sums_on_load(const WalkPlan &w, int most = kSumOnLoadMost) { return w.n_seg >= 3 && w.n_seg <= most; }

// Two workgroups per (b, h) on two column halves of O, on dV and dK (WalkParams::cols, roles), where they would be two segments: no
// totals of half of the sequence come before the walk.  q and k (q and dO) are read by both, within one XCD: its L2 serves the second
// read, at B H 128 and N 2048 to 8192 both kernels fetch every operand once (FETCH_SIZE, 403 and 537 MB at N 4096).  A workgroup
// then walks the whole sequence, at 1.8 to 1.9 us a chunk of 128 columns however many heads there are, where the segments' time
// grows with the bytes of all heads: hence lines by the head count.  `plain`: no normaliser and no feature map.
//   Backward, 128 columns, two segments -> this, forward + backward: B H 128, N 1024 114 / 102 us, N 2048 219 / 204, N 8192 857 / 819; B H
//   112, N 4096 387 / 375; B H 104, N 3072 279 / 268; B H 96, N 1024 98 / 90, N 4096 355 / 350; 72 and 96 columns, B H 88 and 96, N 2048 147
//   to 150 / 151 to 153; 80 columns, B H 128, N 4096 307 / 316, 96 columns, N 3008 251 / 246.  (dQ's walk as well: B H 128, N 4096
//   408 -> 422: it starts from what forward left and has no totals to save.)
//   Forward alone in bf16, inputs that change from pass to pass (with the same ones again and again the Infinity Cache hides the
//   segments' second read of k and v, up to N 4096): 128 columns, N 2048 B H 97 59.0 / 57.9, B H 128 68.8 / 63.0; N 3072 B H 97 85.0 /
//   85.1, B H 112 93.9 / 89.0, B H 128 105 / 95; N 4096 B H 104 116 / 114, B H 116 129 / 118, B H 128 136 / 124 (with backward 422 / 411);
//   N 8192 B H 97 210 / 221, B H 104 222 / 223, B H 112 235 / 230, B H 128 263 / 246; N 16384 B H 116 474 / 469; 96 and 112 columns, B H
//   105 to 128, N 2560 to 8192 0.99 to 1.11.
//   In fp16, where a chunk takes 2.1 us (the state's scale), forward alone: N 1024 B H 100 39.2 / 37.9, B H 128 48.0 / 39.8; N 2048 B H 100
//   65.8 / 68.0, B H 112 69.6 / 68.8, B H 128 77.4 / 74.1; N 3072 B H 112 102 / 106; N 4096 B H 120 139 / 142, B H 128 145 / 145; N 8192 B H
//   128 276 / 288.
bool walk_by_columns(const WalkPlan &w, int64_t bh, int64_t N, int64_t dqk, int64_t dv, bool plain) {
    return plain && w.ok && w.split && dqk > 64 && dv > 64 && w.n_seg == 2 && (bh > 96 || N <= 1024) &&
           (N <= 2048 || (dqk >= 96 && dv >= 96));
}
bool forward_by_columns(const WalkPlan &w, int64_t bh, int64_t N, int64_t dqk, int64_t dv, int dtype, bool plain) {
    return walk_by_columns(w, bh, N, dqk, dv, plain) &&
           (dtype == FLA_DTYPE_F16 ? N <= 1024 || (N <= 2048 && bh > 104) : N <= 2048 || bh > 104);
}

// totals of Y^T Z over the walk's segments into `work`, then the segments' entry states: their sums
// over the segments before (reverse == 0) or after (reverse != 0), written to `entry` (null: over
// the totals in `work`).  Returns where the entry states are.
// `second`: the same for another Y operand of the same layout against the same Z (the other half of a
// wide q / k) in the same launches -- one totals launch and one scan for the two of them.
struct EntryHalf {
    const void *y;  // Y's pointer (Y's strides are the first operand's)
    int64_t dy;
    void *work;
    float *entry;
    const float **where;
};

int walk_entry_states(const WalkPlan &w, const View &y, const View &z, int64_t B, int64_t H, int64_t N, int64_t dy,
                      int64_t dz, int dtype, int reverse, void *work, float *entry, const float **where, hipStream_t s,
                      int map_y = 0, const View *ymap_out = nullptr, const EntryHalf *second = nullptr,
                      bool totals_only = false, bool z_narrow = false, float *vsum = nullptr, bool alone = false) {
    fla::WalkTotalsParams tp{};
    tp.vsum = vsum, tp.alone = alone;
    tp.z_narrow = z_narrow;
    if (map_y) {
        tp.map_y = map_y, tp.ymap_out = const_cast<void *>(ymap_out->ptr);
        tp.yo_b = ymap_out->strides[0], tp.yo_h = ymap_out->strides[1], tp.yo_n = ymap_out->strides[2];
    }
    float *totals = static_cast<float *>(work);
    if (!entry) entry = totals;
    // (two segments: the one total needed is the other segment's entry state; the totals kernel writes it as the
    // walks read it, two partial sums, and no scan follows.  A few segments more: the walks add up the totals
    // themselves as they start -- fla::walk_entries_are_totals -- and no scan follows either)
    // (totals_only: the caller's walk adds them up itself -- WalkParams::init_is_totals; not with two segments)
    const bool direct = w.n_seg == 2;
    const bool summed_on_load = fla::walk_entries_are_totals(w.D, (int)w.n_seg) || (totals_only && !direct);
    const bool no_scan = direct || summed_on_load;
    tp.y = y.ptr, tp.z = z.ptr, tp.totals = no_scan ? entry : totals, tp.direct = direct, tp.frags = summed_on_load;
    tp.ys_b = y.strides[0], tp.ys_h = y.strides[1], tp.ys_n = y.strides[2];
    tp.zs_b = z.strides[0], tp.zs_h = z.strides[1], tp.zs_n = z.strides[2];
    tp.H = (int32_t)H, tp.N = (int32_t)N, tp.BH = (int32_t)(B * H), tp.dy = (int32_t)dy, tp.dz = (int32_t)dz;
    tp.n_chunks = (int32_t)w.n_chunks, tp.seg_chunks = (int32_t)w.seg_chunks, tp.n_seg = (int32_t)w.n_seg;
    // the total of the walk's last segment (first, walking in reverse) is under no sum; a feature map
    // is applied by this kernel, which then has to visit every row
    tp.seg_lo = reverse && !map_y ? 1 : 0;
    tp.seg_hi = (int32_t)(!reverse && !map_y ? w.n_seg - 1 : w.n_seg);
    if (direct) tp.seg_lo = reverse ? 1 : 0, tp.seg_hi = tp.seg_lo + 1;  // (the needed one)
    float *totals2 = nullptr, *entry2 = nullptr;
    if (second) {
        totals2 = static_cast<float *>(second->work);
        entry2 = second->entry ? second->entry : totals2;
        tp.y2 = second->y, tp.dy2 = (int32_t)second->dy, tp.totals2 = no_scan ? entry2 : totals2;
        *second->where = entry2;
    }
    if (fla::walk_totals(dtype, w.D, tp, s) != hipSuccess) return FLA_ERR_LAUNCH;
    *where = entry;
    if (no_scan) return FLA_OK;
    return fla::walk_scan(totals, entry, B * H, (int)w.n_seg, w.D, z_narrow ? 64 : fla::walk_totals_cols(w.D, (int)dy, (int)dz), reverse,
                          s, totals2, entry2) == hipSuccess
               ? FLA_OK
               : FLA_ERR_LAUNCH;
}

// Entry states of both 128-column halves of a wide q / k (Y = the halves of `y`, against the same Z):
// one totals launch and one scan for the two when both halves take the same kernel variant, else
// one after the other.  work[h], entry[h] (null: over work[h]) and where[h] per half.
// `z_narrow`: dz <= 64, and the walks behind leave columns 64 .. of the states out whatever the second half's width
// (walk_fwd_wide_kernel, walk_bwd_rev_wide_kernel): one launch for any D_qk.
int wide_entry_states(const WalkPlan &wp, const View &y, const View &z, int64_t B, int64_t H, int64_t N, int64_t dy_all,
                      int64_t dz, int dtype, int reverse, void *const (&work)[2], float *const (&entry)[2],
                      const float *(&where)[2], hipStream_t s, bool totals_only = false, bool z_narrow = false) {
    const View y1{static_cast<const char *>(y.ptr) + 128 * 2, y.strides};
    const int64_t dy1 = dy_all - 128;
    if (z_narrow || fla::walk_totals_cols(wp.D, 128, (int)dz) == fla::walk_totals_cols(wp.D, (int)dy1, (int)dz)) {
        const EntryHalf other{y1.ptr, dy1, work[1], entry[1], &where[1]};
        return walk_entry_states(wp, y, z, B, H, N, 128, dz, dtype, reverse, work[0], entry[0], &where[0], s, 0, nullptr,
                                 &other, totals_only, z_narrow);
    }
    if (int rc = walk_entry_states(wp, y, z, B, H, N, 128, dz, dtype, reverse, work[0], entry[0], &where[0], s, 0, nullptr,
                                   nullptr, totals_only))
        return rc;
    return walk_entry_states(wp, y1, z, B, H, N, dy1, dz, dtype, reverse, work[1], entry[1], &where[1], s, 0, nullptr,
                             nullptr, totals_only);
}

// The normaliser's terms handed to the walk kernels (fla_chunk_walk.h, WalkParams::denom ...).
struct WalkNorm {
    float *denom;     // forward: receives n
    float eps;
    float *dn;        // backward: dn_i = -(g_i . out_i) / n_i (and the grad_out operand holds g / n)
    void *vec;        // scratch, 2 * walk_vec_bytes(): the segments' totals of k (forward), zc without a saved one; rc
    // backward: g, out and n, from which the kernel in front of the walks forms dO and dn beside the segments' totals (where
    // norm_walks_backward() says that the walks take the call: otherwise they have been formed before it)
    const View *go, *out;
    const float *n;
    bool vec16;       // g and out allow 16-byte loads
    bool fused;       // out: the kernels took the terms (false: the caller runs the passes of fla_norm.h)
    bool dk_pending;  // out: ... all but dK's sum over later rows (and dK's slope, with a feature map)
};

int64_t walk_vec_bytes(int64_t B, int64_t H, int64_t N, int64_t dqk, int64_t dv) {
    const WalkPlan w = walk_plan(B, H, N, dqk, dv);
    return w.ok ? B * H * w.n_chunks * w.D * 4 : 0;
}

// zc, the running sum of k at the entry of every chunk, where forward's is not at hand (D = 128)
int walk_chunk_vectors(const WalkPlan &wp, const View &k, int64_t width, float *out, int64_t B, int64_t H, int64_t N, int dtype,
                       hipStream_t s) {
    fla::WalkVecParams vp{};
    vp.y = k.ptr, vp.ys_b = k.strides[0], vp.ys_h = k.strides[1], vp.ys_n = k.strides[2];
    vp.H = (int32_t)H, vp.N = (int32_t)N, vp.width = (int32_t)width, vp.n_chunks = (int32_t)wp.n_chunks;
    vp.out = out;
    if (fla::walk_vec_sums(dtype, vp, B * H, s) != hipSuccess) return FLA_ERR_LAUNCH;
    return fla::walk_vec_scan(out, B * H, (int)wp.n_chunks, wp.D, s) == hipSuccess ? FLA_OK : FLA_ERR_LAUNCH;
}

// dO and dn of the normalised backward with the segments' totals of Q^T dO (to `work`) and of dn_i q_i (to `rc`), and the
// entry states of the reverse walk from the former where it does not add them up itself (`totals_only`, or by its number of
// segments).  Returns where the entry states are.
int walk_grad_entry_states(const WalkPlan &w, const View &q, const View &dout, const WalkNorm &nx, int64_t B, int64_t H, int64_t N,
                           int64_t dqk, int64_t dv, int dtype, void *work, float *rc_totals, const float **where, bool totals_only,
                           hipStream_t s, bool keep_g = false) {
    fla::WalkGradParams gp{};
    gp.keep_g = keep_g;
    gp.q = q.ptr, gp.qs_b = q.strides[0], gp.qs_h = q.strides[1], gp.qs_n = q.strides[2];
    gp.go = nx.go->ptr, gp.gs_b = nx.go->strides[0], gp.gs_h = nx.go->strides[1], gp.gs_n = nx.go->strides[2];
    gp.o = nx.out->ptr, gp.os_b = nx.out->strides[0], gp.os_h = nx.out->strides[1], gp.os_n = nx.out->strides[2];
    gp.denom = nx.n, gp.dout = const_cast<void *>(dout.ptr), gp.dn = nx.dn, gp.vec = nx.vec16;
    gp.H = (int32_t)H, gp.N = (int32_t)N, gp.BH = (int32_t)(B * H), gp.wqk = (int32_t)dqk, gp.wv = (int32_t)dv;
    gp.n_chunks = (int32_t)w.n_chunks, gp.seg_chunks = (int32_t)w.seg_chunks, gp.n_seg = (int32_t)w.n_seg;
    const bool several = w.n_seg > 1;
    gp.totals = several ? static_cast<float *>(work) : nullptr, gp.rsum = several ? rc_totals : nullptr;
    gp.frags = w.n_seg > 2 && (totals_only || fla::walk_entries_are_totals(w.D, (int)w.n_seg));
    *where = gp.totals;
    if (fla::walk_grad_totals(dtype, w.D, gp, s) != hipSuccess) return FLA_ERR_LAUNCH;
    if (w.n_seg <= 2 || gp.frags) return FLA_OK;
    return fla::walk_scan(gp.totals, gp.totals, B * H, (int)w.n_seg, w.D, w.D, 1, s) == hipSuccess ? FLA_OK : FLA_ERR_LAUNCH;
}

bool states_shareable(int64_t dqk, int64_t dv, int64_t N) {
    if (pad_index(dqk) != pad_index(dv) || padded(dqk) > 128) return false;
    const int rows = chunk_rows(dqk, dv);
    return rows != 0 && N > rows;
}

// The caller's results of any alignment behind aligned stand-ins (packed_forward, packed_backward), of the true widths, for walks
// that can store to them; `done`: they did, for all of the call's results
struct AnyRows {
    const View *o, *dq, *dk, *dv;
    int64_t dqk, wv;
    bool done;
};

// bytes of one rounded running state / of the scratch one state computation needs (fp32 chunk states)
// ---- D_qk in (128, 256] with D_v <= 128 (the small-V operator's shapes).  The scores are a sum over
// the two 128-column halves of q and k and everything is linear in them:
//     O  = tril(Q_0 K_0^T) V + tril(Q_1 K_1^T) V        dV = the same sum of the halves' dV
//     dQ_h = tril(dO V^T) K_h                           dK_h = triu(V dO^T) Q_h
// so each half is a D = 128 walk on column views of q, k, dq, dk (v and dO are padded with zeros in
// LDS, never in memory), and one launch walks both halves of a chunk, O and dV in fp32 from the first
// half to the second.  Forward hands over both halves' entry and final states.  Backward is one reverse
// walk with them and a v of at most 64 columns (wide_backward says when); otherwise a reverse walk for dK
// and dV and a forward-direction walk per half for dQ_h.
struct WidePlan {
    bool ok;
    WalkPlan wp;  // the plan of a 128 / 128 problem of the same B, H, N
};

WidePlan wide_plan(int64_t B, int64_t H, int64_t N, int64_t dqk, int64_t dv) {
    WidePlan w{};
    if (dqk <= 128 || dqk > 256 || dv > 128) return w;
    w.wp = walk_plan(B, H, N, 128, 128, false, 1, true);
    w.ok = w.wp.ok;
    return w;
}

View column_half(const View &t, int h) { return View{static_cast<const char *>(t.ptr) + h * 128 * 2, t.strides}; }

// ---- D_v in (128, 256].  O and dV are column by column in v's (dO's) columns, and dQ, dK
// are sums over them: the two column halves of v (128 and D_v - 128 columns) each run the plan of a
// (D_qk, at most 128) problem -- the walk kernels at D = 128, or the walks over a wide q / k -- on column views
// of v, O, dO, dV; the second half's dQ and dK go to scratch tensors that one element-wise pass each adds to the
// first half's.  (q and k are read once per half; the 256-row chunk kernels with their per-chunk states in
// memory, which these shapes took before, measured 2.4x slower at 256 / 256.)
struct VSplit {
    bool ok;
    int64_t dv1;         // columns of the second half
    int64_t state0;      // bytes of the first half's state (the second half's follows it)
    int64_t temp_bytes;  // one scratch tensor, contiguous (B, H, N, D_qk)
};

int64_t shared_state_bytes(int64_t B, int64_t H, int64_t N, int64_t dqk, int64_t dv);
int64_t chunked_op_workspace_bytes(int64_t B, int64_t H, int64_t N, int64_t dqk, int64_t dv);

VSplit vsplit_plan(int64_t B, int64_t H, int64_t N, int64_t dqk, int64_t dv) {
    VSplit s{};
    if (dv <= 128 || dv > 256 || dqk < 1 || dqk > 256 || B <= 0 || H <= 0 || (dqk <= 128 && N <= 256)) return s;
    s.dv1 = dv - 128;
    auto planned = [&](int64_t d) { return walk_plan(B, H, N, dqk, d, true).ok || wide_plan(B, H, N, dqk, d).ok; };
    s.ok = planned(128) && planned(s.dv1);
    if (!s.ok) return s;
    s.state0 = (shared_state_bytes(B, H, N, dqk, 128) + 255) / 256 * 256;
    s.temp_bytes = (B * H * N * dqk * 2 + 255) / 256 * 256;
    return s;
}

View v_half(const View &t, int j) { return View{static_cast<const char *>(t.ptr) + j * 128 * 2, t.strides}; }

// what the halves' own calls use of the workspace (the scratch tensors follow it)
int64_t vsplit_inner_bytes(const VSplit &vs, int64_t B, int64_t H, int64_t N, int64_t dqk) {
    const int64_t a = chunked_op_workspace_bytes(B, H, N, dqk, 128), b = chunked_op_workspace_bytes(B, H, N, dqk, vs.dv1);
    return ((a > b ? a : b) + 255) / 256 * 256;
}

int64_t state_core_bytes(int64_t B, int64_t H, int64_t N, int64_t dqk, int64_t dv) {
    if (const VSplit vs = vsplit_plan(B, H, N, dqk, dv); vs.ok) return vs.state0 + shared_state_bytes(B, H, N, dqk, vs.dv1);
    const WalkPlan w = walk_plan(B, H, N, dqk, dv, true);
    if (w.ok && !w.split) return w.saved_bytes;  // one state per 128-row chunk (also room for the 256-row chunks' states)
    if (!states_shareable(dqk, dv, N)) {
        const WidePlan wide = wide_plan(B, H, N, dqk, dv);
        return wide.ok ? 2 * wide.wp.saved_bytes : w.ok ? w.saved_bytes : 0;
    }
    const int64_t rows = chunk_rows(dqk, dv);
    const int64_t per_chunk = B * H * ((N + rows - 1) / rows) * padded(dqk) * padded(dv) * 2;
    return w.ok && w.saved_bytes > per_chunk ? w.saved_bytes : per_chunk;  // (split: either path's state fits)
}

// The buffer forward's state goes to: the states above and, behind them, room for the running sums of
// k at the entry of every chunk, which the normalised forward leaves there for its backward.
int64_t shared_state_bytes(int64_t B, int64_t H, int64_t N, int64_t dqk, int64_t dv) {
    const int64_t core = state_core_bytes(B, H, N, dqk, dv);
    return core ? core + walk_vec_bytes(B, H, N, dqk, dv) : 0;
}

// fp16 without the normaliser, up to 64 columns: the saved copies' scales, a float per chunk, lie in that room (null where there is none:
// widths whose paddings differ).  Every such forward leaves them and every such backward reads them, whatever evaluated either: a feature
// map's forward runs the plain walk where the operands' rows keep the map out of it, and its backward maps all the same.
float *saved_scales(const void *state, int64_t B, int64_t H, int64_t N, int64_t dqk, int64_t dv) {
    if (!walk_vec_bytes(B, H, N, dqk, dv)) return nullptr;
    return reinterpret_cast<float *>(static_cast<char *>(const_cast<void *>(state)) + state_core_bytes(B, H, N, dqk, dv));
}

// workspace of the two-halves evaluation: totals and entry states of both halves (two sets of them in
// backward: Q^T dO, and K^T V when forward's entry states are not given)
int64_t wide_workspace_bytes(const WidePlan &w) { return 4 * w.wp.work_bytes; }

int64_t chunked_op_workspace_bytes(int64_t B, int64_t H, int64_t N, int64_t dqk, int64_t dv) {
    const int64_t shared = shared_state_bytes(B, H, N, dqk, dv);
    if (shared) {  // fp32 chunk states (2x) + two rounded states (backward without a saved one); the walk's totals
        const WalkPlan w = walk_plan(B, H, N, dqk, dv, true);
        if (w.ok || states_shareable(dqk, dv, N)) {
            int64_t m = w.ok && w.work_bytes * 2 > shared * 4 ? w.work_bytes * 2 : shared * 4;
            if (pad_index(dqk) != pad_index(dv)) {  // (off the walks these shapes evaluate product by product)
                const int64_t a = chunked_bytes(B, H, N, dqk, dv), b = chunked_bytes(B, H, N, dv, dqk);
                m = a > m ? a : m, m = b > m ? b : m;
            }
            return m;
        }
    }
    int64_t m = chunked_bytes(B, H, N, dqk, dv);
    const int64_t t = chunked_bytes(B, H, N, dv, dqk);
    if (t > m) m = t;
    const WidePlan wide = wide_plan(B, H, N, dqk, dv);
    if (wide.ok && wide_workspace_bytes(wide) > m) m = wide_workspace_bytes(wide);
    if (const VSplit vs = vsplit_plan(B, H, N, dqk, dv); vs.ok) {
        const int64_t need = vsplit_inner_bytes(vs, B, H, N, dqk) + 2 * vs.temp_bytes;
        if (need > m) m = need;
    }
    return m;
}

// the walk that computes out = lower(x y^T) z + x S with S += y^T z (fla::walk_fwd_kernel's roles)
fla::WalkParams lower_walk_params(const WalkPlan &wp, const View &x, const View &y, const View &z, const View &out,
                                  int64_t B, int64_t H, int64_t N, int64_t wxy, int64_t wz, const float *entry) {
    fla::WalkParams w{};
    w.q = x.ptr, w.k = y.ptr, w.v = z.ptr, w.o = const_cast<void *>(out.ptr);
    w.qs_b = x.strides[0], w.qs_h = x.strides[1], w.qs_n = x.strides[2];
    w.ks_b = y.strides[0], w.ks_h = y.strides[1], w.ks_n = y.strides[2];
    w.vs_b = z.strides[0], w.vs_h = z.strides[1], w.vs_n = z.strides[2];
    w.os_b = out.strides[0], w.os_h = out.strides[1], w.os_n = out.strides[2];
    w.H = (int32_t)H, w.N = (int32_t)N, w.BH = (int32_t)(B * H), w.wqk = (int32_t)wxy, w.wv = (int32_t)wz;
    w.n_chunks = (int32_t)wp.n_chunks, w.seg_chunks = (int32_t)wp.seg_chunks, w.n_seg = (int32_t)wp.n_seg;
    w.init = wp.n_seg > 1 ? entry : nullptr;
    return w;
}

// the reverse walk that computes dQ, dK and dV
fla::WalkParams reverse_walk_params(const WalkPlan &wp, const View &go, const View &q, const View &k, const View &v, const View &dq,
                                    const View &dk, const View &dvv, int64_t B, int64_t H, int64_t N, int64_t wqk, int64_t wv) {
    fla::WalkParams r{};
    r.q = q.ptr, r.k = k.ptr, r.v = v.ptr, r.go = go.ptr;
    r.dq = const_cast<void *>(dq.ptr), r.dk = const_cast<void *>(dk.ptr), r.dv = const_cast<void *>(dvv.ptr);
    r.qs_b = q.strides[0], r.qs_h = q.strides[1], r.qs_n = q.strides[2];
    r.ks_b = k.strides[0], r.ks_h = k.strides[1], r.ks_n = k.strides[2];
    r.vs_b = v.strides[0], r.vs_h = v.strides[1], r.vs_n = v.strides[2];
    r.gs_b = go.strides[0], r.gs_h = go.strides[1], r.gs_n = go.strides[2];
    r.dqs_b = dq.strides[0], r.dqs_h = dq.strides[1], r.dqs_n = dq.strides[2];
    r.dks_b = dk.strides[0], r.dks_h = dk.strides[1], r.dks_n = dk.strides[2];
    r.dvs_b = dvv.strides[0], r.dvs_h = dvv.strides[1], r.dvs_n = dvv.strides[2];
    r.H = (int32_t)H, r.N = (int32_t)N, r.BH = (int32_t)(B * H), r.wqk = (int32_t)wqk, r.wv = (int32_t)wv;
    r.n_chunks = (int32_t)wp.n_chunks, r.seg_chunks = (int32_t)wp.seg_chunks, r.n_seg = (int32_t)wp.n_seg;
    return r;
}

fla::WalkRowsOut rows_out(const View &t, int64_t width) {
    return {const_cast<void *>(t.ptr), t.strides[0], t.strides[1], t.strides[2], (int32_t)width};
}
// ... its results to the caller's rows
void results_to_rows(fla::WalkParams &r, AnyRows &any) {
    r.any_rows = 1, any.done = true;
    if (r.dq) r.rows_dq = rows_out(*any.dq, any.dqk);
    r.rows_dk = rows_out(*any.dk, any.dqk), r.rows_dv = rows_out(*any.dv, any.wv);
    r.dq = r.dk = r.dv = nullptr;
}

bool wide_fast_path(const View &q, const View &k, const View &v, const View &o, int64_t B, int64_t H, int64_t N,
                    int64_t dqk, int64_t dv) {
    return fla::fast_path_ok(make_params(q, k, v, o, B, H, N, 128, dv, 0)) &&
           fla::fast_path_ok(make_params(column_half(q, 1), column_half(k, 1), v, o, B, H, N, dqk - 128, dv, 0));
}

int wide_forward(const WidePlan &wide, const View &q, const View &k, const View &v, const View &o, int64_t B, int64_t H,
                 int64_t N, int64_t dqk, int64_t dv, int dtype, void *state_out, void *workspace, hipStream_t s) {
    const WalkPlan &wp = wide.wp;
    char *ws = static_cast<char *>(workspace);
    const float *entry[2] = {nullptr, nullptr};
    // A few segments more than two: no scan -- the walk adds up the totals of the segments before its own as it
    // starts (three of each half in flight together) and writes the entry state it formed for backward
    // (B 4, H 16, N 4096, D_qk 256, D_v 64, four segments: 0.273 -> 0.267 ms per forward + backward, and 0.264 with
    // the reverse walk doing the same).
    const bool sum_on_load = sums_on_load(wp, dv <= 64 ? kSumOnLoadWide : kSumOnLoadMost);
    float *keep[2] = {nullptr, nullptr};
    if (wp.n_seg > 1) {
        // (kept for backward when there is a state buffer: each half's entry states, its final state behind them;
        // otherwise, and the totals that the walk adds up, in the workspace)
        void *work[2];
        for (int h = 0; h < 2; ++h) {
            if (state_out) keep[h] = reinterpret_cast<float *>(static_cast<char *>(state_out) + h * wp.saved_bytes);
            work[h] = keep[h] && !sum_on_load ? static_cast<void *>(keep[h])
                                              : static_cast<void *>(ws + h * wp.work_bytes);
        }
        float *const none[2] = {nullptr, nullptr};
        if (int rc = wide_entry_states(wp, k, v, B, H, N, dqk, dv, dtype, 0, work, sum_on_load ? none : keep, entry, s,
                                       sum_on_load, dv <= 64))
            return rc;
    }
    // one walk over both halves (the second one's columns start 128 elements into q's and k's rows)
    fla::WalkParams w = lower_walk_params(wp, q, k, v, o, B, H, N, 128, dv, entry[0]);
    w.wqk2 = (int32_t)(dqk - 128), w.init2 = wp.n_seg > 1 ? entry[1] : nullptr;
    if (sum_on_load) w.init_is_totals = 1, w.entry_out = keep[0], w.entry_out2 = keep[1];
    if (state_out) {  // (behind each half's entry states: its state after the last chunk)
        w.total_out = reinterpret_cast<float *>(static_cast<char *>(state_out) + wp.entry_bytes);
        w.total_out2 = reinterpret_cast<float *>(static_cast<char *>(state_out) + wp.saved_bytes + wp.entry_bytes);
    }
    return fla::walk_fwd_wide(dtype, w, s) == hipSuccess ? FLA_OK : FLA_ERR_LAUNCH;
}

// With forward's states at hand and a narrow v: one reverse walk over both halves, dQ included, whose state goes
// backwards by subtraction from the state at the segment's end (walk_bwd_rev_wide_kernel).  `causal`, a wider v or no states:
// dQ_h by forward-direction walks.  Backward at B 4, H 16, N 4096: 256 / 64 176 us in one walk, 199 in three; 256 / 128 297 us
// as a reverse walk per half, the second adding to the first one's dV in memory, 279 us in three walks.
int wide_backward(const WidePlan &wide, const View &go, const View &q, const View &k, const View &v, const View &dq,
                  const View &dk, const View &dvv, int64_t B, int64_t H, int64_t N, int64_t dqk, int64_t dv, int dtype,
                  const void *state_in, void *workspace, hipStream_t s, bool causal, bool wide_out, AnyRows *any) {
    const WalkPlan &wp = wide.wp;
    char *ws = static_cast<char *>(workspace);
    const bool one_walk = state_in && dv <= 64 && !causal;
    // entry states of both halves up front: Q_h^T dO over the segments after, and -- when forward's are not
    // at hand -- K_h^T V over the segments before
    const float *fwd_entries[2] = {nullptr, nullptr}, *entries[2] = {nullptr, nullptr};
    // (the reverse walk adds up the totals of the segments after its own itself, as forward does)
    const bool rev_sums_on_load = sums_on_load(wp, dv <= 64 ? kSumOnLoadWide : kSumOnLoadMost);
    // dQ's walks add up their halves' totals of Q^T dO on their way (WalkParams::r_totals).  A totals kernel in front -> this: 256 / 64,
    // B H 32, N 2048 104.5 -> 101.0 us, B H 64, N 4096 293 -> 288.  With a v above 64 columns a walk holds two full states: 256 / 128 eight
    // segments or more 159.8 -> 155.5 (B H 32, N 2048), four 399 -> 403 (B H 64, N 4096), ten short ones 130.6 -> 130.4; and there
    // only with more than 64 columns in q / k's second half too: a v above 64 columns against a half of at most 64 has no such variant
    // of the walk.  bf16 alone: two sets of four tiles and the state are all of the LDS, and an fp16 walk's scale needs a place there
    const bool dq_walk_sums = !one_walk && (dv <= 64 || (dqk > 192 && wp.n_seg >= 8)) && wp.n_seg > 2 && dtype == FLA_DTYPE_BF16;
    if (wp.n_seg > 1) {
        float *const none[2] = {nullptr, nullptr};
        if (state_in) {
            for (int h = 0; h < 2; ++h)
                fwd_entries[h] = reinterpret_cast<const float *>(static_cast<const char *>(state_in) + h * wp.saved_bytes);
        } else {
            void *const work[2] = {ws + 2 * wp.work_bytes, ws + 3 * wp.work_bytes};
            if (int rc = wide_entry_states(wp, k, v, B, H, N, dqk, dv, dtype, 0, work, none, fwd_entries, s, false, dv <= 64))
                return rc;
        }
        void *const work[2] = {ws, ws + wp.work_bytes};
        if (dq_walk_sums) {
            for (int h = 0; h < 2; ++h) entries[h] = static_cast<const float *>(work[h]);
        } else if (int rc = wide_entry_states(wp, q, go, B, H, N, dqk, dv, dtype, 1, work, none, entries, s, rev_sums_on_load, dv <= 64)) {
            return rc;
        }
    }
    fla::WalkParams r = reverse_walk_params(wp, go, q, k, v, dq, dk, dvv, B, H, N, 128, dv);
    r.wqk2 = (int32_t)(dqk - 128);
    r.init = entries[0], r.init2 = entries[1], r.init_is_totals = rev_sums_on_load, r.wide_out = wide_out;
    if (one_walk) {
        const char *half0 = static_cast<const char *>(state_in), *half1 = half0 + wp.saved_bytes;
        r.xinit = reinterpret_cast<const float *>(half0), r.xinit2 = reinterpret_cast<const float *>(half1);
        r.xtotal = reinterpret_cast<const float *>(half0 + wp.entry_bytes);
        r.xtotal2 = reinterpret_cast<const float *>(half1 + wp.entry_bytes);
        return fla::walk_bwd_rev_wide(dtype, r, s) == hipSuccess ? FLA_OK : FLA_ERR_LAUNCH;
    }
    // (dQ, dK straight to the caller's rows; dV's are aligned)
    if (any && dv <= 64 && any->wv == dv) any->done = true;
    const bool rows = any && any->done;
    // dQ_h = lower(dO V^T) K_h + dO S_h^T: the forward walk over (dO, V, K_h)
    for (int h = 0; h < 2; ++h) {
        const View dq_h{static_cast<const char *>(dq.ptr) + h * 128 * (wide_out ? 4 : 2), dq.strides};
        fla::WalkParams w = lower_walk_params(wp, go, v, column_half(k, h), dq_h, B, H, N, dv, h ? dqk - 128 : 128, fwd_entries[h]);
        w.init_transposed = 1, w.wide_out = wide_out;
        if (dq_walk_sums) {
            w.r_q = column_half(q, h).ptr, w.rs_b = q.strides[0], w.rs_h = q.strides[1], w.rs_n = q.strides[2];
            w.r_totals = const_cast<float *>(entries[h]), w.r_frags = rev_sums_on_load;
        }
        if (rows) w.any_rows = 1, w.rows_o = rows_out(column_half(*any->dq, h), h ? any->dqk - 128 : 128), w.o = nullptr;
        if (fla::walk_fwd(dtype, wp.D, w, s) != hipSuccess) return FLA_ERR_LAUNCH;
    }
    if (dq_walk_sums && !rev_sums_on_load) {
        float *const t0 = const_cast<float *>(entries[0]), *const t1 = const_cast<float *>(entries[1]);
        if (fla::walk_scan(t0, t0, B * H, (int)wp.n_seg, wp.D, dv <= 64 ? 64 : 128, 1, s, t1, t1) != hipSuccess) return FLA_ERR_LAUNCH;
    }
    r.dq = nullptr;
    if (rows) r.any_rows = 1, r.rows_dk = rows_out(*any->dk, any->dqk), r.dk = nullptr;
    return fla::walk_bwd_rev_wide(dtype, r, s) == hipSuccess ? FLA_OK : FLA_ERR_LAUNCH;
}

// ---- D_qk and D_v in (128, 256]: two column halves of q / k and two of v, four pairs with a state each.  O in its halves is a walk over
// both halves of q / k against a half of v; so are the gradients, each a sum over the halves of one pair of operands against a half
// of a third, held in fp32 from the first half to the second and rounded once: dQ ascending, from forward's entry states, and dV and dK
// in one launch descending (walk_fwd_wide_kernel, walk_rev_wide_kernel).  Nothing of a row reaches the dQ of the chunks before it, for callers
// with `causal` and without.  A launch works on two halves (grid y), the reverse one on four, so its plan has half as many segments again:
// the fewer states to move, which at B H = 16 outweigh the operands, the fewer chunks at a time.
// 256 / 256, forward + backward: one reverse walk per pair of halves, the second launch adding to the first one's results in memory -> this:
// B H 16, N 4096 235 -> 214 us, B H 64, N 4096 737 -> 623, B H 160, N 700 410 -> 319; dQ, dK and dV 0.87 to 0.93 of its errors.
WalkPlan quad_plan(int64_t B, int64_t H, int64_t N, int64_t dqk, int64_t dv, int64_t parts = 2) {
    if (dqk <= 128 || dqk > 256 || dv <= 128 || dv > 256) return WalkPlan{};
    return walk_plan(B, H, N, 128, 128, false, parts, true);
}

// four sets of entry states in one buffer, and in `state` four final states behind them
float *quad_finals(const WalkPlan &wp, const void *state) {
    return reinterpret_cast<float *>(static_cast<char *>(const_cast<void *>(state)) + 4 * wp.entry_bytes);
}

// the four pairs' segment totals of Y^T Z to `entries`, and the entry states over them where the walk does not add up
int quad_entry_states(const WalkPlan &wp, const View &y, const View &z, int64_t B, int64_t H, int64_t N, int64_t dy, int64_t dz,
                      int dtype, int reverse, float *entries, hipStream_t s, bool pairs = false) {
    fla::WalkTotalsParams tp{};
    tp.pairs = pairs;
    tp.y = y.ptr, tp.y2 = column_half(y, 1).ptr, tp.z = z.ptr;
    tp.totals = entries, tp.totals2 = entries + wp.entry_bytes / 4;
    tp.ys_b = y.strides[0], tp.ys_h = y.strides[1], tp.ys_n = y.strides[2];
    tp.zs_b = z.strides[0], tp.zs_h = z.strides[1], tp.zs_n = z.strides[2];
    tp.H = (int32_t)H, tp.N = (int32_t)N, tp.BH = (int32_t)(B * H);
    tp.dy = tp.dz = 128, tp.dy2 = (int32_t)(dy - 128), tp.dz2 = (int32_t)(dz - 128);
    tp.n_chunks = (int32_t)wp.n_chunks, tp.seg_chunks = (int32_t)wp.seg_chunks, tp.n_seg = (int32_t)wp.n_seg;
    tp.direct = wp.n_seg == 2, tp.frags = sums_on_load(wp);
    tp.seg_lo = reverse ? 1 : 0, tp.seg_hi = (int32_t)(reverse ? wp.n_seg : wp.n_seg - 1);
    if (fla::walk_totals(dtype, wp.D, tp, s) != hipSuccess) return FLA_ERR_LAUNCH;
    if (tp.direct || tp.frags) return FLA_OK;
    return fla::walk_scan(entries, entries, 4 * B * H, (int)wp.n_seg, wp.D, wp.D, reverse, s) == hipSuccess ? FLA_OK : FLA_ERR_LAUNCH;
}

int quad_forward(const WalkPlan &wp, const View &q, const View &k, const View &v, const View &o, int64_t B, int64_t H, int64_t N,
                 int64_t dqk, int64_t dv, int dtype, void *state_out, void *workspace, hipStream_t s) {
    const bool sum_on_load = sums_on_load(wp);
    const int64_t pair = wp.entry_bytes / 4;  // floats
    float *const kept = static_cast<float *>(state_out);
    float *const entries = kept && !sum_on_load ? kept : static_cast<float *>(workspace);
    if (wp.n_seg > 1)
        if (int rc = quad_entry_states(wp, k, v, B, H, N, dqk, dv, dtype, 0, entries, s)) return rc;
    fla::WalkParams w = lower_walk_params(wp, q, k, v, o, B, H, N, 128, 128, entries);
    w.quad = 1, w.wqk2 = (int32_t)(dqk - 128), w.wv2 = (int32_t)(dv - 128);
    w.init2 = w.init ? w.init + pair : nullptr;
    if (sum_on_load) w.init_is_totals = 1, w.entry_out = kept, w.entry_out2 = kept ? kept + pair : nullptr;
    if (kept) w.total_out = quad_finals(wp, kept), w.total_out2 = w.total_out + B * H * wp.D * wp.D;
    return fla::walk_fwd_wide(dtype, w, s) == hipSuccess ? FLA_OK : FLA_ERR_LAUNCH;
}

int quad_backward(const WalkPlan &wp, const View &go, const View &q, const View &k, const View &v, const View &dq, const View &dk,
                  const View &dvv, int64_t B, int64_t H, int64_t N, int64_t dqk, int64_t dv, int dtype, const void *state_in,
                  void *workspace, hipStream_t s) {
    // dQ in its halves: the forward walk over (dO, V, K), from forward's entry states read transposed
    fla::WalkParams w = lower_walk_params(wp, go, v, k, dq, B, H, N, 128, 128, static_cast<const float *>(state_in));
    w.quad = 1, w.wqk2 = (int32_t)(dv - 128), w.wv2 = (int32_t)(dqk - 128), w.init_transposed = 1;
    w.init2 = w.init ? w.init + 2 * (wp.entry_bytes / 4) : nullptr;  // (the first half of k against v's second)
    if (fla::walk_fwd_wide(dtype, w, s) != hipSuccess) return FLA_ERR_LAUNCH;
    // dV and dK in their halves, four workgroups to a segment
    const WalkPlan rp = quad_plan(B, H, N, dqk, dv, 4);
    float *const entries = static_cast<float *>(workspace);
    if (rp.n_seg > 1)
        if (int rc = quad_entry_states(rp, q, go, B, H, N, dqk, dv, dtype, 1, entries, s, true)) return rc;
    fla::WalkParams r = reverse_walk_params(rp, go, q, k, v, dq, dk, dvv, B, H, N, 128, 128);
    r.quad = 1, r.wqk2 = (int32_t)(dqk - 128), r.wv2 = (int32_t)(dv - 128);
    r.init = rp.n_seg > 1 ? entries : nullptr, r.init2 = r.init ? r.init + rp.entry_bytes / 4 : nullptr, r.init_is_totals = sums_on_load(rp);
    return fla::walk_rev_wide(dtype, r, s) == hipSuccess ? FLA_OK : FLA_ERR_LAUNCH;
}

// both column halves of (x4, o4) = (v, O) / (dO, dV) with (a, b) = (q, k) / (dQ, dK) qualify for their plans' kernels
bool vsplit_fast_path(const VSplit &vs, const View &a, const View &b, const View &x4, const View &o4, int64_t B, int64_t H,
                      int64_t N, int64_t dqk) {
    for (int j = 0; j < 2; ++j) {
        const int64_t d = j == 0 ? 128 : vs.dv1;
        const View xj = v_half(x4, j), oj = v_half(o4, j);
        const bool ok = dqk > 128 ? wide_fast_path(a, b, xj, oj, B, H, N, dqk, d)
                                  : fla::fast_path_ok(make_params(a, b, xj, oj, B, H, N, dqk, d, 0));
        if (!ok) return false;
    }
    return true;
}

int chunked_forward(const View &q, const View &k, const View &v, const View &o, int64_t B, int64_t H, int64_t N,
                    int64_t dqk, int64_t dv, int dtype, void *state_out, int32_t *state_valid, void *workspace,
                    int64_t workspace_bytes, void *stream, int fmap, const View *mapped, bool *mapped_done, WalkNorm *nx,
                    AnyRows *any);
int chunked_backward(const View &go, const View &q, const View &k, const View &v, const View &dq, const View &dk,
                     const View &dvv, int64_t B, int64_t H, int64_t N, int64_t dqk, int64_t dv, int dtype,
                     const void *state_in, void *workspace, int64_t workspace_bytes, void *stream, int fmap, WalkNorm *nx,
                     bool causal, bool wide_out, AnyRows *any, bool scaled_state);

// fmap != 0 (feature_forward below): q and k hold the arguments xq, xk of the feature map phi, and
// `mapped` = {phi(xq), phi(xk)} are outputs: the state kernel maps xk as it loads it and writes
// phi(xk), which the main kernel then reads as its Y operand; the main kernel maps its X rows xq
// and writes phi(xq).  Only the shared-state fast path does this; *mapped_done says whether it ran.
int chunked_forward(const View &q, const View &k, const View &v, const View &o, int64_t B, int64_t H, int64_t N,
                    int64_t dqk, int64_t dv, int dtype, void *state_out, int32_t *state_valid, void *workspace,
                    int64_t workspace_bytes, void *stream, int fmap = 0, const View *mapped = nullptr,
                    bool *mapped_done = nullptr, WalkNorm *nx = nullptr, AnyRows *any = nullptr) {
    if (state_valid) *state_valid = 0;
    if (nx) nx->fused = nx->dk_pending = false;
    const View all[] = {q, k, v, o};
    for (const View &t : all)
        if (int rc = check_view(t)) return rc;
    if (int rc = check_alias_fwd(q, k, v, o, B, H, N, dqk, dv)) return rc;
    if (B == 0 || H == 0 || N == 0) return FLA_OK;
    if (!fmap && !nx) {
        // a v wider than 128 columns: its two column halves, one after the other (the second half's state behind the first's)
        const VSplit vs = vsplit_plan(B, H, N, dqk, dv);
        if (vs.ok && vsplit_fast_path(vs, q, k, v, o, B, H, N, dqk)) {
            if (!workspace || reinterpret_cast<uintptr_t>(workspace) % 16 != 0 ||
                workspace_bytes < vsplit_inner_bytes(vs, B, H, N, dqk))
                return FLA_ERR_WORKSPACE;
            if (state_out && reinterpret_cast<uintptr_t>(state_out) % 16 != 0) return FLA_ERR_WORKSPACE;
            if (const WalkPlan quad = quad_plan(B, H, N, dqk, dv); quad.ok) {  // (fits: half the segments of vs's plans)
                if (int rc = quad_forward(quad, q, k, v, o, B, H, N, dqk, dv, dtype, state_out, workspace,
                                          static_cast<hipStream_t>(stream)))
                    return rc;
                if (state_out && state_valid) *state_valid = 1;
                return FLA_OK;
            }
            int32_t valid[2] = {0, 0};
            for (int j = 0; j < 2; ++j) {
                void *st = state_out ? static_cast<char *>(state_out) + j * vs.state0 : nullptr;
                if (int rc = chunked_forward(q, k, v_half(v, j), v_half(o, j), B, H, N, dqk, j == 0 ? 128 : vs.dv1, dtype, st,
                                             &valid[j], workspace, workspace_bytes, stream, 0, nullptr, nullptr, nullptr))
                    return rc;
            }
            if (state_out && state_valid) *state_valid = valid[0] && valid[1];
            return FLA_OK;
        }
        const WidePlan wide = wide_plan(B, H, N, dqk, dv);
        if (wide.ok && wide_fast_path(q, k, v, o, B, H, N, dqk, dv)) {
            if (!workspace || reinterpret_cast<uintptr_t>(workspace) % 16 != 0 || workspace_bytes < wide_workspace_bytes(wide))
                return FLA_ERR_WORKSPACE;
            if (state_out && reinterpret_cast<uintptr_t>(state_out) % 16 != 0) return FLA_ERR_WORKSPACE;
            if (int rc = wide_forward(wide, q, k, v, o, B, H, N, dqk, dv, dtype, state_out, workspace,
                                      static_cast<hipStream_t>(stream)))
                return rc;
            if (state_out && state_valid) *state_valid = 1;
            return FLA_OK;
        }
    }
    const WalkPlan wp = walk_plan(B, H, N, dqk, dv, !fmap && !nx);
    if (wp.ok && fla::fast_path_ok(make_params(q, k, v, o, B, H, N, dqk, dv, 0)) &&
        (!fmap || fla::fast_path_ok(make_params(mapped[0], mapped[1], v, o, B, H, N, dqk, dv, 0)))) {
        // the segments' entry states; with a feature map the same kernel maps xk as it loads it and
        // writes phi(xk), which the walk then reads (so it runs for a single segment as well)
        const bool by_columns = forward_by_columns(wp, B * H, N, dqk, dv, dtype, !fmap && !nx);
        const bool need_totals = wp.n_seg > 1 || fmap;
        // D = 128: the entry states (and the state after the last chunk) are what backward gets, so the scan writes
        // them to state_out (the totals themselves are computed there, and no workspace is used);
        // padded head dims up to 64 hand over the 16-bit state of every chunk instead
        const bool in_state = state_out && wp.split;
        // D = 128, a few segments more than two: the totals go to the workspace, the walk adds them up itself as it starts
        // and writes the entry states it formed to state_out -- no scan launch
        // (a caller may have brought a state buffer and no workspace: then a scan in the former -- but for the plain operator up to
        // kSumOnLoadWorkspace segments, which is refused without its workspace: the reason stands there)
        const bool has_work = workspace && reinterpret_cast<uintptr_t>(workspace) % 16 == 0 && workspace_bytes >= wp.work_bytes;
        const bool sum_on_load = wp.split && sums_on_load(wp) && (!in_state || has_work || (!fmap && !nx && wp.n_seg <= kSumOnLoadWorkspace));
        if (need_totals && (!in_state || sum_on_load) && !has_work) return FLA_ERR_WORKSPACE;
        if (state_out && reinterpret_cast<uintptr_t>(state_out) % 16 != 0) return FLA_ERR_WORKSPACE;
        hipStream_t s = static_cast<hipStream_t>(stream);
        const float *entry = nullptr;
        if (need_totals && !by_columns)
            if (int rc = walk_entry_states(wp, k, v, B, H, N, dqk, dv, dtype, 0,
                                           in_state && !sum_on_load ? state_out : workspace,
                                           in_state && !sum_on_load ? static_cast<float *>(state_out) : nullptr, &entry, s,
                                           fmap, fmap ? &mapped[1] : nullptr, nullptr, sum_on_load, false,
                                           nx ? static_cast<float *>(nx->vec) : nullptr, !state_out))
                return rc;
        const View &kk = fmap ? mapped[1] : k;
        fla::WalkParams w{};
        if (fmap) {
            w.fmap = fmap, w.qmap_out = const_cast<void *>(mapped[0].ptr);
            w.qo_b = mapped[0].strides[0], w.qo_h = mapped[0].strides[1], w.qo_n = mapped[0].strides[2];
        }
        w.q = q.ptr, w.k = kk.ptr, w.v = v.ptr, w.o = const_cast<void *>(o.ptr);
        w.qs_b = q.strides[0], w.qs_h = q.strides[1], w.qs_n = q.strides[2];
        w.ks_b = kk.strides[0], w.ks_h = kk.strides[1], w.ks_n = kk.strides[2];
        w.vs_b = v.strides[0], w.vs_h = v.strides[1], w.vs_n = v.strides[2];
        w.os_b = o.strides[0], w.os_h = o.strides[1], w.os_n = o.strides[2];
        w.H = (int32_t)H, w.N = (int32_t)N, w.BH = (int32_t)(B * H), w.wqk = (int32_t)dqk, w.wv = (int32_t)dv;
        w.n_chunks = (int32_t)wp.n_chunks, w.seg_chunks = (int32_t)wp.seg_chunks, w.n_seg = (int32_t)wp.n_seg;
        w.init = wp.n_seg > 1 ? entry : nullptr, w.saved = in_state ? nullptr : state_out;
        if (w.saved && dtype == FLA_DTYPE_F16 && !nx) w.saved_scale = saved_scales(state_out, B, H, N, dqk, dv);
        if (sum_on_load) w.init_is_totals = 1, w.entry_out = in_state ? static_cast<float *>(state_out) : nullptr;
        if (by_columns) {  // (the state buffer is that of two segments all the same)
            w.cols = 1, w.n_seg = 1, w.seg_chunks = w.n_chunks, w.init = nullptr;
            w.mid_out = in_state ? static_cast<float *>(state_out) : nullptr, w.mid_chunk = (int32_t)wp.seg_chunks;
        }
        if (any && wp.split) {
            w.any_rows = 1, w.rows_o = rows_out(*any->o, any->wv), w.o = nullptr, any->done = true;
        }
        if (in_state) w.total_out = reinterpret_cast<float *>(static_cast<char *>(state_out) + wp.entry_bytes);
        if (nx) {  // the normaliser inside the walk, which carries the running sum of k from the segments' totals of it
            // (kept for backward, at the entry of every chunk, behind the state when there is one)
            w.denom = nx->denom, w.eps = nx->eps, w.vsum = wp.n_seg > 1 ? static_cast<const float *>(nx->vec) : nullptr;
            if (state_out) w.zc_out = reinterpret_cast<float *>(static_cast<char *>(state_out) + state_core_bytes(B, H, N, dqk, dv));
            nx->fused = true;
        }
        if (fla::walk_fwd(dtype, wp.D, w, s) != hipSuccess) return FLA_ERR_LAUNCH;
        if (mapped_done) *mapped_done = true;
        if (state_out && state_valid) *state_valid = 1;
        return FLA_OK;
    }
    TriParams p = make_params(q, fmap ? mapped[1] : k, v, o, B, H, N, dqk, dv, 0);
    // with a feature map: xk is read by the state kernel's loads, and phi(xq), phi(xk) are written with 16-byte stores
    const bool k_fast = !fmap || (fla::fast_path_ok(make_params(q, k, v, o, B, H, N, dqk, dv, 0)) &&
                                  fla::fast_path_ok(make_params(mapped[0], mapped[1], v, o, B, H, N, dqk, dv, 0)));
    if (!states_shareable(dqk, dv, N) || !fla::fast_path_ok(p) || !k_fast) {
        if (fmap) return FLA_OK;  // *mapped_done stays false: the caller maps with a pass of its own
        return run_tri_chunked(q, k, v, o, B, H, N, dqk, dv, 0, dtype, workspace, workspace_bytes, stream);
    }
    if (fmap) {
        p.map_x = fmap, p.xmap_out = const_cast<void *>(mapped[0].ptr);
        p.xo_b = mapped[0].strides[0], p.xo_h = mapped[0].strides[1], p.xo_n = mapped[0].strides[2];
    }
    const int64_t sb = shared_state_bytes(B, H, N, dqk, dv);
    if (!workspace || reinterpret_cast<uintptr_t>(workspace) % 16 != 0 || workspace_bytes < sb * (state_out ? 2 : 3))
        return FLA_ERR_WORKSPACE;
    if (state_out && reinterpret_cast<uintptr_t>(state_out) % 16 != 0) return FLA_ERR_WORKSPACE;
    float *w = static_cast<float *>(workspace);
    void *state = state_out ? state_out : static_cast<char *>(workspace) + 2 * sb;
    if (int rc = chunk_states(k, v, B, H, N, dqk, dv, 0, dtype, w, state, stream, fmap, fmap ? &mapped[1] : nullptr))
        return rc;
    if (int rc = chunk_main(p, dqk, dv, dtype, state, 0, stream)) return rc;
    if (mapped_done) *mapped_done = true;
    // (where the walk kernels exist, backward reads a handed-over state in THEIR format: the 256-row
    // chunks' state written here is not offered, and backward computes its own)
    if (state_out && state_valid && !wp.ok) *state_valid = 1;
    return FLA_OK;
}

// whether walks that can store their results in fp32 (FLA_GRADS_F32) take a backward of these sizes; `plain`: without feature map and
// normaliser
bool wide_grads_sizes(int64_t B, int64_t H, int64_t N, int64_t dqk, int64_t dv, bool plain, bool with_state) {
    if (dqk % 8 || dv % 8 || dv > 128) return false;
    if (dqk > 128) return plain && dv <= 64 && wide_plan(B, H, N, dqk, dv).ok;
    const WalkPlan wp = walk_plan(B, H, N, dqk, dv, plain);
    return wp.ok && (wp.split || with_state) && (states_shareable(dqk, dv, N) || pad_index(dqk) != pad_index(dv));
}

// ... and of these operands
bool wide_grads_walk(const View &go, const View &q, const View &k, const View &v, const View &dq, const View &dk, const View &dvv,
                     int64_t B, int64_t H, int64_t N, int64_t dqk, int64_t dv, int dtype, const void *state_in, bool plain) {
    if (dtype != FLA_DTYPE_BF16 || !wide_grads_sizes(B, H, N, dqk, dv, plain, state_in != nullptr)) return false;
    // (a (b, h) of a result stays within the 1 GiB that a descriptor's offsets reach, as 16-bit operands do)
    for (const View *t : {&dq, &dk, &dvv})
        if (N * t->strides[2] * 4 > fla::kMaxFastExtent) return false;
    if (dqk > 128) return wide_fast_path(q, k, v, go, B, H, N, dqk, dv) && wide_fast_path(dq, dk, dvv, dvv, B, H, N, dqk, dv);
    return fla::fast_path_ok(make_params(go, v, k, dq, B, H, N, dv, dqk, 0)) &&
           fla::fast_path_ok(make_params(k, q, go, dvv, B, H, N, dqk, dv, 1)) &&
           fla::fast_path_ok(make_params(v, go, q, dk, B, H, N, dv, dqk, 1));
}

// whether the walk kernels take the normalised backward of these operands
bool norm_walks_backward(const View &go, const View &q, const View &k, const View &v, const View &dq, const View &dk,
                         const View &dvv, int64_t B, int64_t H, int64_t N, int64_t dqk, int64_t dv, const void *state_in) {
    const WalkPlan wp = walk_plan(B, H, N, dqk, dv);
    return wp.ok && (state_in || wp.split) && states_shareable(dqk, dv, N) && fla::fast_path_ok(make_params(go, v, k, dq, B, H, N, dv, dqk, 0)) &&
           fla::fast_path_ok(make_params(k, q, go, dvv, B, H, N, dqk, dv, 1)) &&
           fla::fast_path_ok(make_params(v, go, q, dk, B, H, N, dv, dqk, 1));
}

// `causal` (D_v up to 128): with forward's states at hand, too, dQ comes from a walk in forward direction (and dK, dV from
// one in reverse), never by subtraction from a later state: nothing of a row reaches the dQ of the chunks before it.
// Backward at D = 128, one reverse walk against two walks: B H 128, N 4096 274 / 292 us; B H 16, N 4096 53 / 58; B H 256, N 1024
// 124 / 128; B H 4, N 8192 66 / 73; 128 / 64, B H 64, N 4096 98 / 113.
int chunked_backward(const View &go, const View &q, const View &k, const View &v, const View &dq, const View &dk,
                     const View &dvv, int64_t B, int64_t H, int64_t N, int64_t dqk, int64_t dv, int dtype,
                     const void *state_in, void *workspace, int64_t workspace_bytes, void *stream, int fmap = 0,
                     WalkNorm *nx = nullptr, bool causal = false, bool wide_out = false, AnyRows *any = nullptr,
                     bool scaled_state = true) {  // (the state is not a normalised forward's: saved_scales)
    if (nx) nx->fused = nx->dk_pending = false;
    const View all[] = {go, q, k, v, dq, dk, dvv};
    for (const View &t : all)
        if (int rc = check_view(t)) return rc;
    if (int rc = check_alias_bwd(go, q, k, v, nullptr, dq, dk, dvv, B, H, N, dqk, dv, wide_out)) return rc;
    if (B == 0 || H == 0 || N == 0) return FLA_OK;
    if (wide_out && !wide_grads_walk(go, q, k, v, dq, dk, dvv, B, H, N, dqk, dv, dtype, state_in, !fmap && !nx))
        return FLA_ERR_UNSUPPORTED;
    // fmap != 0: q and k hold y = phi(x) (what the forward pass wrote), and the gradients leave as
    // gradients with respect to x: dQ and dK are multiplied by phi'(x), computed from y -- in the
    // kernels' epilogue on the fast path, by a pass of its own after the products otherwise.
    TriParams pq = make_params(go, v, k, dq, B, H, N, dv, dqk, 0);   // dQ = lower(dO V^T) K
    TriParams pv = make_params(k, q, go, dvv, B, H, N, dqk, dv, 1);  // dV = upper(K Q^T) dO
    TriParams pk = make_params(v, go, q, dk, B, H, N, dv, dqk, 1);   // dK = upper(V dO^T) Q
    if (!fmap && !nx) {
        // a v wider than 128 columns: dV of each column half; dQ and dK of the second half to scratch tensors, then added
        const VSplit vs = vsplit_plan(B, H, N, dqk, dv);
        if (vs.ok && vsplit_fast_path(vs, q, k, v, go, B, H, N, dqk) && vsplit_fast_path(vs, dq, dk, dvv, dvv, B, H, N, dqk)) {
            const int64_t inner = vsplit_inner_bytes(vs, B, H, N, dqk);
            if (!workspace || reinterpret_cast<uintptr_t>(workspace) % 16 != 0 || workspace_bytes < inner + 2 * vs.temp_bytes)
                return FLA_ERR_WORKSPACE;
            if (state_in && reinterpret_cast<uintptr_t>(state_in) % 16 != 0) return FLA_ERR_WORKSPACE;
            // (without forward's states the halves of v go one after the other: each needs them again, and a walk of its own for dQ)
            if (const WalkPlan quad = quad_plan(B, H, N, dqk, dv); quad.ok && state_in)
                return quad_backward(quad, go, q, k, v, dq, dk, dvv, B, H, N, dqk, dv, dtype, state_in, workspace,
                                     static_cast<hipStream_t>(stream));
            const int64_t temp_strides[4] = {H * N * dqk, N * dqk, dqk, 1};
            const View tq{static_cast<char *>(workspace) + inner, temp_strides};
            const View tk{static_cast<char *>(workspace) + inner + vs.temp_bytes, temp_strides};
            for (int j = 0; j < 2; ++j) {
                const void *st = state_in ? static_cast<const char *>(state_in) + j * vs.state0 : nullptr;
                if (int rc = chunked_backward(v_half(go, j), q, k, v_half(v, j), j == 0 ? dq : tq, j == 0 ? dk : tk,
                                              v_half(dvv, j), B, H, N, dqk, j == 0 ? 128 : vs.dv1, dtype, st, workspace, inner,
                                              stream, 0, nullptr, causal))
                    return rc;
            }
            if (int rc = launch_feature_pass(3, 0, tq, dq, B, H, N, dqk, dtype, stream)) return rc;
            return launch_feature_pass(3, 0, tk, dk, B, H, N, dqk, dtype, stream);
        }
        const WidePlan wide = wide_plan(B, H, N, dqk, dv);
        if (wide.ok && wide_fast_path(q, k, v, go, B, H, N, dqk, dv) && wide_fast_path(dq, dk, dvv, dvv, B, H, N, dqk, dv)) {
            if (!workspace || reinterpret_cast<uintptr_t>(workspace) % 16 != 0 || workspace_bytes < wide_workspace_bytes(wide))
                return FLA_ERR_WORKSPACE;
            if (state_in && reinterpret_cast<uintptr_t>(state_in) % 16 != 0) return FLA_ERR_WORKSPACE;
            return wide_backward(wide, go, q, k, v, dq, dk, dvv, B, H, N, dqk, dv, dtype, state_in, workspace,
                                 static_cast<hipStream_t>(stream), causal, wide_out, any);
        }
    }
    // (with the normaliser's terms still to be added by the caller, so is the slope)
    const int fmap_late = nx ? 0 : fmap;
    const WalkPlan wp = walk_plan(B, H, N, dqk, dv, !fmap && !nx);
    // (what forward saved is in the walks' format; at D = 128 the entry states are cheap to recompute)
    const bool walk = wp.ok && (state_in || wp.split);  // (norm_walks_backward: the same)
    // (padded widths that differ: the walks or product by product -- the 256-row chunks share states between equal ones only)
    const bool mixed_walk = walk && pad_index(dqk) != pad_index(dv);
    if ((!states_shareable(dqk, dv, N) && !mixed_walk) || !fla::fast_path_ok(pq) || !fla::fast_path_ok(pv) ||
        !fla::fast_path_ok(pk)) {
        if (int rc = run_tri_chunked(go, v, k, dq, B, H, N, dv, dqk, 0, dtype, workspace, workspace_bytes, stream))
            return rc;
        if (int rc = run_tri_chunked(k, q, go, dvv, B, H, N, dqk, dv, 1, dtype, workspace, workspace_bytes, stream))
            return rc;
        if (int rc = run_tri_chunked(v, go, q, dk, B, H, N, dv, dqk, 1, dtype, workspace, workspace_bytes, stream))
            return rc;
        if (!fmap_late) return FLA_OK;
        if (int rc = launch_feature_pass(2, fmap, q, dq, B, H, N, dqk, dtype, stream)) return rc;
        return launch_feature_pass(2, fmap, k, dk, B, H, N, dqk, dtype, stream);
    }
    // the normalised forward left zc behind its state
    const float *zc_saved = nx && state_in ? reinterpret_cast<const float *>(static_cast<const char *>(state_in) +
                                                                           state_core_bytes(B, H, N, dqk, dv))
                                           : nullptr;
    if (walk && wp.split) {
        // workspace: totals and entry states of Q^T dO; behind them those of K^T V when forward's are not given
        if (wp.n_seg > 1 && (!workspace || reinterpret_cast<uintptr_t>(workspace) % 16 != 0 ||
                             workspace_bytes < wp.work_bytes * (state_in ? 1 : 2)))
            return FLA_ERR_WORKSPACE;
        if (state_in && reinterpret_cast<uintptr_t>(state_in) % 16 != 0) return FLA_ERR_WORKSPACE;
        hipStream_t s = static_cast<hipStream_t>(stream);
        const float *entry = nullptr;
        // with forward's states at hand (and without the normaliser): one reverse walk
        const bool one_walk = state_in && !nx && !causal;
        // (the reverse walk adds up the totals of the segments after its own itself, as forward does)
        const bool rev_sums_on_load = (one_walk || causal || nx) && sums_on_load(wp);
        float *const rcv = nx ? reinterpret_cast<float *>(static_cast<char *>(nx->vec) + walk_vec_bytes(B, H, N, dqk, dv)) : nullptr;
        // dQ's walk adds up the segments' totals of Q^T dO on its way (WalkParams::r_totals, figures there; bf16 alone: an fp16 walk's
        // scale has no place in the LDS beside two sets of four tiles and the state)
        const bool dq_walk_sums = !one_walk && !nx && !fmap && wp.n_seg > 2 && dtype == FLA_DTYPE_BF16 && dqk > 64;
        const bool by_columns = !one_walk && walk_by_columns(wp, B * H, N, dqk, dv, !fmap && !nx);
        if (wp.n_seg > 1) {
            if (!state_in) {
                const float *fwd_entry = nullptr;
                if (int rc = walk_entry_states(wp, k, v, B, H, N, dqk, dv, dtype, 0, static_cast<char *>(workspace) + wp.work_bytes,
                                               nullptr, &fwd_entry, s))
                    return rc;
                state_in = fwd_entry;
            }
            if (!nx && !dq_walk_sums && !by_columns)
                if (int rc = walk_entry_states(wp, q, go, B, H, N, dqk, dv, dtype, 1, workspace, nullptr, &entry, s, 0, nullptr,
                                               nullptr, rev_sums_on_load))
                    return rc;
        }
        const float *zc = zc_saved;  // (running sum of k at the entry of every chunk)
        if (nx) {
            if (int rc = walk_grad_entry_states(wp, q, go, *nx, B, H, N, dqk, dv, dtype, workspace, rcv, &entry, rev_sums_on_load, s))
                return rc;
            if (!zc) {
                if (int rc = walk_chunk_vectors(wp, k, dqk, static_cast<float *>(nx->vec), B, H, N, dtype, s)) return rc;
                zc = static_cast<const float *>(nx->vec);
            }
        }
        if (one_walk) {
            fla::WalkParams r = reverse_walk_params(wp, go, q, k, v, dq, dk, dvv, B, H, N, dqk, dv);
            r.init = entry, r.fmap = fmap;  // (dQ, dK: the slopes from phi(xq), phi(xk) in the Q and K tiles)
            r.init_is_totals = rev_sums_on_load;
            r.xinit = static_cast<const float *>(state_in);
            r.xtotal = reinterpret_cast<const float *>(static_cast<const char *>(state_in) + wp.entry_bytes);
            r.wide_out = wide_out;
            if (any) results_to_rows(r, *any);
            return fla::walk_bwd_rev(dtype, wp.D, r, s) == hipSuccess ? FLA_OK : FLA_ERR_LAUNCH;
        }
        // dQ = lower(dO V^T) K + dO S^T: the forward walk over (dO, V, K), its states V^T K = S^T
        fla::WalkParams w{};
        w.q = go.ptr, w.k = v.ptr, w.v = k.ptr, w.o = const_cast<void *>(dq.ptr);
        w.qs_b = go.strides[0], w.qs_h = go.strides[1], w.qs_n = go.strides[2];
        w.ks_b = v.strides[0], w.ks_h = v.strides[1], w.ks_n = v.strides[2];
        w.vs_b = k.strides[0], w.vs_h = k.strides[1], w.vs_n = k.strides[2];
        w.os_b = dq.strides[0], w.os_h = dq.strides[1], w.os_n = dq.strides[2];
        w.H = (int32_t)H, w.N = (int32_t)N, w.BH = (int32_t)(B * H), w.wqk = (int32_t)dv, w.wv = (int32_t)dqk;
        w.n_chunks = (int32_t)wp.n_chunks, w.seg_chunks = (int32_t)wp.seg_chunks, w.n_seg = (int32_t)wp.n_seg;
        w.init = wp.n_seg > 1 ? static_cast<const float *>(state_in) : nullptr, w.init_transposed = 1;
        w.wide_out = wide_out;
        if (fmap) {  // q holds phi(xq): dQ leaves multiplied by the slope computed from it
            w.fmap = fmap, w.slope_y = q.ptr;
            w.sy_b = q.strides[0], w.sy_h = q.strides[1], w.sy_n = q.strides[2];
        }
        if (nx) w.dn = nx->dn, w.zc = zc, nx->fused = true;  // dQ's term of the normaliser inside its walk
        if (any) {
            w.any_rows = 1, w.rows_o = rows_out(*any->dq, any->dqk), w.o = nullptr;
        }
        if (dq_walk_sums) {
            w.r_q = q.ptr, w.rs_b = q.strides[0], w.rs_h = q.strides[1], w.rs_n = q.strides[2];
            w.r_totals = static_cast<float *>(workspace), w.r_frags = rev_sums_on_load;
            entry = w.r_totals;
        }
        if (fla::walk_fwd(dtype, wp.D, w, s) != hipSuccess) return FLA_ERR_LAUNCH;
        if (dq_walk_sums && !rev_sums_on_load &&
            fla::walk_scan(entry, static_cast<float *>(workspace), B * H, (int)wp.n_seg, wp.D, fla::walk_totals_cols(wp.D, (int)dqk, (int)dv), 1,
                           s) != hipSuccess)
            return FLA_ERR_LAUNCH;
        // dV, dK: the reverse walk over the same segments
        fla::WalkParams r{};
        r.q = q.ptr, r.k = k.ptr, r.v = v.ptr, r.go = go.ptr;
        r.dk = const_cast<void *>(dk.ptr), r.dv = const_cast<void *>(dvv.ptr);
        r.qs_b = q.strides[0], r.qs_h = q.strides[1], r.qs_n = q.strides[2];
        r.ks_b = k.strides[0], r.ks_h = k.strides[1], r.ks_n = k.strides[2];
        r.vs_b = v.strides[0], r.vs_h = v.strides[1], r.vs_n = v.strides[2];
        r.gs_b = go.strides[0], r.gs_h = go.strides[1], r.gs_n = go.strides[2];
        r.dks_b = dk.strides[0], r.dks_h = dk.strides[1], r.dks_n = dk.strides[2];
        r.dvs_b = dvv.strides[0], r.dvs_h = dvv.strides[1], r.dvs_n = dvv.strides[2];
        r.H = (int32_t)H, r.N = (int32_t)N, r.BH = (int32_t)(B * H), r.wqk = (int32_t)dqk, r.wv = (int32_t)dv;
        r.n_chunks = (int32_t)wp.n_chunks, r.seg_chunks = (int32_t)wp.seg_chunks, r.n_seg = (int32_t)wp.n_seg;
        r.init = entry, r.fmap = fmap;  // (dK: the slope from phi(xk) in the K tile)
        r.init_is_totals = rev_sums_on_load, r.wide_out = wide_out;
        if (by_columns) r.roles = 1, r.n_seg = 1, r.seg_chunks = r.n_chunks, r.init = nullptr;
        if (nx) r.dn = nx->dn, r.rc = wp.n_seg > 1 ? rcv : nullptr;  // dK's terms
        if (any) results_to_rows(r, *any);
        return fla::walk_dkdv(dtype, wp.D, r, s) == hipSuccess ? FLA_OK : FLA_ERR_LAUNCH;
    }
    if (walk) {  // (the states forward saved are per 128-row chunk: only this path reads them)
        if (wp.n_seg > 1 &&
            (!workspace || reinterpret_cast<uintptr_t>(workspace) % 16 != 0 || workspace_bytes < wp.work_bytes))
            return FLA_ERR_WORKSPACE;
        if (reinterpret_cast<uintptr_t>(state_in) % 16 != 0) return FLA_ERR_WORKSPACE;
        hipStream_t s = static_cast<hipStream_t>(stream);
        const float *entry = nullptr;
        if (wp.n_seg > 1 && !nx)
            if (int rc = walk_entry_states(wp, q, go, B, H, N, dqk, dv, dtype, 1, workspace, nullptr, &entry, s)) return rc;
        const View *gv = &go;
        fla::WalkParams w{};
        if (nx) {
            float *const rcv = reinterpret_cast<float *>(static_cast<char *>(nx->vec) + walk_vec_bytes(B, H, N, dqk, dv));
            // (g as aligned rows, as the walk's tile loads ask for, and not from the caches at a few heads: dO is formed where it is
            // used.  A dO written and read -> this, forward + backward, MB of dO, D = 64: 0.13 to 2.1 25.2 -> 25.8 us, 32.2 -> 32.6; 8.4
            // 45.8 -> 46.1, 50.5 -> 50.1, 64.0 -> 63.6; 12.6 57.6 -> 57.2; 16.8 71.8 -> 70.3; 33.6 130 -> 127)
            const bool keep_g = nx->vec16 && B * H * N * dv * 2 > (10 << 20) && fla::fast_path_ok(make_params(q, k, *nx->go, dvv, B, H, N, dqk, dv, 0));
            if (int rc = walk_grad_entry_states(wp, q, go, *nx, B, H, N, dqk, dv, dtype, workspace, rcv, &entry, false, s, keep_g)) return rc;
            gv = keep_g ? nx->go : &go, w.gn = keep_g ? nx->n : nullptr;
            w.dn = nx->dn, w.zc = zc_saved, w.rc = wp.n_seg > 1 ? rcv : nullptr;
            nx->fused = true;
        }
        w.fmap = fmap;  // q, k hold phi(x): the slopes come from the LDS tiles
        w.q = q.ptr, w.k = k.ptr, w.v = v.ptr, w.go = gv->ptr;
        w.dq = const_cast<void *>(dq.ptr), w.dk = const_cast<void *>(dk.ptr), w.dv = const_cast<void *>(dvv.ptr);
        w.qs_b = q.strides[0], w.qs_h = q.strides[1], w.qs_n = q.strides[2];
        w.ks_b = k.strides[0], w.ks_h = k.strides[1], w.ks_n = k.strides[2];
        w.vs_b = v.strides[0], w.vs_h = v.strides[1], w.vs_n = v.strides[2];
        w.gs_b = gv->strides[0], w.gs_h = gv->strides[1], w.gs_n = gv->strides[2];
        w.dqs_b = dq.strides[0], w.dqs_h = dq.strides[1], w.dqs_n = dq.strides[2];
        w.dks_b = dk.strides[0], w.dks_h = dk.strides[1], w.dks_n = dk.strides[2];
        w.dvs_b = dvv.strides[0], w.dvs_h = dvv.strides[1], w.dvs_n = dvv.strides[2];
        w.H = (int32_t)H, w.N = (int32_t)N, w.BH = (int32_t)(B * H), w.wqk = (int32_t)dqk, w.wv = (int32_t)dv;
        w.n_chunks = (int32_t)wp.n_chunks, w.seg_chunks = (int32_t)wp.seg_chunks, w.n_seg = (int32_t)wp.n_seg;
        w.init = entry;
        w.saved = const_cast<void *>(state_in);
        if (dtype == FLA_DTYPE_F16 && !nx && scaled_state) w.saved_scale = saved_scales(state_in, B, H, N, dqk, dv);
        w.wide_out = wide_out;
        return fla::walk_bwd(dtype, wp.D, w, s) == hipSuccess ? FLA_OK : FLA_ERR_LAUNCH;
    }
    if (wp.ok) state_in = nullptr;  // not in the 256-row chunks' format: recomputed below
    if (fmap_late) set_output_slope(pq, fmap, q), set_output_slope(pk, fmap, k);
    const int64_t sb = shared_state_bytes(B, H, N, dqk, dv);
    if (!workspace || reinterpret_cast<uintptr_t>(workspace) % 16 != 0 || workspace_bytes < sb * (state_in ? 3 : 4))
        return FLA_ERR_WORKSPACE;
    float *w = static_cast<float *>(workspace);
    void *state_v = static_cast<char *>(workspace) + 2 * sb;
    const void *state_f = state_in;
    if (!state_f) {
        void *mine = static_cast<char *>(workspace) + 3 * sb;
        if (int rc = chunk_states(k, v, B, H, N, dqk, dv, 0, dtype, w, mine, stream)) return rc;
        state_f = mine;
    }
    if (int rc = chunk_states(q, go, B, H, N, dqk, dv, 1, dtype, w, state_v, stream)) return rc;
    // One launch for the three products: a workgroup evaluates dQ, dV and dK of its chunk in turn,
    // so q, k, v and dO come from memory once.  dQ reads the forward state [D_v][D_qk] as its own
    // [D_c = D_v][D_o = D_qk] transposed state; dK reads the state of dV transposed.
    fla::TriBatch b;
    b.p[0] = pq, b.p[0].state = state_f, b.p[0].state_transposed = 1;
    b.p[1] = pv, b.p[1].state = state_v, b.p[1].state_transposed = 0;
    b.p[2] = pk, b.p[2].state = state_v, b.p[2].state_transposed = 1;
    return lookup_chunked_batch(dtype, dqk)(b, 3, static_cast<hipStream_t>(stream)) == hipSuccess ? FLA_OK
                                                                                                   : FLA_ERR_LAUNCH;
}

// ---- widths that are no multiples of 8: the plain chunk-wise operator on copies with aligned rows (fla_pack.h).
// The copies' columns beyond the true width are zeros, so sums and results are the same.  The walks above 64 columns store results to
// the caller's rows (AnyRows); other kernels to aligned ones, which a copy takes there.  Forward leaves its copies of q, k, v in the state
// buffer, behind the state, and backward takes them from there.
struct PackPlan {
    bool ok;
    int64_t wq, wv;                     // rounded widths
    int64_t q_bytes, v_bytes;           // one copy of width wq / wv (0: that side's rows are taken as they are)
    int64_t inner_state, inner_work;    // of the rounded problem
};

PackPlan pack_plan(int64_t B, int64_t H, int64_t N, int64_t dqk, int64_t dv) {
    PackPlan p{};
    if ((dqk % 8 == 0 && dv % 8 == 0) || dqk < 1 || dv < 1 || B <= 0 || H <= 0 || N <= 0) return p;
    if (B * H > 0x7fffffffLL / N) return p;  // (the copy kernel counts rows in 32 bits)
    p.wq = (dqk + 7) / 8 * 8, p.wv = (dv + 7) / 8 * 8;
    p.ok = true;
    auto up = [](int64_t bytes) { return (bytes + 255) / 256 * 256; };
    p.q_bytes = dqk % 8 ? up(B * H * N * p.wq * 2) : 0, p.v_bytes = dv % 8 ? up(B * H * N * p.wv * 2) : 0;
    p.inner_state = up(shared_state_bytes(B, H, N, p.wq, p.wv));
    p.inner_work = up(chunked_op_workspace_bytes(B, H, N, p.wq, p.wv));
    return p;
}

int64_t packed_state_bytes(const PackPlan &p) { return p.inner_state + 2 * p.q_bytes + p.v_bytes; }
// (backward without forward's copies is the larger: q, k, dQ, dK on one side, v, dO, dV on the other)
int64_t packed_work_bytes(const PackPlan &p) { return p.inner_work + 4 * p.q_bytes + 3 * p.v_bytes; }
// (forward: the copies of q, k, v, unless a state buffer takes them, and of O)
int64_t packed_fwd_work_bytes(const PackPlan &p, bool with_state) {
    return p.inner_work + (with_state ? 0 : 2 * p.q_bytes + p.v_bytes) + p.v_bytes;
}

// Row-packed stand-ins of a call's operands: views of copies carved from a buffer, and the launch that fills
// them (or, for results, copies them back).
struct Packed {
    fla::PackParams pp{};
    int count = 0;
    int64_t B, H, N;
    Packed(int64_t b, int64_t h, int64_t n) : B(b), H(h), N(n) {
        pp.H = (int32_t)h, pp.N = (int32_t)n, pp.rows = (int32_t)(b * h * n);
    }
    void in(const View &from, const View &to, int64_t width, int64_t wp) { add(from, to, width, wp); }
    void out(const View &from, const View &to, int64_t width) { add(from, to, width, width); }
    void add(const View &from, const View &to, int64_t width, int64_t wp) {
        fla::PackItem &t = pp.item[count++];
        t.src = from.ptr, t.dst = const_cast<void *>(to.ptr);
        t.ss_b = from.strides[0], t.ss_h = from.strides[1], t.ss_n = from.strides[2];
        t.ds_b = to.strides[0], t.ds_h = to.strides[1], t.ds_n = to.strides[2];
        t.width = (int32_t)width, t.wp = (int32_t)wp;
    }
    int launch(void *stream) {
        if (!count) return FLA_OK;
        return fla::launch_pack_rows(pp, count, static_cast<hipStream_t>(stream)) == hipSuccess ? FLA_OK : FLA_ERR_LAUNCH;
    }
};

int packed_forward(const PackPlan &p, const View &q, const View &k, const View &v, const View &o, int64_t B, int64_t H,
                   int64_t N, int64_t dqk, int64_t dv, int dtype, void *state_out, int32_t *state_valid, void *workspace,
                   int64_t workspace_bytes, void *stream) {
    if (state_valid) *state_valid = 0;
    const View all[] = {q, k, v, o};
    for (const View &t : all)
        if (int rc = check_view(t)) return rc;
    if (int rc = check_alias_fwd(q, k, v, o, B, H, N, dqk, dv)) return rc;
    const int64_t need = packed_fwd_work_bytes(p, state_out != nullptr);
    if (need > 0 && (!workspace || reinterpret_cast<uintptr_t>(workspace) % 16 != 0 || workspace_bytes < need)) return FLA_ERR_WORKSPACE;
    if (state_out && reinterpret_cast<uintptr_t>(state_out) % 16 != 0) return FLA_ERR_WORKSPACE;
    const int64_t qs[4] = {H * N * p.wq, N * p.wq, p.wq, 1}, vs[4] = {H * N * p.wv, N * p.wv, p.wv, 1};
    char *copies = state_out ? static_cast<char *>(state_out) + p.inner_state : static_cast<char *>(workspace) + p.inner_work;
    char *results = static_cast<char *>(workspace) + need - p.v_bytes;
    const View qp = p.q_bytes ? View{copies, qs} : q, kp = p.q_bytes ? View{copies + p.q_bytes, qs} : k;
    const View vp = p.v_bytes ? View{copies + 2 * p.q_bytes, vs} : v, op = p.v_bytes ? View{results, vs} : o;
    Packed in(B, H, N), out(B, H, N);
    if (p.q_bytes) in.in(q, qp, dqk, p.wq), in.in(k, kp, dqk, p.wq);
    if (p.v_bytes) in.in(v, vp, dv, p.wv), out.out(op, o, dv);
    if (int rc = in.launch(stream)) return rc;
    AnyRows any{&o, nullptr, nullptr, nullptr, dqk, dv, false};
    if (int rc = chunked_forward(qp, kp, vp, op, B, H, N, p.wq, p.wv, dtype, state_out, state_valid, workspace, p.inner_work,
                                 stream, 0, nullptr, nullptr, nullptr, p.v_bytes ? &any : nullptr))
        return rc;
    return any.done ? FLA_OK : out.launch(stream);
}

int packed_backward(const PackPlan &p, const View &go, const View &q, const View &k, const View &v, const View &dq,
                    const View &dk, const View &dvv, int64_t B, int64_t H, int64_t N, int64_t dqk, int64_t dv, int dtype,
                    const void *state_in, void *workspace, int64_t workspace_bytes, void *stream, bool causal) {
    const View all[] = {go, q, k, v, dq, dk, dvv};
    for (const View &t : all)
        if (int rc = check_view(t)) return rc;
    if (int rc = check_alias_bwd(go, q, k, v, nullptr, dq, dk, dvv, B, H, N, dqk, dv)) return rc;
    if (!workspace || reinterpret_cast<uintptr_t>(workspace) % 16 != 0 || workspace_bytes < packed_work_bytes(p))
        return FLA_ERR_WORKSPACE;
    if (state_in && reinterpret_cast<uintptr_t>(state_in) % 16 != 0) return FLA_ERR_WORKSPACE;
    const int64_t qs[4] = {H * N * p.wq, N * p.wq, p.wq, 1}, vs[4] = {H * N * p.wv, N * p.wv, p.wv, 1};
    char *work = static_cast<char *>(workspace) + p.inner_work;
    char *copies = state_in ? const_cast<char *>(static_cast<const char *>(state_in)) + p.inner_state : work;
    char *more = work + 2 * p.q_bytes + p.v_bytes;  // (dQ, dK, dO, dV)
    const View qp = p.q_bytes ? View{copies, qs} : q, kp = p.q_bytes ? View{copies + p.q_bytes, qs} : k;
    const View vp = p.v_bytes ? View{copies + 2 * p.q_bytes, vs} : v;
    const View dqp = p.q_bytes ? View{more, qs} : dq, dkp = p.q_bytes ? View{more + p.q_bytes, qs} : dk;
    const View gop = p.v_bytes ? View{more + 2 * p.q_bytes, vs} : go;
    const View dvp = p.v_bytes ? View{more + 2 * p.q_bytes + p.v_bytes, vs} : dvv;
    Packed in(B, H, N), out(B, H, N);
    if (p.q_bytes) {
        if (!state_in) in.in(q, qp, dqk, p.wq), in.in(k, kp, dqk, p.wq);
        out.out(dqp, dq, dqk), out.out(dkp, dk, dqk);
    }
    if (p.v_bytes) {
        if (!state_in) in.in(v, vp, dv, p.wv);
        in.in(go, gop, dv, p.wv), out.out(dvp, dvv, dv);
    }
    if (int rc = in.launch(stream)) return rc;
    AnyRows any{nullptr, &dq, &dk, &dvv, dqk, dv, false};
    if (int rc = chunked_backward(gop, qp, kp, vp, dqp, dkp, dvp, B, H, N, p.wq, p.wv, dtype, state_in, workspace, p.inner_work,
                                  stream, 0, nullptr, causal, false, &any))
        return rc;
    return any.done ? FLA_OK : out.launch(stream);
}

// takes FLA_GRADS_F32 off a dtype
bool take_wide_flag(int &dtype) {
    const bool wide = (dtype & FLA_GRADS_F32) != 0;
    dtype &= ~FLA_GRADS_F32;
    return wide;
}

int plain_chunked_backward(const View &go, const View &q, const View &k, const View &v, const View &dq, const View &dk,
                           const View &dvv, int64_t B, int64_t H, int64_t N, int64_t dqk, int64_t dv, int dtype,
                           const void *state_in, void *workspace, int64_t workspace_bytes, void *stream, bool causal) {
    const bool wide_out = take_wide_flag(dtype);
    if (int rc = check_common(B, H, N, dtype)) return rc;
    if (dqk < 1 || dqk > 256) return FLA_ERR_HEAD_DIM;
    if (dv < 1 || dv > 256) return FLA_ERR_V_HEAD_DIM;
    if (wide_out && (dv > 128 || dqk % 8 || dv % 8)) return FLA_ERR_UNSUPPORTED;  // (wide_grads_sizes: before any copy)
    // (causal, D_v above 128 without D_qk above 128 or without forward's states: product by product with the states of 256-row chunks in
    // memory, each sum rounded once, where the copies would run as column halves of v)
    if (const PackPlan p = pack_plan(B, H, N, dqk, dv); p.ok && !(causal && dv > 128 && !(state_in && quad_plan(B, H, N, p.wq, p.wv).ok)))
        return packed_backward(p, go, q, k, v, dq, dk, dvv, B, H, N, dqk, dv, dtype, state_in, workspace, workspace_bytes,
                               stream, causal);
    return chunked_backward(go, q, k, v, dq, dk, dvv, B, H, N, dqk, dv, dtype, state_in, workspace, workspace_bytes, stream, 0,
                            nullptr, causal, wide_out);
}

// O = tril(phi(xq) phi(xk)^T) v with mapped = {phi(xq), phi(xk)} as further outputs.  Chunk-wise
// (chunked != 0): the kernels map on load where they can (the state kernel xk, the main kernel its
// rows of xq); any other shape or layout, and the quadratic kernels, get one element-wise pass
// per operand and then the plain operator on phi(xq), phi(xk).
int feature_forward(const View &vxq, const View &vxk, const View &vv, const View &vo, const View (&mapped)[2], int64_t B,
                    int64_t H, int64_t N, int64_t dqk, int64_t dv, int fmap, int dtype, int chunked, void *state_out,
                    int32_t *state_valid, void *workspace, int64_t workspace_bytes, void *stream,
                    WalkNorm *nx = nullptr) {
    const View all[] = {vxq, vxk, vv, vo, mapped[0], mapped[1]};
    for (const View &t : all)
        if (int rc = check_view(t)) return rc;
    {
        const Span ins[] = {span_of(vxq, B, H, N, dqk), span_of(vxk, B, H, N, dqk), span_of(vv, B, H, N, dv)};
        const Span outs[] = {span_of(vo, B, H, N, dv), span_of(mapped[0], B, H, N, dqk), span_of(mapped[1], B, H, N, dqk)};
        if (int rc = check_alias(ins, 3, outs, 3)) return rc;
    }
    if (chunked) {
        bool done = false;
        if (int rc = chunked_forward(vxq, vxk, vv, vo, B, H, N, dqk, dv, dtype, state_out, state_valid, workspace,
                                     workspace_bytes, stream, fmap, mapped, &done, nx))
            return rc;
        if (done) return FLA_OK;
    }
    if (int rc = launch_feature_pass(1, fmap, vxq, mapped[0], B, H, N, dqk, dtype, stream)) return rc;
    if (int rc = launch_feature_pass(1, fmap, vxk, mapped[1], B, H, N, dqk, dtype, stream)) return rc;
    if (!chunked) return run_tri(mapped[0], mapped[1], vv, vo, B, H, N, dqk, dv, 0, dtype, stream);
    return chunked_forward(mapped[0], mapped[1], vv, vo, B, H, N, dqk, dv, dtype, state_out, state_valid, workspace,
                           workspace_bytes, stream, 0, nullptr, nullptr, nx);
}

int forward(const View &q, const View &k, const View &v, const View &o, int64_t B, int64_t H, int64_t N,
            int64_t dqk, int64_t dv, int dtype, void *stream) {
    const View all[] = {q, k, v, o};
    for (const View &t : all)
        if (int rc = check_view(t)) return rc;
    if (int rc = check_alias_fwd(q, k, v, o, B, H, N, dqk, dv)) return rc;
    return run_tri(q, k, v, o, B, H, N, dqk, dv, 0, dtype, stream);
}

// The three gradient products for validated views.
int backward_products(const View &go, const View &q, const View &k, const View &v, const View &dq, const View &dk,
                      const View &dv, int64_t B, int64_t H, int64_t N, int64_t dqk, int64_t dvw, int dtype,
                      void *stream) {
    // dQ = lower(dO V^T) K ; dV = upper(K Q^T) dO ; dK = upper(V dO^T) Q
    if (B == 0 || H == 0 || N == 0) return FLA_OK;
    // Equal padded widths up to 128: all three products run the same kernel, so they go out as
    // one launch (workgroups of the next product fill the previous one's tail).
    if (pad_index(dqk) == pad_index(dvw) && padded(dqk) <= 128) {
        fla::TriBatch b;
        b.p[0] = make_params(go, v, k, dq, B, H, N, dvw, dqk, 0);
        b.p[1] = make_params(k, q, go, dv, B, H, N, dqk, dvw, 1);
        b.p[2] = make_params(v, go, q, dk, B, H, N, dvw, dqk, 1);
        if (fla::fast_path_ok(b.p[0]) && fla::fast_path_ok(b.p[1]) && fla::fast_path_ok(b.p[2])) {
            const hipError_t e = lookup_batch(dtype, dqk)(b, 3, static_cast<hipStream_t>(stream));
            if (e == hipSuccess) return FLA_OK;
            if (e != hipErrorNotSupported) return FLA_ERR_LAUNCH;
        }
    }
    if (int rc = run_tri(go, v, k, dq, B, H, N, dvw, dqk, 0, dtype, stream)) return rc;
    if (int rc = run_tri(k, q, go, dv, B, H, N, dqk, dvw, 1, dtype, stream)) return rc;
    return run_tri(v, go, q, dk, B, H, N, dvw, dqk, 1, dtype, stream);
}

// The same gradients with dV and dK from one stream of (Q, dO) tiles (fla_tri_pair.h) and dQ as a
// product of its own: equal padded head dims up to 128, operands on the fast path.
int backward_fused_dkdv(const View &go, const View &q, const View &k, const View &v, const View &dq, const View &dk,
                        const View &dv, int64_t B, int64_t H, int64_t N, int64_t dqk, int64_t dvw, int dtype,
                        void *stream) {
    const View all[] = {go, q, k, v, dq, dk, dv};
    for (const View &t : all)
        if (int rc = check_view(t)) return rc;
    if (int rc = check_alias_bwd(go, q, k, v, nullptr, dq, dk, dv, B, H, N, dqk, dvw)) return rc;
    if (pad_index(dqk) != pad_index(dvw) || padded(dqk) > 128) return FLA_ERR_UNSUPPORTED;
    if (B == 0 || H == 0 || N == 0) return FLA_OK;
    const TriParams pq = make_params(go, v, k, dq, B, H, N, dvw, dqk, 0);
    const TriParams pv = make_params(k, q, go, dv, B, H, N, dqk, dvw, 1);
    const TriParams pk = make_params(v, go, q, dk, B, H, N, dvw, dqk, 1);
    if (!fla::fast_path_ok(pq) || !fla::fast_path_ok(pv) || !fla::fast_path_ok(pk)) return FLA_ERR_UNSUPPORTED;
    typedef hipError_t (*pair_fn)(const TriParams &, const TriParams &, hipStream_t);
    static const pair_fn table[3][2] = {{fla::FLA_PAIR_NAME(0, 32), fla::FLA_PAIR_NAME(1, 32)},
                                        {fla::FLA_PAIR_NAME(0, 64), fla::FLA_PAIR_NAME(1, 64)},
                                        {fla::FLA_PAIR_NAME(0, 128), fla::FLA_PAIR_NAME(1, 128)}};
    if (table[pad_index(dqk)][dtype](pv, pk, static_cast<hipStream_t>(stream)) != hipSuccess) return FLA_ERR_LAUNCH;
    return run_tri(go, v, k, dq, B, H, N, dvw, dqk, 0, dtype, stream);
}

int backward(const View &go, const View &q, const View &k, const View &v, const View &dq, const View &dk,
             const View &dv, int64_t B, int64_t H, int64_t N, int64_t dqk, int64_t dvw, int dtype, void *stream) {
    const View all[] = {go, q, k, v, dq, dk, dv};
    for (const View &t : all)
        if (int rc = check_view(t)) return rc;
    if (int rc = check_alias_bwd(go, q, k, v, nullptr, dq, dk, dv, B, H, N, dqk, dvw)) return rc;
    return backward_products(go, q, k, v, dq, dk, dv, B, H, N, dqk, dvw, dtype, stream);
}

// ---- the quadratic evaluation of widths that are no multiples of 8, on copies with aligned rows as above: the fast kernels in place of the
// bounds-checked one.  The copies' columns beyond the true width are zeros: scores are the same, a result's columns come from its own.
// Forward, backward: 100 / 100, B H 16, N 1024 117, 351 -> 36, 42 us, N 2048 216, 658 -> 54, 81; 153 / 64, B H 16, N 1024 129, 336 -> 36, 104;
// 250 / 250, B H 128, N 512 439, 1232 -> 100, 242.
bool on_copies(const PackPlan &p, int64_t dqk, int64_t dv) { return p.ok && dqk <= 256 && dv <= 256; }
// (of q, k, v and O; of dO, dQ, dK and dV as well)
int64_t copies_bytes(const PackPlan &p, bool backward) { return backward ? 4 * p.q_bytes + 3 * p.v_bytes : 2 * p.q_bytes + 2 * p.v_bytes; }

int check_copies(const PackPlan &p, int64_t B, int64_t H, int64_t N, int64_t dqk, int64_t dv, int dtype, const void *workspace,
                 int64_t bytes, bool backward) {
    if (int rc = check_common(B, H, N, dtype)) return rc;
    if (dqk < 1 || dqk > 256) return FLA_ERR_HEAD_DIM;
    if (dv < 1 || dv > 256) return FLA_ERR_V_HEAD_DIM;
    if (!on_copies(p, dqk, dv)) return FLA_ERR_UNSUPPORTED;
    if (!workspace || reinterpret_cast<uintptr_t>(workspace) % 16 != 0 || bytes < copies_bytes(p, backward)) return FLA_ERR_WORKSPACE;
    return FLA_OK;
}

int copies_forward(const View &q, const View &k, const View &v, const View &o, int64_t B, int64_t H, int64_t N, int64_t dqk, int64_t dv,
                   int dtype, void *workspace, int64_t workspace_bytes, void *stream) {
    const PackPlan p = pack_plan(B, H, N, dqk, dv);
    if (int rc = check_copies(p, B, H, N, dqk, dv, dtype, workspace, workspace_bytes, false)) return rc;
    const View all[] = {q, k, v, o};
    for (const View &t : all)
        if (int rc = check_view(t)) return rc;
    if (int rc = check_alias_fwd(q, k, v, o, B, H, N, dqk, dv)) return rc;
    const int64_t qs[4] = {H * N * p.wq, N * p.wq, p.wq, 1}, vs[4] = {H * N * p.wv, N * p.wv, p.wv, 1};
    char *at = static_cast<char *>(workspace);
    const View qp = p.q_bytes ? View{at, qs} : q, kp = p.q_bytes ? View{at + p.q_bytes, qs} : k;
    const View vp = p.v_bytes ? View{at + 2 * p.q_bytes, vs} : v, op = p.v_bytes ? View{at + 2 * p.q_bytes + p.v_bytes, vs} : o;
    Packed in(B, H, N), out(B, H, N);
    if (p.q_bytes) in.in(q, qp, dqk, p.wq), in.in(k, kp, dqk, p.wq);
    if (p.v_bytes) in.in(v, vp, dv, p.wv), out.out(op, o, dv);
    if (int rc = in.launch(stream)) return rc;
    if (int rc = forward(qp, kp, vp, op, B, H, N, p.wq, p.wv, dtype, stream)) return rc;
    return out.launch(stream);
}

int copies_backward(const View &go, const View &q, const View &k, const View &v, const View &dq, const View &dk, const View &dvv, int64_t B,
                    int64_t H, int64_t N, int64_t dqk, int64_t dv, int dtype, void *workspace, int64_t workspace_bytes, void *stream) {
    const PackPlan p = pack_plan(B, H, N, dqk, dv);
    if (int rc = check_copies(p, B, H, N, dqk, dv, dtype, workspace, workspace_bytes, true)) return rc;
    const View all[] = {go, q, k, v, dq, dk, dvv};
    for (const View &t : all)
        if (int rc = check_view(t)) return rc;
    if (int rc = check_alias_bwd(go, q, k, v, nullptr, dq, dk, dvv, B, H, N, dqk, dv)) return rc;
    const int64_t qs[4] = {H * N * p.wq, N * p.wq, p.wq, 1}, vs[4] = {H * N * p.wv, N * p.wv, p.wv, 1};
    char *aq = static_cast<char *>(workspace), *av = aq + 4 * p.q_bytes;
    const View qp = p.q_bytes ? View{aq, qs} : q, kp = p.q_bytes ? View{aq + p.q_bytes, qs} : k;
    const View dqp = p.q_bytes ? View{aq + 2 * p.q_bytes, qs} : dq, dkp = p.q_bytes ? View{aq + 3 * p.q_bytes, qs} : dk;
    const View vp = p.v_bytes ? View{av, vs} : v, gop = p.v_bytes ? View{av + p.v_bytes, vs} : go;
    const View dvp = p.v_bytes ? View{av + 2 * p.v_bytes, vs} : dvv;
    Packed in(B, H, N), out(B, H, N);
    if (p.q_bytes) in.in(q, qp, dqk, p.wq), in.in(k, kp, dqk, p.wq), out.out(dqp, dq, dqk), out.out(dkp, dk, dqk);
    if (p.v_bytes) in.in(v, vp, dv, p.wv), in.in(go, gop, dv, p.wv), out.out(dvp, dvv, dv);
    if (int rc = in.launch(stream)) return rc;
    if (int rc = backward(gop, qp, kp, vp, dqp, dkp, dvp, B, H, N, p.wq, p.wv, dtype, stream)) return rc;
    return out.launch(stream);
}

// ---- normalised linear attention: out = tril(Q K^T) V / (q . cumsum(k) + eps)

struct NormLayout {
    int lpr;
    int64_t chunks, sums_bytes, do_bytes, dn_bytes;
    int64_t vec_bytes;    // chunk-wise walk kernels: one set of per-chunk running vectors (two are kept)
    int64_t norm_bytes;   // the normaliser's own scratch: dO, dn, two sets of chunk sums, two sets of vectors
    int64_t chunk_bytes;  // behind it: scratch of the chunk-wise product evaluation (0 when quadratic)
};

NormLayout norm_layout(int64_t B, int64_t H, int64_t N, int64_t dqk, int64_t dv, int chunked) {
    NormLayout l;
    l.lpr = fla::norm_lanes_per_row((int)(dqk > dv ? dqk : dv));
    const int64_t rows = fla::norm_chunk_rows(l.lpr);
    l.chunks = (N + rows - 1) / rows;
    l.sums_bytes = B * H * l.chunks * (l.lpr * 8) * 4;
    l.do_bytes = (B * H * N * dv * 2 + 15) / 16 * 16;
    l.dn_bytes = (B * H * N * 4 + 15) / 16 * 16;
    l.sums_bytes = (l.sums_bytes + 15) / 16 * 16;
    l.vec_bytes = chunked ? walk_vec_bytes(B, H, N, dqk, dv) : 0;
    l.norm_bytes = l.do_bytes + l.dn_bytes + 2 * l.sums_bytes + 2 * l.vec_bytes;
    l.chunk_bytes = chunked ? chunked_op_workspace_bytes(B, H, N, dqk, dv) : 0;
    return l;
}

void norm_common(fla::NormParams &p, const View &q, const View &k, int64_t B, int64_t H, int64_t N, int64_t dqk,
                 int64_t dv, const NormLayout &l) {
    p = fla::NormParams{};
    p.q = q.ptr, p.k = k.ptr;
    p.qs_b = q.strides[0], p.qs_h = q.strides[1], p.qs_n = q.strides[2];
    p.ks_b = k.strides[0], p.ks_h = k.strides[1], p.ks_n = k.strides[2];
    p.H = (int32_t)H, p.N = (int32_t)N, p.BH = (int32_t)(B * H), p.dqk = (int32_t)dqk, p.dv = (int32_t)dv;
    p.n_chunks = (int32_t)l.chunks;
    p.vec_q = vec_ok(q, dqk), p.vec_k = vec_ok(k, dqk);
}

hipError_t norm_launch(int which, int dtype, int lpr, const fla::NormParams &p, void *stream) {
    hipStream_t s = static_cast<hipStream_t>(stream);
    // the operands this pass touches all allow 16-byte accesses?
    const bool vec = which == 0   ? (p.vec_q && p.vec_k && p.vec_a && p.vec_out)
                     : which == 1 ? (p.vec_a && p.vec_b && p.vec_out && (!p.zc || p.vec_q))
                                  : (p.vec_q && p.vec_k && p.vec_dq && p.vec_dk);
    return dtype == FLA_DTYPE_BF16 ? fla::launch_norm<__bf16>(which, lpr, vec, p, s)
                                   : fla::launch_norm<_Float16>(which, lpr, vec, p, s);
}

int check_norm_args(int64_t B, int64_t H, int64_t N, int64_t dqk, int64_t dv, int dtype) {
    if (int rc = check_common(B, H, N, dtype)) return rc;
    if (dqk < 1 || dqk > 256) return FLA_ERR_HEAD_DIM;
    if (dv < 1 || dv > 256) return FLA_ERR_V_HEAD_DIM;
    // the grid's second dimension is the (batch, head) index
    if (B * H > 65535) return FLA_ERR_SHAPE;
    return FLA_OK;
}

// Forward with the normaliser inside the product kernel: the row sums of the masked scores are
// the normaliser (q_i . sum_{j<=i} k_j = sum_j q_i . k_j), so the fast kernel divides before it
// stores and no extra pass runs.  Returns 1 when this shape / layout has no such kernel (the
// caller then normalises with the separate passes), 0 on success, a negative code on failure.
int fused_normalised_forward(const View &q, const View &k, const View &v, const View &o, float *denom, int64_t B,
                             int64_t H, int64_t N, int64_t dqk, int64_t dv, float eps, int dtype, void *stream) {
    const bool split = dv > 128 && (dqk <= 64 || dqk > 128);
    const int64_t w0 = split ? 128 : dv;
    TriParams p0 = make_params(q, k, v, o, B, H, N, dqk, w0, 0);
    if (chunk_rows(dqk, w0) == 0 || !fla::fast_path_ok(p0)) return 1;
    p0.denom = denom, p0.eps = eps;
    if (!split) return lookup(dtype, dqk, w0)(p0, static_cast<hipStream_t>(stream)) == hipSuccess ? FLA_OK : FLA_ERR_LAUNCH;
    const View v_hi{static_cast<const char *>(v.ptr) + 128 * 2, v.strides};
    const View o_hi{static_cast<const char *>(o.ptr) + 128 * 2, o.strides};
    TriParams p1 = make_params(q, k, v_hi, o_hi, B, H, N, dqk, dv - 128, 0);
    if (chunk_rows(dqk, dv - 128) == 0 || !fla::fast_path_ok(p1)) return 1;
    p1.denom = denom, p1.eps = eps;  // both halves see the same scores and write the same n
    if (lookup(dtype, dqk, w0)(p0, static_cast<hipStream_t>(stream)) != hipSuccess) return FLA_ERR_LAUNCH;
    return lookup(dtype, dqk, dv - 128)(p1, static_cast<hipStream_t>(stream)) == hipSuccess ? FLA_OK : FLA_ERR_LAUNCH;
}

// fmap != 0: q0, k0 hold the arguments xq, xk of the feature map and mapped = {phi(xq), phi(xk)} are
// further outputs; the normaliser is that of phi(xq), phi(xk).
int normalised_forward(const View &q0, const View &k0, const View &v, const View &o, float *denom, int64_t B, int64_t H,
                       int64_t N, int64_t dqk, int64_t dv, float eps, int dtype, int chunked, void *workspace,
                       int64_t workspace_bytes, void *stream, int fmap = 0, const View *mapped = nullptr,
                       void *state_out = nullptr, int32_t *state_valid = nullptr) {
    if (state_valid) *state_valid = 0;
    const View all[] = {q0, k0, v, o};
    for (const View &t : all)
        if (int rc = check_view(t)) return rc;
    if (!denom) return FLA_ERR_NULL_POINTER;
    if (int rc = check_alias_fwd(q0, k0, v, o, B, H, N, dqk, dv)) return rc;
    if (B == 0 || H == 0 || N == 0) return FLA_OK;
    const NormLayout l = norm_layout(B, H, N, dqk, dv, chunked);
    if ((l.chunks > 1 || l.chunk_bytes > 0) &&
        (!workspace || reinterpret_cast<uintptr_t>(workspace) % 16 != 0 || workspace_bytes < l.norm_bytes + l.chunk_bytes))
        return FLA_ERR_WORKSPACE;
    if (fmap && !chunked) {
        // quadratic product: phi by element-wise passes, then the operator on phi(xq), phi(xk)
        for (int i = 0; i < 2; ++i)
            if (int rc = check_view(mapped[i])) return rc;
        if (int rc = launch_feature_pass(1, fmap, q0, mapped[0], B, H, N, dqk, dtype, stream)) return rc;
        if (int rc = launch_feature_pass(1, fmap, k0, mapped[1], B, H, N, dqk, dtype, stream)) return rc;
        return normalised_forward(mapped[0], mapped[1], v, o, denom, B, H, N, dqk, dv, eps, dtype, 0, workspace,
                                  workspace_bytes, stream);
    }
    // chunk-wise walk kernels compute n and divide by it themselves
    WalkNorm nx{denom, eps, nullptr,
                workspace ? static_cast<char *>(workspace) + l.do_bytes + l.dn_bytes + 2 * l.sums_bytes : nullptr,
                nullptr, nullptr, nullptr, false, false, false};
    const View &q = fmap ? mapped[0] : q0, &k = fmap ? mapped[1] : k0;
    if (!chunked) {
        const int rc = fused_normalised_forward(q, k, v, o, denom, B, H, N, dqk, dv, eps, dtype, stream);
        if (rc <= 0) return rc;
    }
    if (fmap) {
        const View both[2] = {mapped[0], mapped[1]};
        if (int rc = feature_forward(q0, k0, v, o, both, B, H, N, dqk, dv, fmap, dtype, 1, state_out, state_valid,
                                     static_cast<char *>(workspace) + l.norm_bytes, l.chunk_bytes, stream, &nx))
            return rc;
        if (nx.fused) return FLA_OK;
    } else if (chunked) {
        if (int rc = chunked_forward(q, k, v, o, B, H, N, dqk, dv, dtype, state_out, state_valid,
                                     static_cast<char *>(workspace) + l.norm_bytes, l.chunk_bytes, stream, 0, nullptr,
                                     nullptr, &nx))
            return rc;
        if (nx.fused) return FLA_OK;
    } else if (int rc = run_tri(q, k, v, o, B, H, N, dqk, dv, 0, dtype, stream)) {
        return rc;
    }
    fla::NormParams p;
    norm_common(p, q, k, B, H, N, dqk, dv, l);
    p.a = o.ptr, p.out = const_cast<void *>(o.ptr);  // normalised in place
    p.as_b = p.os_b = o.strides[0], p.as_h = p.os_h = o.strides[1], p.as_n = p.os_n = o.strides[2];
    p.vec_a = p.vec_out = vec_ok(o, dv);
    p.denom = denom;
    p.ksum = static_cast<float *>(workspace);
    p.eps = eps;
    return norm_launch(0, dtype, l.lpr, p, stream) == hipSuccess ? FLA_OK : FLA_ERR_LAUNCH;
}

int normalised_backward(const View &go, const View &q, const View &k, const View &v, const View &o,
                        const float *denom, const View &dq, const View &dk, const View &dvv, int64_t B, int64_t H,
                        int64_t N, int64_t dqk, int64_t dv, int dtype, int chunked, void *workspace,
                        int64_t workspace_bytes, void *stream, int fmap = 0, const void *state_in = nullptr, bool wide_out = false) {
    // fmap != 0: q, k hold phi(xq), phi(xk) and dq, dk leave as gradients with respect to xq, xk (the
    // slope is multiplied in by the last pass, after the normaliser's own terms have been added)
    const View all[] = {go, q, k, v, o, dq, dk, dvv};
    for (const View &t : all)
        if (int rc = check_view(t)) return rc;
    if (!denom) return FLA_ERR_NULL_POINTER;
    if (int rc = check_alias_bwd(go, q, k, v, &o, dq, dk, dvv, B, H, N, dqk, dv, wide_out)) return rc;
    if (B == 0 || H == 0 || N == 0) return FLA_OK;
    const NormLayout l = norm_layout(B, H, N, dqk, dv, chunked);
    if (!workspace || reinterpret_cast<uintptr_t>(workspace) % 16 != 0 || workspace_bytes < l.norm_bytes + l.chunk_bytes)
        return FLA_ERR_WORKSPACE;
    char *ws = static_cast<char *>(workspace);
    void *dO = ws;
    float *dn = reinterpret_cast<float *>(ws + l.do_bytes);
    float *ksum = reinterpret_cast<float *>(ws + l.do_bytes + l.dn_bytes);
    float *wsum = reinterpret_cast<float *>(ws + l.do_bytes + l.dn_bytes + l.sums_bytes);
    const int64_t do_strides[4] = {H * N * dv, N * dv, dv, 1};
    const View dOv{dO, do_strides};

    fla::NormParams p;
    norm_common(p, q, k, B, H, N, dqk, dv, l);
    p.denom = const_cast<float *>(denom), p.dn = dn, p.ksum = ksum, p.wsum = wsum;
    // dO = g / n, dn = -(g . out) / n: by the first kernel of the walks where they take the call, else by a pass of its own
    p.a = go.ptr, p.as_b = go.strides[0], p.as_h = go.strides[1], p.as_n = go.strides[2], p.vec_a = vec_ok(go, dv);
    p.b = o.ptr, p.bs_b = o.strides[0], p.bs_h = o.strides[1], p.bs_n = o.strides[2], p.vec_b = vec_ok(o, dv);
    p.out = dO, p.os_b = do_strides[0], p.os_h = do_strides[1], p.os_n = do_strides[2], p.vec_out = vec_ok(dOv, dv);
    // (chunked == 2: the plain products chunk-wise, the normaliser's terms behind them as in the quadratic evaluation)
    const bool apart = chunked == FLA_CHUNKED_PRODUCTS && !fmap;
    const bool walks = chunked && !apart && norm_walks_backward(dOv, q, k, v, dq, dk, dvv, B, H, N, dqk, dv, state_in);
    if (wide_out && !(walks && wide_grads_walk(dOv, q, k, v, dq, dk, dvv, B, H, N, dqk, dv, dtype, state_in, false)))
        return FLA_ERR_UNSUPPORTED;
    // behind the walks: the forward walk's running sums of k, at the entry of each of its chunks, spare the passes' own, and the sums of
    // dn q are formed with dn (device time behind the walks, B H 48, N 17148, D 64: 11 units of 105 MB in six launches -> 10 in four)
    const WalkPlan wp = walk_plan(B, H, N, dqk, dv);
    if (apart && state_in && dtype == FLA_DTYPE_BF16 && norm_walks_backward(dOv, q, k, v, dq, dk, dvv, B, H, N, dqk, dv, state_in)) {
        p.zc = reinterpret_cast<const float *>(static_cast<const char *>(state_in) + state_core_bytes(B, H, N, dqk, dv));
        p.walk_chunks = (int32_t)wp.n_chunks, p.walk_step = fla::norm_chunk_rows(l.lpr) / wp.rows;
    }
    if (!walks && norm_launch(1, dtype, l.lpr, p, stream) != hipSuccess) return FLA_ERR_LAUNCH;
    // gradients of the unnormalised product
    WalkNorm nx{nullptr, 0.f, dn, ws + l.do_bytes + l.dn_bytes + 2 * l.sums_bytes, &go, &o, denom, p.vec_a && p.vec_b, false, false};
    if (apart) {
        if (int rc = chunked_backward(dOv, q, k, v, dq, dk, dvv, B, H, N, dqk, dv, dtype, state_in, ws + l.norm_bytes, l.chunk_bytes,
                                      stream, 0, nullptr, true, false, nullptr, false))
            return rc;
    } else if (chunked) {
        // the walk kernels add the normaliser's terms (and apply the slope of a feature map) themselves
        if (int rc = chunked_backward(dOv, q, k, v, dq, dk, dvv, B, H, N, dqk, dv, dtype, state_in, ws + l.norm_bytes,
                                      l.chunk_bytes, stream, fmap, &nx, false, wide_out))
            return rc;
        if (nx.fused && !nx.dk_pending) return FLA_OK;
    } else if (int rc = backward_products(dOv, q, k, v, dq, dk, dvv, B, H, N, dqk, dv, dtype, stream)) {
        return rc;
    }
    // the normaliser's own terms
    p.dq = const_cast<void *>(dq.ptr), p.dqs_b = dq.strides[0], p.dqs_h = dq.strides[1], p.dqs_n = dq.strides[2];
    p.dk = const_cast<void *>(dk.ptr), p.dks_b = dk.strides[0], p.dks_h = dk.strides[1], p.dks_n = dk.strides[2];
    p.vec_dq = vec_ok(dq, dqk), p.vec_dk = vec_ok(dk, dqk);
    p.fmap = fmap;
    p.only_dk = nx.fused && nx.dk_pending;  // (dq is complete, slope included)
    return norm_launch(2, dtype, l.lpr, p, stream) == hipSuccess ? FLA_OK : FLA_ERR_LAUNCH;
}

// ---- polynomial score map: out = lower(f(Xq Xk^T)) V, f(u) = c0 + c1 u + c2 u^2

// [a | x] side by side, 8 elements per thread: columns [0, split) hold a (zero beyond its width),
// columns [split, split + rp) hold x (zero beyond its width); out is contiguous (B, H, N, split + rp).
// bias_mode 1 / 2 puts one more value right after a, in column wa: bias[row] / the constant 1.
template <typename T>
__global__ __launch_bounds__(256) void pack_pair_kernel(const T *a, int64_t as_b, int64_t as_h, int64_t as_n, int wa,
                                                        const T *x, int64_t xs_b, int64_t xs_h, int64_t xs_n, int wx,
                                                        T *out, int H, int64_t N, int split, int rp, int64_t total,
                                                        int bias_mode, const float *bias) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= total) return;
    const int cpr = (split + rp) / 8;  // 8-element chunks per row
    const int64_t row = t / cpr;
    const int c8 = (int)(t - row * cpr) * 8;
    const int64_t bh = row / N, n = row - bh * N;
    const int64_t b = bh / H, h = bh - b * H;
    fla::u32x4 w = {0u, 0u, 0u, 0u};
    if (c8 < split) {
        if (c8 < wa) {
            w = *reinterpret_cast<const fla::u32x4 *>(a + b * as_b + h * as_h + n * as_n + c8);
        } else if (c8 == wa && bias_mode) {
            const T one = static_cast<T>(bias_mode == 1 ? bias[row] : 1.0f);
            w[0] = (uint32_t)__builtin_bit_cast(unsigned short, one);
        }
    } else if (c8 - split < wx) {
        w = *reinterpret_cast<const fla::u32x4 *>(x + b * xs_b + h * xs_h + n * xs_n + (c8 - split));
    }
    *reinterpret_cast<fla::u32x4 *>(out + row * (split + rp) + c8) = w;
}

template <typename T>
hipError_t launch_pack(const View &a, int wa, const View &x, int wx, void *out, int64_t B, int64_t H, int64_t N, int split,
                 int rp, int bias_mode, const float *bias, hipStream_t s) {
    const int64_t total = B * H * N * ((split + rp) / 8);
    return fla::launch_kernel<pack_pair_kernel<T>>(dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s,
                              static_cast<const T *>(a.ptr), a.strides[0], a.strides[1], a.strides[2], wa,
                              static_cast<const T *>(x.ptr), x.strides[0], x.strides[1], x.strides[2], wx,
                              static_cast<T *>(out), (int)H, N, split, rp, total, bias_mode, bias);
}

struct PolyLayout {
    int64_t split, rp, width, packed_bytes;
    int mode;  // TriParams::poly_on of the dual-score products: 2 (half layout) or 3 (tail layout)
    // normalised backward: dO = g / n and dn, then the packed operands
    int64_t do_bytes, dn_bytes;
};

// split: where the second operand starts; rp: r rounded up to whole 16-byte chunks.  Without the
// bias column the first operand is padded to half of the contraction the dual-score kernel is built
// for (the kernel skips the empty chunks); with it (normalised backward) D_v + 1 columns are needed,
// and when those do not fit the half the second operand goes to the last 32 columns instead.
PolyLayout poly_layout(int64_t B, int64_t H, int64_t N, int64_t r, int64_t dv, int with_bias) {
    PolyLayout l;
    const int64_t need = dv + (with_bias ? 8 : 0);  // the bias takes a 16-byte chunk of its own
    const int64_t half = need <= 32 ? 32 : need <= 64 ? 64 : need <= 128 ? 128 : 0;
    const int64_t dc_tail = need + 32 <= 64 ? 64 : need + 32 <= 128 ? 128 : 256;
    if (half != 0 && 2 * half <= dc_tail) {
        l.split = half, l.mode = 2;
    } else {
        l.split = dc_tail - 32, l.mode = 3;
    }
    l.rp = l.mode == 3 ? 32 : (r + 7) / 8 * 8;
    l.width = l.split + l.rp;
    l.packed_bytes = (B * H * N * l.width * 2 + 15) / 16 * 16;
    l.do_bytes = with_bias ? (B * H * N * dv * 2 + 15) / 16 * 16 : 0;
    l.dn_bytes = with_bias ? (B * H * N * 4 + 15) / 16 * 16 : 0;
    return l;
}

int check_poly_args(int64_t B, int64_t H, int64_t N, int64_t r, int64_t dv, int dtype, const float *coef) {
    if (int rc = check_common(B, H, N, dtype)) return rc;
    if (!coef) return FLA_ERR_NULL_POINTER;
    if (r < 1 || r > 32) return FLA_ERR_HEAD_DIM;
    if (dv < 1 || dv > 128) return FLA_ERR_V_HEAD_DIM;
    return FLA_OK;
}

// every product of this operator exists only as a fast-path kernel
bool poly_ok(const TriParams &p, int64_t dc, int64_t dout) { return chunk_rows(dc, dout) != 0 && fla::fast_path_ok(p); }

int launch_poly(TriParams p, int64_t dc, int64_t dout, int dtype, int mode, float c0, float c1, float c2, void *stream) {
    p.poly[0] = c0, p.poly[1] = c1, p.poly[2] = c2, p.poly_on = mode;
    const hipError_t e = lookup(dtype, dc, dout)(p, static_cast<hipStream_t>(stream));
    return e == hipSuccess ? FLA_OK : e == hipErrorNotSupported ? FLA_ERR_UNSUPPORTED : FLA_ERR_LAUNCH;
}

int poly_forward(const View &xq, const View &xk, const View &v, const View &o, float *denom, int64_t B, int64_t H,
                 int64_t N, int64_t r, int64_t dv, const float *coef, float eps, int dtype, void *stream) {
    const View all[] = {xq, xk, v, o};
    for (const View &t : all)
        if (int rc = check_view(t)) return rc;
    if (int rc = check_alias_fwd(xq, xk, v, o, B, H, N, r, dv)) return rc;
    if (B == 0 || H == 0 || N == 0) return FLA_OK;
    if (denom && B * H > 65535) return FLA_ERR_SHAPE;
    TriParams p = make_params(xq, xk, v, o, B, H, N, r, dv, 0);
    if (!poly_ok(p, r, dv)) return FLA_ERR_UNSUPPORTED;
    p.denom = denom, p.eps = eps;
    return launch_poly(p, r, dv, dtype, 1, coef[0], coef[1], coef[2], stream);
}

int poly_backward(const View &go, const View &xq, const View &xk, const View &v, const View *o, const float *denom,
                  const View &dxq, const View &dxk, const View &dvv, int64_t B, int64_t H, int64_t N, int64_t r,
                  int64_t dv, const float *coef, int dtype, void *workspace, int64_t workspace_bytes, void *stream) {
    const View all[] = {go, xq, xk, v, dxq, dxk, dvv};
    for (const View &t : all)
        if (int rc = check_view(t)) return rc;
    const bool normalised = o != nullptr;
    if (normalised) {
        if (int rc = check_view(*o)) return rc;
        if (!denom) return FLA_ERR_NULL_POINTER;
        if (B * H > 65535) return FLA_ERR_SHAPE;
    }
    if (int rc = check_alias_bwd(go, xq, xk, v, o, dxq, dxk, dvv, B, H, N, r, dv)) return rc;
    if (B == 0 || H == 0 || N == 0) return FLA_OK;
    const PolyLayout l = poly_layout(B, H, N, r, dv, normalised);
    if (!workspace || reinterpret_cast<uintptr_t>(workspace) % 16 != 0 ||
        workspace_bytes < 2 * l.packed_bytes + l.do_bytes + l.dn_bytes)
        return FLA_ERR_WORKSPACE;
    // the packing kernel and the products below use 16-byte accesses throughout
    if (!(vec_ok(go, dv) && vec_ok(v, dv) && vec_ok(xq, r) && vec_ok(xk, r) && vec_ok(dxq, r) && vec_ok(dxk, r) &&
          vec_ok(dvv, dv)))
        return FLA_ERR_UNSUPPORTED;
    hipStream_t s = static_cast<hipStream_t>(stream);
    char *ws = static_cast<char *>(workspace);
    void *p1 = ws, *p2 = ws + l.packed_bytes;  // [dO (| dn) | xq], [V (| 1) | xk]
    void *dO = ws + 2 * l.packed_bytes;
    float *dn = reinterpret_cast<float *>(ws + 2 * l.packed_bytes + l.do_bytes);
    const int64_t do_strides[4] = {H * N * dv, N * dv, dv, 1};
    View g = go;
    if (normalised) {
        // out = O / n: dO = g / n, dn = -(g . out) / n; the dn term enters u1 as a bias column
        const int lpr = fla::norm_lanes_per_row((int)dv);
        fla::NormParams np{};
        np.H = (int32_t)H, np.N = (int32_t)N, np.BH = (int32_t)(B * H), np.dqk = (int32_t)dv, np.dv = (int32_t)dv;
        const int64_t rows = fla::norm_chunk_rows(lpr);
        np.n_chunks = (int32_t)((N + rows - 1) / rows);
        np.denom = const_cast<float *>(denom), np.dn = dn;
        np.a = go.ptr, np.as_b = go.strides[0], np.as_h = go.strides[1], np.as_n = go.strides[2], np.vec_a = vec_ok(go, dv);
        np.b = o->ptr, np.bs_b = o->strides[0], np.bs_h = o->strides[1], np.bs_n = o->strides[2], np.vec_b = vec_ok(*o, dv);
        np.out = dO, np.os_b = do_strides[0], np.os_h = do_strides[1], np.os_n = do_strides[2], np.vec_out = 1;
        if (norm_launch(1, dtype, lpr, np, stream) != hipSuccess) return FLA_ERR_LAUNCH;
        g = View{dO, do_strides};
    }
    const int bias1 = normalised ? 1 : 0, bias2 = normalised ? 2 : 0;
    const auto pack = dtype == FLA_DTYPE_BF16 ? launch_pack<__bf16> : launch_pack<_Float16>;
    if (pack(g, (int)dv, xq, (int)r, p1, B, H, N, (int)l.split, (int)l.rp, bias1, dn, s) != hipSuccess) return FLA_ERR_LAUNCH;
    if (pack(v, (int)dv, xk, (int)r, p2, B, H, N, (int)l.split, (int)l.rp, bias2, nullptr, s) != hipSuccess)
        return FLA_ERR_LAUNCH;
    const int64_t ps[4] = {H * N * l.width, N * l.width, l.width, 1};
    const View P1{p1, ps}, P2{p2, ps};
    // dV = upper(f(Xk Xq^T)) dO
    const TriParams pv = make_params(xk, xq, g, dvv, B, H, N, r, dv, 1);
    // dXq = lower((dO V^T + dn 1^T) f'(Xq Xk^T)) Xk, dXk = upper((V dO^T + 1 dn^T) f'(Xk Xq^T)) Xq; f'(u) = c1 + 2 c2 u
    const TriParams pq = make_params(P1, P2, xk, dxq, B, H, N, l.width, r, 0);
    const TriParams pk = make_params(P2, P1, xq, dxk, B, H, N, l.width, r, 1);
    if (!poly_ok(pv, r, dv) || !poly_ok(pq, l.width, r) || !poly_ok(pk, l.width, r)) return FLA_ERR_UNSUPPORTED;
    if (int rc = launch_poly(pv, r, dv, dtype, 1, coef[0], coef[1], coef[2], stream)) return rc;
    if (int rc = launch_poly(pq, l.width, r, dtype, l.mode, coef[1], 2.0f * coef[2], 0.f, stream)) return rc;
    return launch_poly(pk, l.width, r, dtype, l.mode, coef[1], 2.0f * coef[2], 0.f, stream);
}

// ---- the polynomial score map chunk-wise (fla_poly_walk.h)
struct PolyPlan {
    bool ok;
    int64_t n_chunks, seg_chunks, n_seg, state_bytes, work_bytes;
    int64_t halves, part_bytes;  // halves of v's columns, each planned as a head; room behind the totals for one of dq_part, dk_part
    // more than 16 columns of q and k: three parts with states of their own, and their sums behind the totals (PolyWalkParams::part)
    bool parts;
    int64_t sums_bytes, total_bytes, fwd_bytes, state_at[4];  // (fwd_bytes: work_bytes of forward)
};

PolyPlan poly_plan(int64_t B, int64_t H, int64_t N, int64_t r, int64_t dv) {
    PolyPlan p{};
    if (B <= 0 || H <= 0 || N <= 0 || r < 1 || r > 32 || r % 8 || dv < 1 || dv > 128 || dv % 8) return p;
    p.halves = dv > 64 ? 2 : 1;
    const int64_t heads = B * H * p.halves;
    if (heads > 0x7fffffff) return p;
    p.ok = true;
    p.n_chunks = (N + fla::PolyLds::C - 1) / fla::PolyLds::C;
    // (one workgroup per CU: as many equal segments per (b, h) as run at once, the walk kernels' rule)
    int64_t segs = 256 / heads > 1 ? 256 / heads : 1;
    if (segs > p.n_chunks) segs = p.n_chunks;
    p.seg_chunks = (p.n_chunks + segs - 1) / segs;
    p.n_seg = (p.n_chunks + p.seg_chunks - 1) / p.seg_chunks;
    p.parts = r > 16;
    const int64_t slots = heads * p.n_seg * 4, cross = fla::PolyFeatures::kCross * 65;
    p.part_bytes = p.halves == 2 ? heads * N * (p.parts ? 32 : 16) * 4 : 0;
    // (backward: dV, dq, dk; forward: O and n)
    p.sums_bytes = p.parts ? heads * N * (64 + 32 + 32) * 4 : 0;
    p.total_bytes = p.n_seg > 1 ? slots * (p.parts ? cross : fla::PolyFeatures::kState) : 0;
    p.work_bytes = p.total_bytes + p.sums_bytes + 2 * p.part_bytes;
    p.fwd_bytes = p.total_bytes + (p.parts ? heads * N * (64 + 1) * 4 : 0);
    // (a single segment per (b, h) hands nothing over: a token)
    p.state_bytes = p.n_seg == 1 ? 16 : slots * (p.parts ? 2 * fla::PolyFeatures::kState + cross : fla::PolyFeatures::kStateRoom);
    p.state_at[fla::kPolySecond] = p.parts ? slots * fla::PolyFeatures::kState : 0;
    p.state_at[fla::kPolyCross] = 2 * p.state_at[fla::kPolySecond];
    return p;
}

int check_poly_chunked(const PolyPlan &pl, int dtype, int64_t need, int64_t workspace_bytes, const void *workspace, const void *state) {
    if (!pl.ok || dtype != FLA_DTYPE_BF16) return FLA_ERR_UNSUPPORTED;
    if (need && (!workspace || reinterpret_cast<uintptr_t>(workspace) % 16 != 0 || workspace_bytes < need)) return FLA_ERR_WORKSPACE;
    return reinterpret_cast<uintptr_t>(state) % 16 != 0 ? FLA_ERR_WORKSPACE : FLA_OK;
}

// totals over the segments and -- beyond kSumOnLoadPoly of them -- their scan
int poly_entries(const PolyPlan &pl, fla::PolyWalkParams &w, bool bwd, void *workspace, hipStream_t s) {
    if (pl.n_seg == 1) return FLA_OK;
    w.totals = static_cast<float *>(workspace);
    if (fla::poly_totals(w, bwd, s) != hipSuccess) return FLA_ERR_LAUNCH;
    w.sum_entries = pl.n_seg <= kSumOnLoadPoly;
    if (w.sum_entries) return FLA_OK;
    return fla::poly_scan(w.totals, w.BH, w.n_seg, bwd ? 1 : 0, w.part, s) == hipSuccess ? FLA_OK : FLA_ERR_LAUNCH;
}

// totals and walks, in backward of dq and of dk and dV; of rows of two halves part by part
int poly_run(const PolyPlan &pl, fla::PolyWalkParams &w, bool bwd, const void *state, void *workspace, hipStream_t s) {
    static const int parts[] = {fla::kPolyCross, fla::kPolySecond, fla::kPolyFirst};
    char *const at = static_cast<char *>(workspace) + pl.total_bytes;
    if (pl.parts) {
        w.acc = reinterpret_cast<float *>(at);
        float *const next = w.acc + (int64_t)w.BH * w.N * 64;
        if (bwd)
            w.acc_q = next, w.acc_k = next + (int64_t)w.BH * w.N * 32;
        else
            w.acc_n = next;
    }
    for (int i = 0; i < (pl.parts ? 3 : 1); ++i) {
        w.part = pl.parts ? parts[i] : fla::kPolyWhole;
        if (pl.n_seg > 1 && state)
            w.entries = reinterpret_cast<float *>(static_cast<char *>(const_cast<void *>(state)) + pl.state_at[w.part]);
        // (with two segments half of the workgroups would have the totals' work beside dq)
        if (bwd && !pl.parts && pl.n_seg >= 3 && pl.n_seg <= kSumOnLoadPoly) {
            w.totals = static_cast<float *>(workspace), w.sum_entries = w.u_totals = 1;
        } else if (int rc = poly_entries(pl, w, bwd, workspace, s)) {
            return rc;
        }
        if (fla::poly_walk(w, bwd, s) != hipSuccess) return FLA_ERR_LAUNCH;
    }
    return FLA_OK;
}

void poly_common(fla::PolyWalkParams &w, const PolyPlan &pl, const View &xq, const View &xk, const View &v, int64_t B, int64_t H,
                 int64_t N, int64_t r, int64_t dv, const float *coef) {
    w.q = xq.ptr, w.qs_b = xq.strides[0], w.qs_h = xq.strides[1], w.qs_n = xq.strides[2];
    w.k = xk.ptr, w.ks_b = xk.strides[0], w.ks_h = xk.strides[1], w.ks_n = xk.strides[2];
    w.v = v.ptr, w.vs_b = v.strides[0], w.vs_h = v.strides[1], w.vs_n = v.strides[2];
    w.H = (int32_t)H, w.N = (int32_t)N, w.BH = (int32_t)(B * H * pl.halves), w.r = (int32_t)r, w.wv = (int32_t)dv;
    w.vhalf = pl.halves == 2;
    w.n_chunks = (int32_t)pl.n_chunks, w.seg_chunks = (int32_t)pl.seg_chunks, w.n_seg = (int32_t)pl.n_seg;
    w.c0 = coef[0], w.c1 = coef[1], w.c2 = coef[2];
}

int poly_chunked_forward(const View &xq, const View &xk, const View &v, const View &o, float *denom, int64_t B, int64_t H,
                         int64_t N, int64_t r, int64_t dv, const float *coef, float eps, int dtype, void *state_out,
                         void *workspace, int64_t workspace_bytes, void *stream) {
    const View all[] = {xq, xk, v, o};
    for (const View &t : all)
        if (int rc = check_view(t)) return rc;
    if (int rc = check_alias_fwd(xq, xk, v, o, B, H, N, r, dv)) return rc;
    if (B == 0 || H == 0 || N == 0) return FLA_OK;
    const PolyPlan pl = poly_plan(B, H, N, r, dv);
    if (int rc = check_poly_chunked(pl, dtype, pl.fwd_bytes, workspace_bytes, workspace, state_out)) return rc;
    if (!vec_ok(xq, r) || !vec_ok(xk, r) || !vec_ok(v, dv) || !vec_ok(o, dv)) return FLA_ERR_UNSUPPORTED;
    fla::PolyWalkParams w{};
    poly_common(w, pl, xq, xk, v, B, H, N, r, dv, coef);
    w.out = const_cast<void *>(o.ptr), w.us_b = o.strides[0], w.us_h = o.strides[1], w.us_n = o.strides[2];
    w.eps = eps, w.denom = denom;
    hipStream_t s = static_cast<hipStream_t>(stream);
    return poly_run(pl, w, false, state_out, workspace, s);
}

int poly_chunked_backward(const View &go, const View &xq, const View &xk, const View &v, const View *o, const float *denom,
                          const View &dxq, const View &dxk, const View &dvv, int64_t B, int64_t H, int64_t N, int64_t r,
                          int64_t dv, const float *coef, int dtype, const void *state_in, void *workspace,
                          int64_t workspace_bytes, void *stream, bool wide_out) {
    const View all[] = {go, xq, xk, v, dxq, dxk, dvv};
    for (const View &t : all)
        if (int rc = check_view(t)) return rc;
    if ((o == nullptr) != (denom == nullptr)) return FLA_ERR_NULL_POINTER;
    if (o)
        if (int rc = check_view(*o)) return rc;
    if (int rc = check_alias_bwd(go, xq, xk, v, o, dxq, dxk, dvv, B, H, N, r, dv, wide_out)) return rc;
    if (B == 0 || H == 0 || N == 0) return FLA_OK;
    if (!state_in) return FLA_ERR_NULL_POINTER;
    const PolyPlan pl = poly_plan(B, H, N, r, dv);
    if (int rc = check_poly_chunked(pl, dtype, pl.work_bytes, workspace_bytes, workspace, state_in)) return rc;
    if (!vec_ok(go, dv) || !vec_ok(xq, r) || !vec_ok(xk, r) || !vec_ok(v, dv) || !vec_ok(dxq, r) || !vec_ok(dxk, r) ||
        !vec_ok(dvv, dv) || (o && !vec_ok(*o, dv)))
        return FLA_ERR_UNSUPPORTED;
    fla::PolyWalkParams w{};
    poly_common(w, pl, xq, xk, v, B, H, N, r, dv, coef);
    w.wide_out = wide_out;
    w.go = go.ptr, w.gs_b = go.strides[0], w.gs_h = go.strides[1], w.gs_n = go.strides[2];
    if (o) w.o = o->ptr, w.os_b = o->strides[0], w.os_h = o->strides[1], w.os_n = o->strides[2];
    w.dq = const_cast<void *>(dxq.ptr), w.dqs_b = dxq.strides[0], w.dqs_h = dxq.strides[1], w.dqs_n = dxq.strides[2];
    w.dk = const_cast<void *>(dxk.ptr), w.dks_b = dxk.strides[0], w.dks_h = dxk.strides[1], w.dks_n = dxk.strides[2];
    w.dv = const_cast<void *>(dvv.ptr), w.dvs_b = dvv.strides[0], w.dvs_h = dvv.strides[1], w.dvs_n = dvv.strides[2];
    w.denom = const_cast<float *>(denom);
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (w.vhalf) {
        w.dq_part = reinterpret_cast<float *>(static_cast<char *>(workspace) + pl.total_bytes + pl.sums_bytes);
        w.dk_part = w.dq_part + pl.part_bytes / 4;
    }
    return poly_run(pl, w, true, state_in, workspace, s);
}

// Which evaluation is faster on MI355X (bench.py --crossover): the quadratic kernels' time grows with W = B H N^2 D (D: the
// larger padded head dim) above the time of one workgroup's longest row tile, which grows with N; the chunk-wise kernels'
// with B H N D above a floor of launches.  Measured quadratic time over chunk-wise time, widths 32 ... 128 and 64/32, 128/64, 128/32, B H 1 ...
// 192, N 256 ... 8192.  Forward + backward (dQ by its own walk, see chunked_backward), equal widths: from W = B H N^2 D = 4e9
// (8e9 at 128) 1.17 to 4.8 with few heads or many (0.90 at 32 columns, B H 16, N 3072); few heads and long: N = 4096 1.5 to
// 3.1, N = 2048 1.42 to 2.0 at 64 and 128 columns, 0.88 to 1.19 at 32; N = 1024 0.67 to 1.2.  Widths that differ (small-V
// operator): N = 1024 1.38 to 2.1, from W = 5e8 (1e9 below 128) 1.08 to 1.6.  Forward alone, at its line below: W from 1.2e10
// (5e9 at 32 columns) 1.1 to 2, N = 2048 1.17 to 1.9, and earlier by width.
int prefers_chunked(int64_t B, int64_t H, int64_t N, int64_t D_qk, int64_t D_v, bool backward) {
    if (B < 1 || H < 1 || N < 1 || D_qk < 1 || D_qk > 256 || D_v < 1 || D_v > 256) return 0;
    const double w = (double)B * (double)H * (double)N * (double)N * (double)padded(D_qk > D_v ? D_qk : D_v);
    const WalkPlan wp = walk_plan(B, H, N, D_qk, D_v, true);
    // Widths that are no multiples of 8: the quadratic operator runs the bounds-checked kernel, the chunk-wise one the
    // fast kernels of either kind on copies with aligned rows, at the cost of two copy launches.  Quadratic time over
    // chunk-wise time, B H = 1 ... 64, at the last N below and the first N from the line on -- forward alone: 20 columns
    // 0.95 to 1.06 at 512, 1.3 to 1.8 at 1024; 36 columns 0.80 to 0.86 at 128, 1.12 to 1.18 at 256; 91/64 and 100 0.91 to
    // 1.1 at 64, 1.17 to 1.4 at 128; wider (153/64, 153/128) 1.15 to 2.1 from 64 to 256.  Forward + backward: 20 columns
    // 0.80 to 0.87 at 128, 1.12 to 1.21 at 256; 36 columns 0.92 to 0.97 at 64, 1.24 to 1.27 at 128; wider 1.1 to 3.3.
    // (A v wider than 128 columns: the rule of multiples of 8 below -- dQ and dK would be rounded once per half of v.)
    if (D_v <= 128 && pack_plan(B, H, N, D_qk, D_v).ok) {
        const int64_t d = padded(D_qk > D_v ? D_qk : D_v);
        if (backward) return d <= 32 ? N >= 256 : d <= 64 ? N >= 128 : 1;
        return d <= 32 ? N > 512 : d <= 64 ? N >= 256 : d <= 128 ? N >= 128 : 1;
    }
    // (padded widths that differ: the quadratic side is the small-V operator, whose wide products are two launches)
    // Forward alone, B H 1 ... 520: 64 columns 1.10 to 1.4 at N = 768 (0.90 to 1.2 at 576), 32 and 128 columns 1.06 to 1.3 at 1024
    // (0.94 to 1.2 at 768), 64 / 32, 128 / 64 and 128 / 32 1.06 to 1.5 at 1024; a single segment per head, which has no totals to
    // wait for, 1.12 to 2.3 from N = 320 on.
    const bool equal = pad_index(D_qk) == pad_index(D_v), one = wp.n_seg == 1 && N > 256;
    // Up to 256 rows above 64 columns (widths that differ: one segment of two to four chunks).  Pairs, 128 / 64 and 128 / 32: B H 300 ... 1024
    // 1.22 to 1.42 from N = 128 on (the quadratic products' second round of workgroups); up to 256 heads 1.04 to 1.30 from W = 1.7e9 on, 0.93 to
    // 1.09 below it, where two launches wait for the host for 36 us and three for 38.  Forward alone, B H 2000, N 256 1.21 and 1.27.
    if (wp.ok && N < 128 && wp.split) return 0;
    if (wp.ok && !backward) return one || N >= (wp.D == 64 && equal ? 768 : 1024) || w >= (wp.D <= 32 ? 5e9 : 1.2e10);
    if (wp.ok && !equal && wp.split && N <= 256) return B * H > 256 || w >= 1.7e9;
    if (wp.ok && !equal) return N >= 1024 || w >= (wp.D <= 64 ? 1e9 : 5e8);
    // Equal padded head dims up to 128.  (Pairs gain earlier on the GPU -- 64 columns 1.2 to 1.5 from N = 768 on --, but there the
    // host, 58 us for the quadratic pair's two launches and 72 for the chunk-wise one's four, takes longer than either.  Single
    // segments of 128 columns: B H 130 N 448 74 / 64 us, B H 256 N 320 92 / 61.)
    if (wp.ok) return N >= (wp.D <= 32 ? 4096 : 2048) || w >= (wp.D <= 64 ? 4e9 : one ? 3.2e9 : 8e9);
    // D_qk in (128, 256].  D_v <= 64: pairs 1.13 to 5 from N = 1024 or W = 1e9 on (192 / 64 and 256 / 64, N 128 ... 256, B H 60 ... 1024 1.15 to
    // 1.51), forward alone 1.13 to 2.9 from N = 1024 (N = 512 0.82 to 1.1).  D_v in (64, 128]: pairs 1.35 to 3.1 from N = 2048, 1.3 from
    // W = 2.5e10 (1.0 at 1.7e10, N = 1024; at N = 256 0.99 to 1.07); forward alone 1.14 to 1.55 from N = 4096, at N = 2048 1.1 to 1.4 with
    // B H <= 4 and 0.93 with 16.
    if (wide_plan(B, H, N, D_qk, D_v).ok) {
        if (N < 128 || (D_v > 64 && N <= 256)) return 0;
        if (D_v <= 64) return N >= 1024 || (backward && w >= 1e9);
        return backward ? N >= 2048 || w >= 2.5e10 : N >= 4096 || (N >= 2048 && B * H <= 4) || w >= 5e10;
    }
    if (vsplit_plan(B, H, N, D_qk, D_v).ok) return w >= 3e10;  // D_v in (128, 256] as two column halves of v
    return N >= 4096;  // chunk states in memory, a launch per product and state (measured at 256 / 256)
}

// The operators' choice: the table above, whose answers callers of the C ABI go by, and earlier with both widths in (128, 256], where the
// gradients are summed in fp32 over both halves and rounded once.  Those, widths 160, 192 and 256, B H 1 ... 300 (400 from N = 320 on): at N 128, 192 and
// 256 (one segment per head) pairs 1.04 to 1.84, forward alone 1.13 to 1.8; from N = 320 on pairs 1.13 to 2.1 up to N = 700, 1.5 to 2.4 at N = 1024,
// 2.2 to 4 at 2048, 4.2 to 25 beyond; forward alone 0.97 to 4.7, but 0.81 to 0.96 below N = 640 with two segments per head (33 to 64 heads).
// Errors over the quadratic kernels', N 128 ... 1024, 192 heads each: dQ and dK 0.997 to 1.004, O and dV 0.69 to 1.002.
int operators_prefer_chunked(int64_t B, int64_t H, int64_t N, int64_t D_qk, int64_t D_v, bool backward) {
    if (const WalkPlan quad = quad_plan(B, H, N, D_qk, D_v); quad.ok && D_qk % 8 == 0 && D_v % 8 == 0)
        return N >= 128 && (backward || quad.n_seg != 2 || N >= 640);
    return prefers_chunked(B, H, N, D_qk, D_v, backward);
}

// Quadratic time over chunk-wise time of the polynomial map.  R 8 and 16, with and without the normaliser, B H 1 ... 1024, N 100 ... 4096.  Pairs,
// D_v 64: 1.0 to 4.8 (0.91 to 0.99 at a few N of 200).  D_v 32, up to 256 heads: 0.94 to 4.2 (0.88 at B H 128, N 512); 512
// and 1024 heads: N 128 1.07 to 1.6, N 200 to 512 0.59 to 1.06, N 1024 0.85 to 1.18, N 2048 1.34 to 1.7.  Forward
// alone: N 4096 1.07 to 2.6; N 2048 1.1 to 1.5 with at most four heads, 0.62 to 1.09 with more; below 0.36 to 1.0.
// D_v above 64, two halves.  Pairs, one chunk (N up to 128): 0.95 to 1.15 (normalised 1.0 to 1.36 at 128), N 64 with 800 and 1024 heads 0.83
// to 0.93.  Beyond, 120 and 128 columns, plain and normalised at 120: N 160 to 512 0.60 to 1.08, N 700 0.92 to 1.2, N 1000 0.97 to 1.5, N 2048 1.0 to 2.4,
// 4096 1.8 to 5.5; normalised at 128: N 160 and 200 0.97 to 1.09 up to 128 heads and 0.75 to 1.02 above, N 256 0.92 to 1.18, N 384 0.99 to 1.32, N 700 1.15 to
// 1.4.  72 and 104 columns, whose second half is half padding or more: up to 33 heads N 512 0.96 to 1.02, N 700 0.95 to 1.21, N 1000 1.2 to 1.5; 48 heads
// N 1000 to 2048 0.91 to 1.09, 4096 1.7 to 2.1; more heads N 2048 1.04 to 1.6.  Forward alone: up to 16 heads 1.3 to 2.2 from N 1024 on, 4096 1.5 to 4.
// R above 16, three launches a walk, 24 and 32 columns over 32 to 128: pairs at N 8192 with 16 heads and more 1.02 to 1.7 (72 columns normalised 0.92 to
// 1.02; N 9216 1.24 to 1.9), with up to 8 1.35 to 4, N 4096 up to 8 heads 1.08 to 2.4, N 16384 1.7 to 6; forward alone N 16384 1.2 to 2.9, N 8192 up to 4 heads 0.94 to 1.9 (32
// columns of v 0.88 and 0.95 with 4 heads, 1.12 to 1.4 with up to 2).
bool poly_prefers_chunked(int64_t B, int64_t H, int64_t N, int64_t R, int64_t D_v, int dtype, bool backward, bool normalised) {
    if (dtype != FLA_DTYPE_BF16 || !poly_plan(B, H, N, R, D_v).ok) return false;
    const int64_t heads = B * H;
    if (R > 16) {
        if (!backward) return N >= 16384 || (N >= 8192 && heads <= (D_v > 32 ? 4 : 2));
        return N >= (heads <= 8 ? 4096 : D_v > 64 && D_v <= 96 ? 9216 : 8192);
    }
    if (D_v > 64) {
        if (!backward) return N >= 4096 || (N >= 1024 && heads <= 16);
        if (N <= 128) return (D_v > 112 || heads <= 48) && (N > 64 || heads <= 512);
        if (D_v > 120 && normalised) return N >= 256 || heads <= 128;
        if (D_v > 112 || heads <= 33) return N >= 768;
        return N >= (heads <= 48 ? 3072 : 2048);
    }
    if (backward) return D_v > 32 || heads <= 256 || N <= 128 || N >= 2048;
    return N >= 4096 || (N >= 2048 && heads <= 4);
}

}  // namespace

extern "C" {

#if defined(FLA_TRACE_LAUNCHES)
// The launchers' choice of a map of workgroups to (head, part), and the kernels' map, for all of a grid: `items` receives both of every
// workgroup (head < 0: none).
int fla_trace_xcd_place(int BH, int parts, int64_t stride_h, int most, int resident) { return fla::xcd_place(BH, parts, stride_h, most, resident); }
uint32_t fla_trace_xcd_inverse(int parts) { return fla::xcd_inverse(parts); }
void fla_trace_xcd_items(int grid, int BH, int parts, int place, uint32_t inverse, int32_t *items) {  // (inverse 1: the kernel divides)
    for (int wg = 0; wg < grid; ++wg) {
        const fla::XcdItem item = inverse == 1 ? fla::xcd_item(wg, BH, parts, place) : fla::xcd_item(wg, BH, parts, place, inverse);
        items[2 * wg] = item.bh, items[2 * wg + 1] = item.part;
    }
}
#endif

int fla_abi_version(void) { return FLA_ABI_VERSION; }

int fla_convert(const void *const *src, void *const *dst, const int64_t *counts, int n, int widen, int dtype, void *stream) {
    if (dtype != FLA_DTYPE_BF16 && dtype != FLA_DTYPE_F16) return FLA_ERR_DTYPE;
    if (n < 0 || n > 4 || !src || !dst || !counts) return n == 0 ? FLA_OK : FLA_ERR_SHAPE;
    fla::ConvertParams p{};
    for (int i = 0; i < n; ++i) {
        if (counts[i] < 0) return FLA_ERR_SHAPE;
        if (counts[i] && (!src[i] || !dst[i])) return FLA_ERR_NULL_POINTER;
        // (the 16-byte side in 16-byte accesses, the fp32 side in 32-byte ones that the compiler splits)
        if (reinterpret_cast<uintptr_t>(src[i]) % 16 || reinterpret_cast<uintptr_t>(dst[i]) % 16) return FLA_ERR_UNSUPPORTED;
        p.src[i] = src[i], p.dst[i] = dst[i], p.count[i] = counts[i];
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    const hipError_t e = dtype == FLA_DTYPE_BF16 ? fla::launch_convert<__bf16>(p, n, widen != 0, s)
                                                 : fla::launch_convert<_Float16>(p, n, widen != 0, s);
    return e == hipSuccess ? FLA_OK : FLA_ERR_LAUNCH;
}

const char *fla_strerror(int status) {
    switch (status) {
        case FLA_OK: return "ok";
        case FLA_ERR_NULL_POINTER: return "a required pointer is NULL";
        case FLA_ERR_DTYPE: return "dtype must be FLA_DTYPE_BF16 or FLA_DTYPE_F16";
        case FLA_ERR_HEAD_DIM: return "Only head_dims <= 256 are supported.";
        case FLA_ERR_V_HEAD_DIM:
            return "value head dimension must be a power of 2 no larger than the padded query/key head dimension";
        case FLA_ERR_SHAPE: return "B, H and N must be non-negative and B*H, N at most 2^30";
        case FLA_ERR_STRIDE: return "strides must be given, non-negative, with innermost stride 1";
        case FLA_ERR_LAUNCH: return "the HIP runtime rejected the kernel launch";
        case FLA_ERR_UNSUPPORTED: return "no kernel was built for this combination";
        case FLA_ERR_WORKSPACE: return "workspace is NULL, not 16-byte aligned, or smaller than fla_chunked_workspace_bytes()";
        case FLA_ERR_ALIAS: return "an output tensor overlaps an input or another output in memory";
        default: return "unknown fla status";
    }
}

int fla_linear_attn_fwd(const void *q, const void *k, const void *v, void *o, int64_t B, int64_t H, int64_t N,
                        int64_t D, const int64_t *q_strides, const int64_t *k_strides, const int64_t *v_strides,
                        const int64_t *o_strides, int dtype, void *stream) {
    if (int rc = check_common(B, H, N, dtype)) return rc;
    if (D < 1 || D > 256) return FLA_ERR_HEAD_DIM;
    return forward({q, q_strides}, {k, k_strides}, {v, v_strides}, {o, o_strides}, B, H, N, D, D, dtype, stream);
}

int fla_linear_attn_bwd(const void *grad_out, const void *q, const void *k, const void *v, void *dq, void *dk,
                        void *dv, int64_t B, int64_t H, int64_t N, int64_t D, const int64_t *go_strides,
                        const int64_t *q_strides, const int64_t *k_strides, const int64_t *v_strides,
                        const int64_t *dq_strides, const int64_t *dk_strides, const int64_t *dv_strides, int dtype,
                        void *stream) {
    if (int rc = check_common(B, H, N, dtype)) return rc;
    if (D < 1 || D > 256) return FLA_ERR_HEAD_DIM;
    return backward({grad_out, go_strides}, {q, q_strides}, {k, k_strides}, {v, v_strides}, {dq, dq_strides},
                    {dk, dk_strides}, {dv, dv_strides}, B, H, N, D, D, dtype, stream);
}

int fla_linear_attn_smallv_fwd(const void *q, const void *k, const void *v, void *o, int64_t B, int64_t H,
                               int64_t N, int64_t D_qk, int64_t D_v, const int64_t *q_strides,
                               const int64_t *k_strides, const int64_t *v_strides, const int64_t *o_strides,
                               int dtype, void *stream) {
    if (int rc = check_common(B, H, N, dtype)) return rc;
    if (D_qk < 1 || D_qk > 256) return FLA_ERR_HEAD_DIM;
    if (D_v < 1 || next_pow2(D_v) != D_v || D_v > next_pow2(D_qk)) return FLA_ERR_V_HEAD_DIM;
    return forward({q, q_strides}, {k, k_strides}, {v, v_strides}, {o, o_strides}, B, H, N, D_qk, D_v, dtype,
                   stream);
}

int fla_linear_attn_smallv_bwd(const void *grad_out, const void *q, const void *k, const void *v, void *dq,
                               void *dk, void *dv, int64_t B, int64_t H, int64_t N, int64_t D_qk, int64_t D_v,
                               const int64_t *go_strides, const int64_t *q_strides, const int64_t *k_strides,
                               const int64_t *v_strides, const int64_t *dq_strides, const int64_t *dk_strides,
                               const int64_t *dv_strides, int dtype, void *stream) {
    if (int rc = check_common(B, H, N, dtype)) return rc;
    if (D_qk < 1 || D_qk > 256) return FLA_ERR_HEAD_DIM;
    if (D_v < 1 || D_v > 256) return FLA_ERR_V_HEAD_DIM;
    return backward({grad_out, go_strides}, {q, q_strides}, {k, k_strides}, {v, v_strides}, {dq, dq_strides},
                    {dk, dk_strides}, {dv, dv_strides}, B, H, N, D_qk, D_v, dtype, stream);
}

int64_t fla_linear_attn_copies_bytes(int64_t B, int64_t H, int64_t N, int64_t D_qk, int64_t D_v, int backward) {
    const PackPlan p = pack_plan(B, H, N, D_qk, D_v);
    return on_copies(p, D_qk, D_v) ? copies_bytes(p, backward != 0) : 0;
}

// Measured, fp16, widths 20 ... 250, B H 1 ... 128, N 64 ... 2048, bounds-checked time over the copies': forward above 64 columns 1.0 (N 64) to
// 7; up to 64 columns 0.7 to 1.0 up to N 256, where the copies' two launches weigh more, 1.2 to 3.5 from N 512 on (20 columns, B H 128,
// N 512 0.95, N 1024 1.2).  Backward 1.2 to 14, at 20 columns and N 64 1.0.
int fla_linear_attn_prefers_copies(int64_t B, int64_t H, int64_t N, int64_t D_qk, int64_t D_v, int backward) {
    if (!on_copies(pack_plan(B, H, N, D_qk, D_v), D_qk, D_v)) return 0;
    const int64_t widest = D_qk > D_v ? D_qk : D_v;
    if (backward) return widest > 32 || N >= 128;
    return widest > 64 || N >= (widest > 32 ? 512 : 1024);
}

// Through the operators the host weighs in, which the two copy launches keep for 4 us of the 65 to 80 of a pair.  fp16 pairs, B H 1 ... 300,
// bounds-checked time over the copies': 20 columns N 256 0.95 to 1.01, 512 1.19 to 1.34; 36 and 60 N 64 0.92 to 0.96, 128 0.91 to 1.05, 256 1.29 to 1.5; 100 and
// 153 / 64 N 64 0.90 to 0.95 and with 300 heads 1.6 to 1.8, 128 1.24 to 2.1; 250 N 64 2.2 to 3.4.  Forward alone, 91 / 64, N 64 1.24 to 1.38 up to 128 heads, 0.90
// with 300.
int fla_linear_attn_operator_prefers_copies(int64_t B, int64_t H, int64_t N, int64_t D_qk, int64_t D_v, int backward) {
    if (!fla_linear_attn_prefers_copies(B, H, N, D_qk, D_v, backward)) return 0;
    const int64_t heads = B * H, widest = D_qk > D_v ? D_qk : D_v;
    if (!backward) return N > 64 || D_v > 64 || D_qk > 128 || heads <= 128;
    return N >= (widest <= 32 ? 512 : widest <= 64 ? 256 : 128) || (D_qk > 128 && D_v > 128) || (widest > 64 && heads > 256);
}

int fla_linear_attn_copies_fwd(const void *q, const void *k, const void *v, void *o, int64_t B, int64_t H, int64_t N, int64_t D_qk,
                               int64_t D_v, const int64_t *q_strides, const int64_t *k_strides, const int64_t *v_strides,
                               const int64_t *o_strides, int dtype, void *workspace, int64_t workspace_bytes, void *stream) {
    return copies_forward({q, q_strides}, {k, k_strides}, {v, v_strides}, {o, o_strides}, B, H, N, D_qk, D_v, dtype, workspace,
                          workspace_bytes, stream);
}

int fla_linear_attn_copies_bwd(const void *grad_out, const void *q, const void *k, const void *v, void *dq, void *dk, void *dv,
                               int64_t B, int64_t H, int64_t N, int64_t D_qk, int64_t D_v, const int64_t *go_strides,
                               const int64_t *q_strides, const int64_t *k_strides, const int64_t *v_strides, const int64_t *dq_strides,
                               const int64_t *dk_strides, const int64_t *dv_strides, int dtype, void *workspace,
                               int64_t workspace_bytes, void *stream) {
    return copies_backward({grad_out, go_strides}, {q, q_strides}, {k, k_strides}, {v, v_strides}, {dq, dq_strides}, {dk, dk_strides},
                           {dv, dv_strides}, B, H, N, D_qk, D_v, dtype, workspace, workspace_bytes, stream);
}

int fla_linear_attn_bwd_fused_dkdv(const void *grad_out, const void *q, const void *k, const void *v, void *dq, void *dk,
                                   void *dv, int64_t B, int64_t H, int64_t N, int64_t D_qk, int64_t D_v,
                                   const int64_t *go_strides, const int64_t *q_strides, const int64_t *k_strides,
                                   const int64_t *v_strides, const int64_t *dq_strides, const int64_t *dk_strides,
                                   const int64_t *dv_strides, int dtype, void *stream) {
    if (int rc = check_common(B, H, N, dtype)) return rc;
    if (D_qk < 1 || D_qk > 256) return FLA_ERR_HEAD_DIM;
    if (D_v < 1 || D_v > 256) return FLA_ERR_V_HEAD_DIM;
    return backward_fused_dkdv({grad_out, go_strides}, {q, q_strides}, {k, k_strides}, {v, v_strides}, {dq, dq_strides},
                               {dk, dk_strides}, {dv, dv_strides}, B, H, N, D_qk, D_v, dtype, stream);
}

int fla_tri_xyt_z(const void *x, const void *y, const void *z, void *out, int64_t B, int64_t H, int64_t N,
                  int64_t D_c, int64_t D_o, const int64_t *x_strides, const int64_t *y_strides,
                  const int64_t *z_strides, const int64_t *out_strides, int upper, int dtype, void *stream) {
    if (int rc = check_common(B, H, N, dtype)) return rc;
    if (D_c < 1 || D_c > 256 || D_o < 1 || D_o > 256) return FLA_ERR_HEAD_DIM;
    const View vx{x, x_strides}, vy{y, y_strides}, vz{z, z_strides}, vo{out, out_strides};
    const View all[] = {vx, vy, vz, vo};
    for (const View &t : all)
        if (int rc = check_view(t)) return rc;
    if (int rc = check_alias_fwd(vx, vy, vz, vo, B, H, N, D_c, D_o)) return rc;
    return run_tri(vx, vy, vz, vo, B, H, N, D_c, D_o, upper, dtype, stream);
}

int64_t fla_chunked_workspace_bytes(int64_t B, int64_t H, int64_t N, int64_t D_c, int64_t D_o) {
    if (B < 0 || H < 0 || N < 0 || D_c < 1 || D_c > 256 || D_o < 1 || D_o > 256) return 0;
    return chunked_bytes(B, H, N, D_c, D_o);
}

int fla_tri_xyt_z_chunked(const void *x, const void *y, const void *z, void *out, int64_t B, int64_t H, int64_t N,
                          int64_t D_c, int64_t D_o, const int64_t *x_strides, const int64_t *y_strides,
                          const int64_t *z_strides, const int64_t *out_strides, int upper, int dtype,
                          void *workspace, int64_t workspace_bytes, void *stream) {
    if (int rc = check_common(B, H, N, dtype)) return rc;
    if (D_c < 1 || D_c > 256 || D_o < 1 || D_o > 256) return FLA_ERR_HEAD_DIM;
    const View vx{x, x_strides}, vy{y, y_strides}, vz{z, z_strides}, vo{out, out_strides};
    const View all[] = {vx, vy, vz, vo};
    for (const View &t : all)
        if (int rc = check_view(t)) return rc;
    if (int rc = check_alias_fwd(vx, vy, vz, vo, B, H, N, D_c, D_o)) return rc;
    return run_tri_chunked(vx, vy, vz, vo, B, H, N, D_c, D_o, upper, dtype, workspace, workspace_bytes, stream);
}

int fla_linear_attn_prefers_chunked(int64_t B, int64_t H, int64_t N, int64_t D_qk, int64_t D_v) {
    return prefers_chunked(B, H, N, D_qk, D_v, true);
}
int fla_linear_attn_forward_prefers_chunked(int64_t B, int64_t H, int64_t N, int64_t D_qk, int64_t D_v) {
    return prefers_chunked(B, H, N, D_qk, D_v, false);
}

int fla_linear_attn_operator_prefers_chunked(int64_t B, int64_t H, int64_t N, int64_t D_qk, int64_t D_v, int backward) {
    return operators_prefer_chunked(B, H, N, D_qk, D_v, backward != 0);
}
// fp16 with gradients: the widths whose walks scale their states in both directions, and the lines.  Through autograd the quadratic pair's two
// launches wait for the host for 58 us, the chunk-wise one's four or five for 68 to 80.  Quadratic time over chunk-wise time, B H 2 ... 600,
// below and above: 128 columns N 2048 76 / 81 us (B H 2), 98 / 83 (16), N 1024 96 / 85 (64), N 4096 171 / 81 (2); 128 / 64 and 128 / 32 N 1024 74 / 78
// (16), 88 / 76 (64), N 2048 122 / 85 (2); 64 columns N 1024 58 / 69 (64), 126 / 75 (200), N 2048 58 / 68 (2), 64 / 67 (16), 129 / 68 (64), N 4096 110 /
// 67 (2); 32 columns N 2048 69 / 73 (64), 200 / 72 (200), N 4096 66 / 68 (2), 92 / 70 (16), N 768 134 / 66 (600).
int fla_linear_attn_f16_pair_prefers_chunked(int64_t B, int64_t H, int64_t N, int64_t D_qk, int64_t D_v) {
    if (B < 1 || H < 1 || N < 768 || D_qk < 1 || D_v < 1 || D_qk > 128 || D_v > 128 || D_qk % 8 || D_v % 8) return 0;
    const int64_t d = padded(D_qk > D_v ? D_qk : D_v);
    const bool equal = padded(D_qk) == padded(D_v);
    const double w = (double)B * (double)H * (double)N * (double)N * (double)d;
    if (d == 128) return N >= (equal ? 3072 : 1536) || w >= 8e9;
    if (!equal) return 0;  // (no room for the saved copies' scales)
    return d == 64 ? N >= 3072 || w >= 7e9 : N >= 4096 || w >= 1e10;
}
int64_t fla_linear_attn_chunked_state_bytes(int64_t B, int64_t H, int64_t N, int64_t D_qk, int64_t D_v) {
    if (B < 0 || H < 0 || N < 0 || D_qk < 1 || D_qk > 256 || D_v < 1 || D_v > 256) return 0;
    const int64_t plain = shared_state_bytes(B, H, N, D_qk, D_v);  // (the normalised operator's, whatever the widths)
    const PackPlan p = pack_plan(B, H, N, D_qk, D_v);
    return p.ok && packed_state_bytes(p) > plain ? packed_state_bytes(p) : plain;
}

int64_t fla_linear_attn_chunked_workspace_bytes(int64_t B, int64_t H, int64_t N, int64_t D_qk, int64_t D_v) {
    if (B < 0 || H < 0 || N < 0 || D_qk < 1 || D_qk > 256 || D_v < 1 || D_v > 256) return 0;
    const int64_t plain = chunked_op_workspace_bytes(B, H, N, D_qk, D_v);  // (the feature-map operator's, whatever the widths)
    const PackPlan p = pack_plan(B, H, N, D_qk, D_v);
    return p.ok && packed_work_bytes(p) > plain ? packed_work_bytes(p) : plain;
}

int64_t fla_linear_attn_chunked_fwd_workspace_bytes(int64_t B, int64_t H, int64_t N, int64_t D_qk, int64_t D_v, int with_state) {
    if (B < 0 || H < 0 || N < 0 || D_qk < 1 || D_qk > 256 || D_v < 1 || D_v > 256) return 0;
    if (const PackPlan p = pack_plan(B, H, N, D_qk, D_v); p.ok) return packed_fwd_work_bytes(p, with_state != 0);
    return chunked_op_workspace_bytes(B, H, N, D_qk, D_v);
}

int fla_linear_attn_chunked_state_operands(int64_t B, int64_t H, int64_t N, int64_t D_qk, int64_t D_v, int64_t *offsets,
                                           int64_t *pitches) {
    if (B < 0 || H < 0 || N < 0 || D_qk < 1 || D_qk > 256 || D_v < 1 || D_v > 256 || !offsets || !pitches) return 0;
    const PackPlan p = pack_plan(B, H, N, D_qk, D_v);
    if (!p.ok) return 0;
    for (int i = 0; i < 3; ++i) {
        const bool copied = i < 2 ? p.q_bytes != 0 : p.v_bytes != 0;
        offsets[i] = copied ? p.inner_state + i * p.q_bytes : -1, pitches[i] = i < 2 ? p.wq : p.wv;
    }
    return 1;
}

int fla_linear_attn_chunked_grads_f32(int64_t B, int64_t H, int64_t N, int64_t D_qk, int64_t D_v, int plain, int with_state) {
    if (B < 1 || H < 1 || N < 1 || D_qk < 1 || D_qk > 256 || D_v < 1 || D_v > 256) return 0;
    return wide_grads_sizes(B, H, N, D_qk, D_v, plain != 0, with_state != 0);
}

int fla_linear_attn_chunked_fwd(const void *q, const void *k, const void *v, void *o, int64_t B, int64_t H, int64_t N,
                                int64_t D_qk, int64_t D_v, const int64_t *q_strides, const int64_t *k_strides,
                                const int64_t *v_strides, const int64_t *o_strides, int dtype, void *state_out,
                                int32_t *state_valid, void *workspace, int64_t workspace_bytes, void *stream) {
    if (state_valid) *state_valid = 0;
    if (int rc = check_common(B, H, N, dtype)) return rc;
    if (D_qk < 1 || D_qk > 256) return FLA_ERR_HEAD_DIM;
    if (D_v < 1 || D_v > 256) return FLA_ERR_V_HEAD_DIM;
    if (const PackPlan p = pack_plan(B, H, N, D_qk, D_v); p.ok)
        return packed_forward(p, {q, q_strides}, {k, k_strides}, {v, v_strides}, {o, o_strides}, B, H, N, D_qk, D_v, dtype,
                              state_out, state_valid, workspace, workspace_bytes, stream);
    return chunked_forward({q, q_strides}, {k, k_strides}, {v, v_strides}, {o, o_strides}, B, H, N, D_qk, D_v, dtype,
                           state_out, state_valid, workspace, workspace_bytes, stream);
}

int fla_linear_attn_chunked_fwd_static(const void *q, const void *k, const void *v, void *o, int64_t B, int64_t H,
                                       int64_t N, int64_t D_qk, int64_t D_v, const int64_t *q_strides,
                                       const int64_t *k_strides, const int64_t *v_strides, const int64_t *o_strides,
                                       int dtype, void *stream) {
    if (int rc = check_common(B, H, N, dtype)) return rc;
    if (D_qk < 1 || D_qk > 256) return FLA_ERR_HEAD_DIM;
    if (D_v < 1 || D_v > 256) return FLA_ERR_V_HEAD_DIM;
    // what this call's kernels use of the workspace: without a state to hand over the walk path needs
    // the segments' entry states only; operands off that path take the 256-row chunks with their states
    const View vq{q, q_strides}, vk{k, k_strides}, vv{v, v_strides}, vo{o, o_strides};
    const View all[] = {vq, vk, vv, vo};
    for (const View &t : all)
        if (int rc = check_view(t)) return rc;
    const WalkPlan wp = walk_plan(B, H, N, D_qk, D_v, true);
    int64_t need = chunked_op_workspace_bytes(B, H, N, D_qk, D_v);
    if (wp.ok)
        need = fla::fast_path_ok(make_params(vq, vk, vv, vo, B, H, N, D_qk, D_v, 0)) ? wp.work_bytes
                                                                                      : chunked_bytes(B, H, N, D_qk, D_v);
    if (need > (int64_t)FLA_STATIC_SCRATCH_BYTES) return FLA_ERR_WORKSPACE;
    void *ws = nullptr;
    if (int rc = static_scratch(&ws)) return rc;
    return chunked_forward({q, q_strides}, {k, k_strides}, {v, v_strides}, {o, o_strides}, B, H, N, D_qk, D_v, dtype,
                           nullptr, nullptr, ws, FLA_STATIC_SCRATCH_BYTES, stream);
}

int fla_feature_attn_fwd(const void *xq, const void *xk, const void *v, void *o, void *q_out, void *k_out, int64_t B,
                         int64_t H, int64_t N, int64_t D_qk, int64_t D_v, const int64_t *xq_strides,
                         const int64_t *xk_strides, const int64_t *v_strides, const int64_t *o_strides,
                         const int64_t *q_out_strides, const int64_t *k_out_strides, int feature_map, int dtype,
                         void *state_out, int32_t *state_valid, void *workspace, int64_t workspace_bytes, void *stream) {
    if (state_valid) *state_valid = 0;
    if (int rc = check_common(B, H, N, dtype)) return rc;
    if (D_qk < 1 || D_qk > 256) return FLA_ERR_HEAD_DIM;
    if (D_v < 1 || D_v > 256) return FLA_ERR_V_HEAD_DIM;
    if (feature_map != FLA_MAP_ELU1 && feature_map != FLA_MAP_SOFTPLUS) return FLA_ERR_UNSUPPORTED;
    const View mapped[2] = {{q_out, q_out_strides}, {k_out, k_out_strides}};
    return feature_forward({xq, xq_strides}, {xk, xk_strides}, {v, v_strides}, {o, o_strides}, mapped, B, H, N, D_qk, D_v,
                           feature_map, dtype, 1, state_out, state_valid, workspace, workspace_bytes, stream);
}

int fla_feature_attn_bwd(const void *grad_out, const void *xq, const void *xk, const void *v, void *dxq, void *dxk,
                         void *dv, int64_t B, int64_t H, int64_t N, int64_t D_qk, int64_t D_v,
                         const int64_t *go_strides, const int64_t *xq_strides, const int64_t *xk_strides,
                         const int64_t *v_strides, const int64_t *dxq_strides, const int64_t *dxk_strides,
                         const int64_t *dv_strides, int feature_map, int dtype, const void *state_in, void *workspace,
                         int64_t workspace_bytes, void *stream) {
    // (xq, xk name the forward's q_out, k_out here: phi(xq), phi(xk))
    const bool wide_out = take_wide_flag(dtype);
    if (int rc = check_common(B, H, N, dtype)) return rc;
    if (D_qk < 1 || D_qk > 256) return FLA_ERR_HEAD_DIM;
    if (D_v < 1 || D_v > 256) return FLA_ERR_V_HEAD_DIM;
    if (feature_map != FLA_MAP_ELU1 && feature_map != FLA_MAP_SOFTPLUS) return FLA_ERR_UNSUPPORTED;
    return chunked_backward({grad_out, go_strides}, {xq, xq_strides}, {xk, xk_strides}, {v, v_strides},
                            {dxq, dxq_strides}, {dxk, dxk_strides}, {dv, dv_strides}, B, H, N, D_qk, D_v, dtype,
                            state_in, workspace, workspace_bytes, stream, feature_map, nullptr, false, wide_out);
}

int fla_linear_attn_chunked_bwd(const void *grad_out, const void *q, const void *k, const void *v, void *dq, void *dk,
                                void *dv, int64_t B, int64_t H, int64_t N, int64_t D_qk, int64_t D_v,
                                const int64_t *go_strides, const int64_t *q_strides, const int64_t *k_strides,
                                const int64_t *v_strides, const int64_t *dq_strides, const int64_t *dk_strides,
                                const int64_t *dv_strides, int dtype, const void *state_in, void *workspace,
                                int64_t workspace_bytes, void *stream) {
    return plain_chunked_backward({grad_out, go_strides}, {q, q_strides}, {k, k_strides}, {v, v_strides}, {dq, dq_strides},
                                  {dk, dk_strides}, {dv, dv_strides}, B, H, N, D_qk, D_v, dtype, state_in, workspace,
                                  workspace_bytes, stream, false);
}

int fla_linear_attn_chunked_bwd_causal(const void *grad_out, const void *q, const void *k, const void *v, void *dq, void *dk,
                                       void *dv, int64_t B, int64_t H, int64_t N, int64_t D_qk, int64_t D_v,
                                       const int64_t *go_strides, const int64_t *q_strides, const int64_t *k_strides,
                                       const int64_t *v_strides, const int64_t *dq_strides, const int64_t *dk_strides,
                                       const int64_t *dv_strides, int dtype, const void *state_in, void *workspace,
                                       int64_t workspace_bytes, void *stream) {
    return plain_chunked_backward({grad_out, go_strides}, {q, q_strides}, {k, k_strides}, {v, v_strides}, {dq, dq_strides},
                                  {dk, dk_strides}, {dv, dv_strides}, B, H, N, D_qk, D_v, dtype, state_in, workspace,
                                  workspace_bytes, stream, true);
}

int fla_feature_attn_normalised_fwd(const void *xq, const void *xk, const void *v, void *o, void *q_out, void *k_out,
                                    float *denom, int64_t B, int64_t H, int64_t N, int64_t D_qk, int64_t D_v,
                                    const int64_t *xq_strides, const int64_t *xk_strides, const int64_t *v_strides,
                                    const int64_t *o_strides, const int64_t *q_out_strides,
                                    const int64_t *k_out_strides, int feature_map, float eps, int dtype, int chunked,
                                    void *state_out, int32_t *state_valid, void *workspace, int64_t workspace_bytes,
                                    void *stream) {
    if (state_valid) *state_valid = 0;
    if (int rc = check_norm_args(B, H, N, D_qk, D_v, dtype)) return rc;
    if (feature_map != FLA_MAP_ELU1 && feature_map != FLA_MAP_SOFTPLUS) return FLA_ERR_UNSUPPORTED;
    const View mapped[2] = {{q_out, q_out_strides}, {k_out, k_out_strides}};
    return normalised_forward({xq, xq_strides}, {xk, xk_strides}, {v, v_strides}, {o, o_strides}, denom, B, H, N, D_qk,
                              D_v, eps, dtype, chunked, workspace, workspace_bytes, stream, feature_map, mapped,
                              state_out, state_valid);
}

int fla_feature_attn_normalised_bwd(const void *grad_out, const void *q, const void *k, const void *v, const void *o,
                                    const float *denom, void *dxq, void *dxk, void *dv, int64_t B, int64_t H,
                                    int64_t N, int64_t D_qk, int64_t D_v, const int64_t *go_strides,
                                    const int64_t *q_strides, const int64_t *k_strides, const int64_t *v_strides,
                                    const int64_t *o_strides, const int64_t *dxq_strides, const int64_t *dxk_strides,
                                    const int64_t *dv_strides, int feature_map, int dtype, int chunked,
                                    const void *state_in, void *workspace, int64_t workspace_bytes, void *stream) {
    const bool wide_out = take_wide_flag(dtype);
    if (int rc = check_norm_args(B, H, N, D_qk, D_v, dtype)) return rc;
    if (feature_map != FLA_MAP_ELU1 && feature_map != FLA_MAP_SOFTPLUS) return FLA_ERR_UNSUPPORTED;
    return normalised_backward({grad_out, go_strides}, {q, q_strides}, {k, k_strides}, {v, v_strides}, {o, o_strides},
                               denom, {dxq, dxq_strides}, {dxk, dxk_strides}, {dv, dv_strides}, B, H, N, D_qk, D_v,
                               dtype, chunked, workspace, workspace_bytes, stream, feature_map, state_in, wide_out);
}

int64_t fla_poly_attn_workspace_bytes(int64_t B, int64_t H, int64_t N, int64_t R, int64_t D_v) {
    if (B < 0 || H < 0 || N < 0 || R < 1 || R > 32 || D_v < 1 || D_v > 128) return 0;
    const PolyLayout l = poly_layout(B, H, N, R, D_v, 1);  // the normalised backward needs the most
    return 2 * l.packed_bytes + l.do_bytes + l.dn_bytes;
}

int fla_poly_attn_fwd(const void *xq, const void *xk, const void *v, void *o, float *denom, int64_t B, int64_t H,
                      int64_t N, int64_t R, int64_t D_v, const int64_t *xq_strides, const int64_t *xk_strides,
                      const int64_t *v_strides, const int64_t *o_strides, const float *coef, float eps, int dtype,
                      void *stream) {
    if (int rc = check_poly_args(B, H, N, R, D_v, dtype, coef)) return rc;
    return poly_forward({xq, xq_strides}, {xk, xk_strides}, {v, v_strides}, {o, o_strides}, denom, B, H, N, R, D_v,
                        coef, eps, dtype, stream);
}

int fla_poly_attn_bwd(const void *grad_out, const void *xq, const void *xk, const void *v, const void *o,
                      const float *denom, void *dxq, void *dxk, void *dv, int64_t B, int64_t H, int64_t N, int64_t R,
                      int64_t D_v, const int64_t *go_strides, const int64_t *xq_strides, const int64_t *xk_strides,
                      const int64_t *v_strides, const int64_t *o_strides, const int64_t *dxq_strides,
                      const int64_t *dxk_strides, const int64_t *dv_strides, const float *coef, int dtype,
                      void *workspace, int64_t workspace_bytes, void *stream) {
    if (int rc = check_poly_args(B, H, N, R, D_v, dtype, coef)) return rc;
    const View ov{o, o_strides};
    return poly_backward({grad_out, go_strides}, {xq, xq_strides}, {xk, xk_strides}, {v, v_strides},
                         o ? &ov : nullptr, denom, {dxq, dxq_strides}, {dxk, dxk_strides}, {dv, dv_strides}, B, H, N,
                         R, D_v, coef, dtype, workspace, workspace_bytes, stream);
}

// Forward alone, measured (bf16, quadratic time over chunk-wise time, widths 32, 64, 128, B H 2 ... 192, N 256 ... 4096): N = 2048
// 1.3 to 1.9, N = 4096 2.1 to 3.8; at N = 1024 1.06 to 1.5 up to 64 columns, but 0.8 to 1.3 at 128.  Errors against fp64 are the
// smaller ones (0.86 to 0.97 of the quadratic evaluation's).  Where gradients are wanted, chunked == 1 is not chosen: the quadratic
// kernels add the normaliser's part of dQ to the rounded rest, these walks before rounding, and where the two cancel
// (early rows) single elements of dQ come out up to 1.2 of its root mean square apart (FLA_CHUNKED_PRODUCTS: 0.03 to 0.14).  fp16 stays
// quadratic: the normalised walks do not scale their state.
int fla_normalised_forward_prefers_chunked(int64_t B, int64_t H, int64_t N, int64_t D_qk, int64_t D_v, int dtype) {
    if (dtype != FLA_DTYPE_BF16 || D_qk < 1 || D_v < 1 || D_qk % 8 != 0 || D_v % 8 != 0) return 0;
    const WalkPlan wp = walk_plan(B, H, N, D_qk, D_v);
    if (!wp.ok) return 0;
    const double w = (double)B * (double)H * (double)N * (double)N * (double)wp.D;
    // (a single segment per head: 1.03 to 2.1 from N = 320 on, B H 130 ... 600)
    return N >= 2048 || (N >= 1024 && wp.D <= 64) || w >= 1.2e10 || (wp.n_seg == 1 && N > 256);
}
// Pairs, quadratic time over the time with FLA_CHUNKED_PRODUCTS (forward's totals and walk; dO, dn and its sums; the plain backward walks;
// the normaliser's terms), widths 32, 64, 96 and 128, B H 2 ... 400, N 200 ... 4096: at N = 4096 with 2 and 8 heads 1.1 to 1.7 at 32
// columns, 1.7 to 2.8 at 64, 1.9 to 2.9 at 96 and 128; N = 2048 with 2 and 8 heads 1.2 to 1.6 above 64 columns, 0.9 to 1.0 below, where both wait for
// the host (77 us of four launches, 82 of six); from W = 6e9 (5e9 above 64 columns) 1.05 to 2.1; a single segment per head 1.1 to 1.3 from
// W = 2e9 on, above 64 columns 1.11 to 1.2 from N = 300.  B H 48, N 17148, D 64 5190 -> 540 us.  Errors against fp64 0.87 to 1.00 of the
// quadratic evaluation's in out and dV, 0.97 to 1.00 in dQ and dK.
int fla_normalised_prefers_chunked(int64_t B, int64_t H, int64_t N, int64_t D_qk, int64_t D_v, int dtype) {
    if (dtype != FLA_DTYPE_BF16 || D_qk < 1 || D_v < 1 || D_qk % 8 != 0 || D_v % 8 != 0) return 0;
    const WalkPlan wp = walk_plan(B, H, N, D_qk, D_v);
    if (!wp.ok) return 0;
    const double w = (double)B * (double)H * (double)N * (double)N * (double)wp.D;
    const bool one = wp.n_seg == 1 && N > 256;
    if (wp.D > 64) return N >= 2048 || w >= 5e9 || one;
    return N >= (wp.D <= 32 ? 4096 : 3072) || w >= 6e9 || (one && w >= 2e9);
}
int fla_poly_attn_prefers_chunked(int64_t B, int64_t H, int64_t N, int64_t R, int64_t D_v, int dtype, int backward) {
    return poly_prefers_chunked(B, H, N, R, D_v, dtype, backward != 0, false);
}
int fla_poly_attn_operator_prefers_chunked(int64_t B, int64_t H, int64_t N, int64_t R, int64_t D_v, int dtype, int backward, int normalised) {
    return poly_prefers_chunked(B, H, N, R, D_v, dtype, backward != 0, normalised != 0);
}

int64_t fla_poly_attn_chunked_state_bytes(int64_t B, int64_t H, int64_t N, int64_t R, int64_t D_v) {
    return poly_plan(B, H, N, R, D_v).state_bytes;
}

int64_t fla_poly_attn_chunked_workspace_bytes(int64_t B, int64_t H, int64_t N, int64_t R, int64_t D_v) {
    return poly_plan(B, H, N, R, D_v).work_bytes;
}
int64_t fla_poly_attn_chunked_fwd_workspace_bytes(int64_t B, int64_t H, int64_t N, int64_t R, int64_t D_v) {
    return poly_plan(B, H, N, R, D_v).fwd_bytes;
}

int fla_poly_attn_chunked_fwd(const void *xq, const void *xk, const void *v, void *o, float *denom, int64_t B, int64_t H,
                              int64_t N, int64_t R, int64_t D_v, const int64_t *xq_strides, const int64_t *xk_strides,
                              const int64_t *v_strides, const int64_t *o_strides, const float *coef, float eps, int dtype,
                              void *state_out, void *workspace, int64_t workspace_bytes, void *stream) {
    if (int rc = check_poly_args(B, H, N, R, D_v, dtype, coef)) return rc;
    return poly_chunked_forward({xq, xq_strides}, {xk, xk_strides}, {v, v_strides}, {o, o_strides}, denom, B, H, N, R, D_v, coef,
                                eps, dtype, state_out, workspace, workspace_bytes, stream);
}

int fla_poly_attn_chunked_bwd(const void *grad_out, const void *xq, const void *xk, const void *v, const void *o,
                              const float *denom, void *dxq, void *dxk, void *dv, int64_t B, int64_t H, int64_t N, int64_t R,
                              int64_t D_v, const int64_t *go_strides, const int64_t *xq_strides, const int64_t *xk_strides,
                              const int64_t *v_strides, const int64_t *o_strides, const int64_t *dxq_strides,
                              const int64_t *dxk_strides, const int64_t *dv_strides, const float *coef, int dtype,
                              const void *state_in, void *workspace, int64_t workspace_bytes, void *stream) {
    const bool wide_out = take_wide_flag(dtype);
    if (int rc = check_poly_args(B, H, N, R, D_v, dtype, coef)) return rc;
    const View ov{o, o_strides};
    return poly_chunked_backward({grad_out, go_strides}, {xq, xq_strides}, {xk, xk_strides}, {v, v_strides}, o ? &ov : nullptr,
                                 denom, {dxq, dxq_strides}, {dxk, dxk_strides}, {dv, dv_strides}, B, H, N, R, D_v, coef, dtype,
                                 state_in, workspace, workspace_bytes, stream, wide_out);
}

int64_t fla_normalised_workspace_bytes(int64_t B, int64_t H, int64_t N, int64_t D_qk, int64_t D_v, int chunked) {
    if (B < 0 || H < 0 || N < 0 || D_qk < 1 || D_qk > 256 || D_v < 1 || D_v > 256) return 0;
    const NormLayout l = norm_layout(B, H, N, D_qk, D_v, chunked);
    return l.norm_bytes + l.chunk_bytes;
}

int fla_linear_attn_normalised_fwd(const void *q, const void *k, const void *v, void *o, float *denom, int64_t B,
                                   int64_t H, int64_t N, int64_t D_qk, int64_t D_v, const int64_t *q_strides,
                                   const int64_t *k_strides, const int64_t *v_strides, const int64_t *o_strides,
                                   float eps, int dtype, int chunked, void *state_out, int32_t *state_valid,
                                   void *workspace, int64_t workspace_bytes, void *stream) {
    if (state_valid) *state_valid = 0;
    if (int rc = check_norm_args(B, H, N, D_qk, D_v, dtype)) return rc;
    return normalised_forward({q, q_strides}, {k, k_strides}, {v, v_strides}, {o, o_strides}, denom, B, H, N, D_qk,
                              D_v, eps, dtype, chunked, workspace, workspace_bytes, stream, 0, nullptr, state_out,
                              state_valid);
}

int fla_linear_attn_normalised_bwd(const void *grad_out, const void *q, const void *k, const void *v, const void *o,
                                   const float *denom, void *dq, void *dk, void *dv, int64_t B, int64_t H,
                                   int64_t N, int64_t D_qk, int64_t D_v, const int64_t *go_strides,
                                   const int64_t *q_strides, const int64_t *k_strides, const int64_t *v_strides,
                                   const int64_t *o_strides, const int64_t *dq_strides, const int64_t *dk_strides,
                                   const int64_t *dv_strides, int dtype, int chunked, const void *state_in,
                                   void *workspace, int64_t workspace_bytes, void *stream) {
    const bool wide_out = take_wide_flag(dtype);
    if (int rc = check_norm_args(B, H, N, D_qk, D_v, dtype)) return rc;
    return normalised_backward({grad_out, go_strides}, {q, q_strides}, {k, k_strides}, {v, v_strides},
                               {o, o_strides}, denom, {dq, dq_strides}, {dk, dk_strides}, {dv, dv_strides}, B, H, N,
                               D_qk, D_v, dtype, chunked, workspace, workspace_bytes, stream, 0, state_in, wide_out);
}

}  // extern "C"

#include "fla_trace_structs.h"  // (the trace build's descriptions of the parameter structs; empty otherwise)
