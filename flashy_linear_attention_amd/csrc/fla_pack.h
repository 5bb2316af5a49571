// Copies of (B, H, N, width) operands with rows the LDS-DMA kernels can read -- 16-byte aligned, a whole number of
// 8-element chunks, zeros in the columns beyond the true width -- and of results from such rows back to the
// caller's.  For widths that are no multiples of 8 (Taylor features without duplicates: 91, 153 columns; head
// dims like 100), whose products otherwise run on the bounds-checked kernel with element-wise loads.
//
// Bound by memory: a thread moves one 8-element chunk of a row (a whole one with one 16-byte access at the
// row's own alignment, which is 2 bytes in general), all tensors of a call in one launch.  B H 32, N 2048,
// D_qk 153 over D_v 64, forward + backward: 999 us on the bounds-checked kernel, 128 us this way (17 of them copies of q and k; the
// walks store dQ and dK to the caller's rows themselves).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fla_launch.h"

namespace fla {

struct PackItem {
    const void *src;
    void *dst;
    int64_t ss_b, ss_h, ss_n, ds_b, ds_h, ds_n;  // element strides
    int32_t width, wp;                           // true width; dst's width: wp > width, columns width .. wp - 1 zero (packing)
                                                 // or wp == width (unpacking)
};

struct PackParams {
    PackItem item[4];
    int32_t H, N;
    int32_t rows;  // B H N
};

inline __host__ __device__ int pack_chunks(const PackItem &t) { return (t.wp + 7) / 8; }

// (a template only so that the header can be included by several translation units)
template <int kUnused = 0>
__global__ __launch_bounds__(256) void pack_rows_kernel(const PackParams p) {
    typedef uint16_t u16;
    typedef uint32_t chunk_t __attribute__((ext_vector_type(4)));
    const PackItem &t = p.item[blockIdx.y];
    const int cpr = pack_chunks(t), rpb = 256 / cpr;  // chunks per row (at most 32), rows per workgroup
    const int r = (int)threadIdx.x / cpr, c8 = ((int)threadIdx.x - r * cpr) * 8;
    const int64_t row = (int64_t)blockIdx.x * rpb + r;
    if (r >= rpb || row >= p.rows) return;
    const uint32_t bh = (uint32_t)row / (uint32_t)p.N, n = (uint32_t)row - bh * (uint32_t)p.N;
    const uint32_t b = bh / (uint32_t)p.H, h = bh - b * (uint32_t)p.H;
    const u16 *src = static_cast<const u16 *>(t.src) + b * t.ss_b + h * t.ss_h + n * t.ss_n + c8;
    u16 *dst = static_cast<u16 *>(t.dst) + b * t.ds_b + h * t.ds_h + n * t.ds_n + c8;
    chunk_t v = {0u, 0u, 0u, 0u};
    if (c8 + 8 <= t.width) {
        __builtin_memcpy(&v, src, 16);
    } else {
        u16 e[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (c8 + i < t.width) e[i] = src[i];
        __builtin_memcpy(&v, e, 16);
    }
    if (c8 + 8 <= t.wp) {
        __builtin_memcpy(dst, &v, 16);
    } else {
        u16 e[8];
        __builtin_memcpy(e, &v, 16);
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (c8 + i < t.wp) dst[i] = e[i];
    }
}

inline hipError_t launch_pack_rows(PackParams &p, int count, hipStream_t stream) {
    if (count < 1 || count > 4) return hipErrorInvalidValue;
    unsigned grid = 0;
    for (int i = 0; i < count; ++i) {
        const int cpr = pack_chunks(p.item[i]);
        if (cpr < 1 || cpr > 32) return hipErrorInvalidValue;
        const unsigned g = (unsigned)((p.rows + 256 / cpr - 1) / (256 / cpr));
        grid = g > grid ? g : grid;
    }
    return launch_kernel<pack_rows_kernel<0>>(dim3(grid, (unsigned)count), dim3(256), 0, stream, p);
}

}  // namespace fla
