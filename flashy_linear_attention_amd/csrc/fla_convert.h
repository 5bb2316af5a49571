// fp32 <-> 16-bit copies of up to four dense buffers in one launch: what autocast asks of an operator's operands and of
// their gradients.  Bound by memory and, at the sizes of a training step's activations, by its launch: B 2 H 12 N 1500
// D 80, three operands, 7 us in one launch against 3 x 4.4 us as three (and as much again for the gradients).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fla_launch.h"

namespace fla {

struct ConvertParams {
    const void *src[4];
    void *dst[4];
    int64_t count[4];  // elements
};

// eight elements per thread: two 16-byte accesses on the fp32 side, one on the other
template <typename T, bool WIDEN>
__global__ __launch_bounds__(256) void convert_kernel(const ConvertParams p) {
    typedef T t8 __attribute__((ext_vector_type(8)));
    typedef float f8 __attribute__((ext_vector_type(8), aligned(16)));
    const int i = blockIdx.y;
    const int64_t n = p.count[i], at = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 8;
    if (at >= n) return;
    if constexpr (WIDEN) {
        const T *s = static_cast<const T *>(p.src[i]) + at;
        float *d = static_cast<float *>(p.dst[i]) + at;
        if (at + 8 <= n)
            *reinterpret_cast<f8 *>(d) = __builtin_convertvector(*reinterpret_cast<const t8 *>(s), f8);
        else
            for (int e = 0; at + e < n; ++e) d[e] = static_cast<float>(s[e]);
    } else {
        const float *s = static_cast<const float *>(p.src[i]) + at;
        T *d = static_cast<T *>(p.dst[i]) + at;
        if (at + 8 <= n)
            *reinterpret_cast<t8 *>(d) = __builtin_convertvector(*reinterpret_cast<const f8 *>(s), t8);
        else
            for (int e = 0; at + e < n; ++e) d[e] = static_cast<T>(s[e]);
    }
}

template <typename T>
hipError_t launch_convert(const ConvertParams &p, int n, bool widen, hipStream_t stream) {
    int64_t most = 0;
    for (int i = 0; i < n; ++i) most = p.count[i] > most ? p.count[i] : most;
    const int64_t grid = (most + 2047) / 2048;
    if (grid < 1) return hipSuccess;
    if (grid > 0x7fffffffLL) return hipErrorInvalidConfiguration;
    const dim3 g((unsigned)grid, (unsigned)n);
    return widen ? launch_kernel<convert_kernel<T, true>>(g, dim3(256), 0, stream, p)
                 : launch_kernel<convert_kernel<T, false>>(g, dim3(256), 0, stream, p);
}

}  // namespace fla
