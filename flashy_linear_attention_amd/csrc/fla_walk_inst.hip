// Instantiations of the walk kernels (fla_chunk_walk.h) for one storage type (FLA_WALK_DTYPE: 0 bf16, 1 fp16) and one
// group of kernels (FLA_WALK_PART: 0 totals and forward walks, 1 backward walks and the normalised backward's first pass), padded head dims 32, 64 and 128
// (128: backward is a forward-direction walk for dQ and a kernel for dK and dV, or one reverse walk where
// a caller asks for it and forward handed its states over).
#include "fla_dispatch.h"

namespace fla {

#if FLA_WALK_DTYPE == 0
using WalkT = __bf16;
#else
using WalkT = _Float16;
#endif
#define FLA_WALK_FN(fn) FLA_WALK_NAME(fn, FLA_WALK_DTYPE)
#define FLA_WALK_DISPATCH(fn, ...) return D == 32 ? fn<WalkT, 32>(__VA_ARGS__) : fn<WalkT, 64>(__VA_ARGS__)
#define FLA_WALK_DISPATCH3(fn, ...)                     \
    if (D == 128) return fn<WalkT, 128>(__VA_ARGS__); \
    FLA_WALK_DISPATCH(fn, __VA_ARGS__)

#if FLA_WALK_PART == 1
hipError_t FLA_WALK_FN(walk_bwd)(int D, const WalkParams &p, hipStream_t stream) {
    if (D == 128) return hipErrorNotSupported;
    FLA_WALK_DISPATCH(launch_walk_bwd, p, stream);
}
hipError_t FLA_WALK_FN(walk_dkdv)(int D, const WalkParams &p, hipStream_t stream) {
    return D == 128 ? launch_walk_dkdv<WalkT, 128>(p, stream) : hipErrorNotSupported;
}
hipError_t FLA_WALK_FN(walk_bwd_rev)(int D, const WalkParams &p, hipStream_t stream) {
    return D == 128 ? launch_walk_bwd_rev<WalkT, 128>(p, stream) : hipErrorNotSupported;
}
hipError_t FLA_WALK_FN(walk_grad_totals)(int D, const WalkGradParams &p, hipStream_t stream) {
    FLA_WALK_DISPATCH3(launch_walk_grad_totals, p, stream);
}
hipError_t FLA_WALK_FN(walk_bwd_rev_wide)(const WalkParams &p, hipStream_t stream) {
    return launch_walk_bwd_rev_wide<WalkT>(p, stream);
}
#else
hipError_t FLA_WALK_FN(walk_totals)(int D, const WalkTotalsParams &p, hipStream_t stream) {
    FLA_WALK_DISPATCH3(launch_walk_totals, p, stream);
}
hipError_t FLA_WALK_FN(walk_fwd)(int D, const WalkParams &p, hipStream_t stream) {
    FLA_WALK_DISPATCH3(launch_walk_fwd, p, stream);
}
hipError_t FLA_WALK_FN(walk_fwd_wide)(const WalkParams &p, hipStream_t stream) { return launch_walk_fwd_wide<WalkT>(p, stream); }
hipError_t FLA_WALK_FN(walk_vec_sums)(const WalkVecParams &p, int64_t BH, hipStream_t stream) {
    return launch_walk_vec_sums<WalkT, 128>(p, BH, stream);
}
#if FLA_WALK_DTYPE == 0  // (fp32 throughout: once)
hipError_t walk_vec_scan(float *v, int64_t BH, int n_chunks, int D, hipStream_t stream) {
    return launch_walk_vec_scan(v, BH, n_chunks, D, stream);
}
hipError_t walk_scan(const float *totals, float *entry, int64_t BH, int n_seg, int D, int cols, int reverse,
                     hipStream_t stream, const float *totals_b, float *entry_b) {
    return launch_walk_scan(totals, entry, BH, n_seg, D, cols, reverse, stream, totals_b, entry_b);
}
#endif
#endif

}  // namespace fla

#include "fla_trace_structs.h"  // (the trace build's descriptions of the parameter structs; empty otherwise)
