// Instantiations of the chunk-wise polynomial kernels (fla_poly_walk.h): bf16 only (the running sums are rounded to
// the storage type, and in fp16 its range would narrow what may be passed in).
#include "fla_dispatch.h"
#include "fla_poly_walk.h"

namespace fla {

hipError_t poly_totals(const PolyWalkParams &p, bool bwd, hipStream_t stream) { return launch_poly_totals<__bf16>(p, bwd, stream); }
hipError_t poly_walk(const PolyWalkParams &p, bool bwd, hipStream_t stream) { return launch_poly_walk<__bf16>(p, bwd, stream); }
hipError_t poly_scan(float *totals, int64_t BH, int n_seg, int reverse, hipStream_t stream) {
    return launch_poly_scan(totals, BH, n_seg, reverse, stream);
}

}  // namespace fla

#include "fla_trace_structs.h"  // (the trace build's descriptions of the parameter structs; empty otherwise)
