// What the encoder (vq_encode.hip) and the Lloyd iterations around it (vq_lloyd.hip) share.
#pragma once

#include "vq_common.h"

namespace vq {

// eight waves per workgroup of the matrix-core scan (more per unit than two such, in smaller workgroups, gained nothing), or sixteen
constexpr int kScanThreads = 512, kScanWideThreads = 1024;

// floats of one workgroup's partial result of a Lloyd iteration: per entry `vec` sums and a count, then the error
__host__ __device__ inline int64_t lloyd_row(int entries, int vec) { return (int64_t)entries * (vec + 1) + 1; }

// An addition to a number in the LDS whose old value nobody asks for.
__device__ __forceinline__ void lds_add(double *p, double v)
{
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// The assignment step of a Lloyd iteration: codes, and one row of partial results per workgroup, lloyd_assign_rows(p) of them
// per codebook; `sums` false: the errors only.  Codebooks whose sums do not fit the LDS beside the table are not supported.
int lloyd_assign_rows(const ProblemB &p);
hipError_t launch_lloyd_assign(const half_t *w, const ProblemB &p, void *codes_out, float *partials, bool sums, hipStream_t s);

}  // namespace vq
