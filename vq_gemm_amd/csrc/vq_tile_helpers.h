// Device helpers shared by the tiled MFMA kernels (prefill kernels, plain tiled GEMM).
#pragma once

#include "vq_common.h"

namespace vq {

namespace {

// s_waitcnt for the vector-memory counter only (gfx9 encoding: vmcnt = simm16[15:14]:[3:0]).
template <int N>
__device__ __forceinline__ void wait_vmcnt()
{
    static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit counter");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// acc += a . b with the accumulator pinned to one AGPR tuple.  Left to itself the register
// allocator renames the 64 four-register accumulators from MFMA to MFMA and pays for it with
// copies at the loop edge and with spills.  The compiler cannot see into the statement, so the
// callers keep dependent MFMAs (same accumulator) far apart and pad before the accumulators are
// read back.
__device__ __forceinline__ void mfma_in_place(float4_t &acc, const half8_t &a, const half8_t &b)
{
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}

// 16-byte store of a result that this kernel does not read again: the non-temporal hint lets the
// write leave the L2 as it is issued instead of waiting for the write-back at the end of the kernel
// (all workgroups of a round finish at about the same time).
__device__ __forceinline__ void st_global_16_streaming(void *p, uint4_t v)
{
    __builtin_nontemporal_store(v, reinterpret_cast<uint4_t *>(p));
}

// Eight results of a row; `left`: columns up to the row's end.  Rows that are no multiple of 16 bytes (aligned false) begin
// anywhere: still one store, the memory takes any address, and only the row's last piece goes element by element.
__device__ __forceinline__ void store_eight(half_t *dst, uint4_t v, int left, bool aligned)
{
    if (left <= 0) return;
    if (aligned) {
        st_global_16_streaming(dst, v);
    } else if (left >= 8) {
        __builtin_memcpy(dst, &v, 16);
    } else {
        const half8_t h = __builtin_bit_cast(half8_t, v);
#pragma unroll
        for (int e = 0; e < 7; e++)
            if (e < left) dst[e] = h[e];
    }
}

// Holds the accumulators where they are (the AGPRs) up to here.  Called behind the wait for the last MFMAs: the compiler
// does not see what an inline-assembly MFMA is still writing, and where a loop's last pass is peeled off it would copy
// each accumulator out right behind its last MFMA.
template <int A, int B>
__device__ __forceinline__ void hold_accumulators(float4_t (&acc)[A][B])
{
#pragma unroll
    for (int a = 0; a < A; a++)
#pragma unroll
        for (int b = 0; b < B; b++) asm volatile("" : "+a"(acc[a][b]));
}

}  // namespace

}  // namespace vq
