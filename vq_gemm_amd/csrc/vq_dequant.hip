// Stand-alone dequantisation kernels: codes + codebook -> fp16 weights in HBM.
// Pure indexing and bit copies, so results are bit-exact by construction.  The kernels are
// bound by the write stream (16 B written per code byte read for vec = 8).
#include "vq_common.h"

namespace vq {

// ---- geometry B ------------------------------------------------------------------------
// One thread per code; consecutive threads take consecutive codes of a row, so each wave
// stores 64 * VEC * 2 contiguous bytes.  Codebooks stay in global memory: they are a few
// KB and every lookup after the first hits the L2.
template <int VEC, typename CodeT>
__global__ __launch_bounds__(256) void dequant_b_kernel(const CodeT *__restrict__ codes,
                                                        const half_t *__restrict__ cb,
                                                        half_t *__restrict__ w, int N, int J,
                                                        int entries, int rows_per_cb)
{
    typedef half_t vec_t __attribute__((ext_vector_type(VEC)));
    const int64_t total = (int64_t)N * J;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
        const int n = (int)(i / J);
        uint32_t c = codes[i];
        c = c < (uint32_t)entries ? c : (uint32_t)entries - 1;  // memory safety only
        const half_t *src = cb + ((int64_t)(n / rows_per_cb) * entries + c) * VEC;
        *reinterpret_cast<vec_t *>(w + i * VEC) = *reinterpret_cast<const vec_t *>(src);
    }
}

// The same for enough of them: a workgroup takes a run of one codebook's codes (they lie together, so that no code is divided by
// anything) and keeps the codebook in the LDS, where 64 codewords take 3 to 5 ns; out of the caches they are 64 lines of
// the L1.  A lane stores sixteen bytes, one to four codewords, the lanes of a wave side by side.
// What bounds it: the stores.  4096 x 4096, us (a fill of the weights 7.6): 8-vectors 9.3 -> 8.3, 4-vectors of 256 entries
// 12.0 -> 8.4, of 4096 13.9 -> 9.3, 2-vectors 16.6 -> 8.4.
constexpr int kDequantThreads = 1024, kDequantUnroll = 4;
constexpr size_t kDequantTable = 64 * 1024;

template <int VEC, typename CodeT>
__global__ __launch_bounds__(kDequantThreads) void dequant_b_table_kernel(const CodeT *__restrict__ codes, const half_t *__restrict__ cb,
                                                                          half_t *__restrict__ w, int64_t codes_per_cb, int entries, int wgs_per_cb)
{
    typedef half_t vec_t __attribute__((ext_vector_type(VEC)));
    constexpr int CPL = 8 / VEC, U = kDequantUnroll;   // codes of a lane and store
    typedef CodeT code_t __attribute__((ext_vector_type(CPL)));
    extern __shared__ __align__(16) uint8_t smem[];
    vec_t *table = reinterpret_cast<vec_t *>(smem);
    const int g = blockIdx.x / wgs_per_cb, part = blockIdx.x % wgs_per_cb;
    const vec_t *book = reinterpret_cast<const vec_t *>(cb + (int64_t)g * entries * VEC);
    for (int e = threadIdx.x; e < entries; e += kDequantThreads) table[e] = book[e];
    __syncthreads();
    const CodeT *src = codes + g * codes_per_cb;
    half_t *dst = w + g * codes_per_cb * VEC;
    auto entry = [&](uint32_t c) { return table[min(c, (uint32_t)entries - 1)]; };   // memory safety only
    constexpr int kStep = kDequantThreads * CPL;
    int64_t at = (int64_t)part * (kStep * U) + threadIdx.x * CPL;
    for (; at + (U - 1) * kStep + CPL <= codes_per_cb; at += (int64_t)wgs_per_cb * (kStep * U)) {
        code_t c[U];
#pragma unroll
        for (int u = 0; u < U; u++) __builtin_memcpy(&c[u], src + at + u * kStep, sizeof(code_t));
#pragma unroll
        for (int u = 0; u < U; u++) {
            vec_t v[CPL];
#pragma unroll
            for (int i = 0; i < CPL; i++) v[i] = entry(c[u][i]);
            __builtin_memcpy(dst + (at + u * kStep) * VEC, v, 16);
        }
    }
    for (int u = 0; u < U; u++)   // the run's end
        for (int64_t i = at + u * kStep; i < at + u * kStep + CPL && i < codes_per_cb; i++) *reinterpret_cast<vec_t *>(dst + i * VEC) = entry(src[i]);
}

// Any vector length (scalar copies).
template <typename CodeT>
__global__ __launch_bounds__(256) void dequant_b_anyvec_kernel(const CodeT *__restrict__ codes,
                                                               const half_t *__restrict__ cb,
                                                               half_t *__restrict__ w, int N, int J,
                                                               int vec, int entries, int rows_per_cb)
{
    const int64_t total = (int64_t)N * J;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
        const int n = (int)(i / J);
        uint32_t c = codes[i];
        c = c < (uint32_t)entries ? c : (uint32_t)entries - 1;
        const half_t *src = cb + ((int64_t)(n / rows_per_cb) * entries + c) * vec;
        for (int t = 0; t < vec; t++) w[i * vec + t] = src[t];
    }
}

template <typename CodeT>
static hipError_t dequant_b_typed(const ProblemB &p, half_t *w_out, hipStream_t s)
{
    const int J = p.K / p.vec;
    const int64_t total = (int64_t)p.N * J;
    if (total == 0) return hipSuccess;
    int64_t blocks = (total + 255) / 256;
    const int64_t cap = (int64_t)device_cu_count() * 32;
    if (blocks > cap) blocks = cap;
    const CodeT *codes = static_cast<const CodeT *>(p.codes);
    dim3 grid((unsigned)blocks), block(256);
    // Vector copies need codeword-aligned source and destination; otherwise copy scalars.
    const bool aligned = (((uintptr_t)w_out | (uintptr_t)p.cb) % (uintptr_t)(p.vec * 2)) == 0;
    // a table for every workgroup, where a compute unit, and a codebook's rows, come to four times as much or more and there are
    // workgroups for three units in eight (4-vectors: 1024 x 3072, 96 of them, 4.4 us -> 4.0; 2320 x 576, 42, 3.3 -> 3.7)
    const size_t table = (size_t)p.entries * p.vec * 2;
    const int64_t per_cb = (int64_t)p.rows_per_cb * J, step = (int64_t)kDequantThreads * kDequantUnroll * 8 / p.vec, have = (per_cb + step - 1) / step;
    if (aligned && table <= kDequantTable && total * p.vec * 2 >= 4 * (int64_t)table * device_cu_count() && per_cb >= 4 * p.entries &&
        have * p.n_codebooks * 8 >= 3 * device_cu_count()) {
        const int64_t want = (2 * device_cu_count() + p.n_codebooks - 1) / p.n_codebooks;
        const int wgs = (int)(want < have ? want : have);
        auto launch = [&](auto kern) { return launch_kernel(kern, dim3((unsigned)(wgs * p.n_codebooks)), dim3(kDequantThreads), table, s, codes, p.cb, w_out, per_cb, p.entries, wgs); };
        switch (p.vec) {
        case 2: return launch(dequant_b_table_kernel<2, CodeT>);
        case 4: return launch(dequant_b_table_kernel<4, CodeT>);
        case 8: return launch(dequant_b_table_kernel<8, CodeT>);
        default: break;
        }
    }
    switch (aligned ? p.vec : 0) {
    case 2: return launch_kernel((dequant_b_kernel<2, CodeT>), grid, block, 0, s, codes, p.cb, w_out, p.N, J, p.entries, p.rows_per_cb);
    case 4: return launch_kernel((dequant_b_kernel<4, CodeT>), grid, block, 0, s, codes, p.cb, w_out, p.N, J, p.entries, p.rows_per_cb);
    case 8: return launch_kernel((dequant_b_kernel<8, CodeT>), grid, block, 0, s, codes, p.cb, w_out, p.N, J, p.entries, p.rows_per_cb);
    default: return launch_kernel((dequant_b_anyvec_kernel<CodeT>), grid, block, 0, s, codes, p.cb, w_out, p.N, J, p.vec, p.entries, p.rows_per_cb);
    }
}

hipError_t launch_dequant_b(const ProblemB &p, half_t *w_out, hipStream_t s)
{
    return p.code_bits == 8 ? dequant_b_typed<uint8_t>(p, w_out, s) : dequant_b_typed<uint16_t>(p, w_out, s);
}

// ---- geometry A ------------------------------------------------------------------------
// W_dec[k, 2n + r] = cb[n/4][w[k,n]][r]: one thread per code writes one 4-byte codeword;
// a wave writes 256 contiguous bytes of a W_dec row.
__global__ __launch_bounds__(256) void dequant_a_kernel(const uint8_t *__restrict__ w,
                                                        const half_t *__restrict__ cb,
                                                        half_t *__restrict__ out, int K, int Nc)
{
    const int64_t total = (int64_t)K * Nc;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
        const int n = (int)(i % Nc);
        const uint32_t c = w[i];
        const half_t *src = cb + ((int64_t)(n >> 2) * 256 + c) * 2;
        *reinterpret_cast<half2_t *>(out + i * 2) = *reinterpret_cast<const half2_t *>(src);
    }
}

// The same for enough of them: a workgroup keeps the codebooks of 64 code columns in the LDS and goes down its rows of them; a lane
// takes the four codes of a codebook and stores sixteen bytes.  (One code at a time, each divided by Nc and looked up
// through the L1: K = 4096, Nc = 4096 48.2 us -> 17.8, Nc = 640 12.0 -> 6.1.)
constexpr int kDequantACols = 64;

__global__ __launch_bounds__(kDequantThreads) void dequant_a_table_kernel(const uint8_t *__restrict__ w, const half_t *__restrict__ cb,
                                                                          half_t *__restrict__ out, int K, int Nc, int col_blocks, int rows_per_wg)
{
    __shared__ uint32_t table[kDequantACols / 4 * 256];
    constexpr int kLanes = kDequantACols / 4, kRows = kDequantThreads / kLanes;   // lanes a row, rows a pass
    const int block = blockIdx.x % col_blocks, part = blockIdx.x / col_blocks;
    const int books = min(kLanes, (Nc - block * kDequantACols) / 4);
    const uint32_t *src = reinterpret_cast<const uint32_t *>(cb) + (int64_t)block * kLanes * 256;
    for (int i = threadIdx.x; i < books * 256; i += kDequantThreads) table[i] = src[i];
    __syncthreads();
    const int book = threadIdx.x % kLanes;
    if (book >= books) return;
    const int first = part * rows_per_wg, last = min(first + rows_per_wg, K);
    const int col = block * kDequantACols + book * 4;
#pragma unroll 4
    for (int k = first + threadIdx.x / kLanes; k < last; k += kRows) {
        uint32_t c, v[4];
        __builtin_memcpy(&c, w + (int64_t)k * Nc + col, 4);
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = table[book * 256 + ((c >> (8 * i)) & 0xffu)];
        __builtin_memcpy(out + ((int64_t)k * Nc + col) * 2, v, 16);
    }
}

hipError_t launch_dequant_a(const ProblemA &p, half_t *w_out, hipStream_t s)
{
    const int64_t total = (int64_t)p.K * p.Nc;
    if (total == 0) return hipSuccess;
    const int64_t table = kDequantACols / 4 * 1024;
    if (((uintptr_t)p.cb & 3) == 0 && ((uintptr_t)w_out & 3) == 0 && total * 4 >= table * device_cu_count()) {
        const int col_blocks = (p.Nc + kDequantACols - 1) / kDequantACols, parts = (2 * device_cu_count() + col_blocks - 1) / col_blocks;
        const int rows = (p.K + parts - 1) / parts;
        return launch_kernel(dequant_a_table_kernel, dim3((unsigned)(col_blocks * ((p.K + rows - 1) / rows))), dim3(kDequantThreads), 0, s, p.w, p.cb, w_out, p.K, p.Nc,
                             col_blocks, rows);
    }
    int64_t blocks = (total + 255) / 256;
    const int64_t cap = (int64_t)device_cu_count() * 32;
    if (blocks > cap) blocks = cap;
    return launch_kernel(dequant_a_kernel, dim3((unsigned)blocks), dim3(256), 0, s, p.w, p.cb, w_out, p.K, p.Nc);
}

}  // namespace vq
