// Lloyd iterations of the vector quantiser on the device: the assignment step is the encoder's scan with per-entry sums
// (encode_scan_kernel<..., ACCUMULATE>, vq_encode.hip), the update step is here, and nothing comes back to the host in
// between.  The scan's workgroups leave one row of partial results each - per entry the sums of the vectors assigned to it
// and their number, then the error -, and a second kernel adds the rows up in a fixed order and writes the next codebook.
//
// As device-wide tensor operations an iteration was 24 launches and ten passes over arrays of the weights' size (two
// scatter-adds of 244 us each on 2.1 M vectors: atomics on 256 entries): 840 us, and the host waited for every error.  With
// the sums kept in the LDS of the workgroups that assign (larger codebooks keep to the tensor operations)
// it is the assignment plus a few microseconds.
#include "vq_encode.h"

namespace vq {

namespace {

constexpr int kUpdateThreads = 512;
constexpr int kUpdateEntries = 4;  // entries per workgroup: runs of a cache line and a half per row (an iteration of 4096 x 4096: eight entries and 1024 threads 0.5 to 0.8 us longer)

// One slot (an element's sum, or the count) of kUpdateEntries entries per thread and slice of the rows; the slices are
// added up in order.  The last workgroup adds up the errors (`cb_out` null: the only one).  What bounds it is
// latency: a thread has all of a slice's loads, up to eight, on the way before it adds them (one behind the other, and the errors
// ahead of the first workgroup's entries, 4.8 us; so 4.6).
template <int VEC>
__global__ __launch_bounds__(kUpdateThreads) void lloyd_update_kernel(const float *__restrict__ partials, int rows_per_cb,
                                                                      const half_t *__restrict__ cb_in, half_t *__restrict__ cb_out,
                                                                      int entries, int n_codebooks, double *__restrict__ error)
{
    constexpr int kSlots = kUpdateEntries * (VEC + 1), kSlices = kUpdateThreads / kSlots;
    __shared__ float part[kSlices][kSlots];
    __shared__ double errors[kUpdateThreads / 64];
    const int64_t row = lloyd_row(entries, VEC);
    const int tid = threadIdx.x;
    const int wgs_per_cb = (entries + kUpdateEntries - 1) / kUpdateEntries;
    if (blockIdx.x == gridDim.x - 1) {
        double e = 0.0;
        for (int i = tid; i < rows_per_cb * n_codebooks; i += kUpdateThreads) e += (double)partials[(int64_t)i * row + row - 1];
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) e += __shfl_xor(e, d);
        if ((tid & 63) == 0) errors[tid >> 6] = e;
        __syncthreads();
        if (tid == 0) {
            double t = 0.0;
            for (int i = 0; i < kUpdateThreads / 64; i++) t += errors[i];
            *error = t;
        }
        return;
    }
    const int g = blockIdx.x / wgs_per_cb, e0 = (blockIdx.x % wgs_per_cb) * kUpdateEntries;
    const int slots = min(kUpdateEntries, entries - e0) * (VEC + 1);
    const int slice = tid / kSlots, slot = tid % kSlots;
    if (slice < kSlices && slot < slots) {
        const float *src = partials + (int64_t)g * rows_per_cb * row + e0 * (VEC + 1) + slot;
        float sum = 0.f;
        for (int r0 = slice; r0 < rows_per_cb; r0 += 8 * kSlices) {
            float v[8];
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const int r = r0 + i * kSlices;
                const float x = src[min(r, rows_per_cb - 1) * row];
                v[i] = r < rows_per_cb ? x : 0.f;
            }
#pragma unroll
            for (int i = 0; i < 8; i++) sum += v[i];
        }
        part[slice][slot] = sum;
    }
    __syncthreads();
    if (tid < slots) {
        float sum = 0.f;
        for (int i = 0; i < kSlices; i++) sum += part[i][tid];
        part[0][tid] = sum;
    }
    __syncthreads();
    if (tid < slots) {
        const int e = tid / (VEC + 1), t = tid % (VEC + 1);
        if (t < VEC) {
            const float count = part[0][e * (VEC + 1) + VEC];
            const int64_t at = ((int64_t)g * entries + e0 + e) * VEC + t;
            // an entry nothing was assigned to keeps its value
            cb_out[at] = count > 0.f ? (half_t)(part[0][tid] / count) : cb_in[at];
        }
    }
}

// initial entries: entry e of codebook g is vector pick[g][e] of the codebook's block
template <int VEC>
__global__ __launch_bounds__(256) void lloyd_pick_kernel(const half_t *__restrict__ w, const int32_t *__restrict__ pick,
                                                         half_t *__restrict__ cb, int64_t vectors_per_cb, int entries, int total)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= total) return;
    const int64_t v = (int64_t)(i / entries) * vectors_per_cb + pick[i];
#pragma unroll
    for (int t = 0; t < VEC; t++) cb[(int64_t)i * VEC + t] = w[v * VEC + t];
}

struct LloydLayout {
    size_t partials, books[2], bytes;
};
LloydLayout lloyd_layout(const ProblemB &p)
{
    auto up = [](size_t n) { return (n + 255) & ~(size_t)255; };
    LloydLayout l;
    l.partials = 0;
    l.books[0] = up((size_t)lloyd_assign_rows(p) * p.n_codebooks * lloyd_row(p.entries, p.vec) * 4);
    const size_t book = up((size_t)p.n_codebooks * p.entries * p.vec * 2);
    l.books[1] = l.books[0] + book;
    l.bytes = l.books[1] + book;
    return l;
}

template <int VEC>
hipError_t lloyd_typed(const half_t *w, const ProblemB &p, const int32_t *pick, int iters, void *codes_out, half_t *cb_out,
                       double *errors, uint8_t *workspace, hipStream_t s)
{
    const LloydLayout l = lloyd_layout(p);
    float *partials = reinterpret_cast<float *>(workspace + l.partials);
    half_t *books[2] = {reinterpret_cast<half_t *>(workspace + l.books[0]), reinterpret_cast<half_t *>(workspace + l.books[1])};
    const int rows = lloyd_assign_rows(p);
    const int picks = p.n_codebooks * p.entries;
    ProblemB q = p;
    half_t *book = iters == 0 ? cb_out : books[0];
    hipError_t e = launch_kernel(lloyd_pick_kernel<VEC>, dim3((picks + 255) / 256), dim3(256), 0, s, w, pick, book,
                       (int64_t)p.rows_per_cb * (p.K / VEC), p.entries, picks);
    for (int it = 0; it <= iters && e == hipSuccess; it++) {
        q.cb = book;
        e = launch_lloyd_assign(w, q, codes_out, partials, it < iters, s);
        if (e != hipSuccess) return e;
        half_t *next = it == iters ? nullptr : it + 1 == iters ? cb_out : books[(it + 1) & 1];
        const int wgs = (next ? p.n_codebooks * ((p.entries + kUpdateEntries - 1) / kUpdateEntries) : 0) + 1;
        e = launch_kernel(lloyd_update_kernel<VEC>, dim3(wgs), dim3(kUpdateThreads), 0, s, partials, rows, book, next, p.entries,
                           p.n_codebooks, errors + it);
        book = next;
    }
    return e;
}

}  // namespace

size_t lloyd_workspace_bytes(const ProblemB &p) { return lloyd_layout(p).bytes; }

hipError_t launch_lloyd(const half_t *w, const ProblemB &p, const int32_t *pick, int iters, void *codes_out, half_t *cb_out,
                        double *errors, void *workspace, hipStream_t s)
{
    uint8_t *ws = static_cast<uint8_t *>(workspace);
    switch (p.vec) {
    case 8: return lloyd_typed<8>(w, p, pick, iters, codes_out, cb_out, errors, ws, s);
    case 4: return lloyd_typed<4>(w, p, pick, iters, codes_out, cb_out, errors, ws, s);
    case 2: return lloyd_typed<2>(w, p, pick, iters, codes_out, cb_out, errors, ws, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace vq
