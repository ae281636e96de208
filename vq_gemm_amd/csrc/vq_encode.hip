// Nearest-codeword encoder, geometry B: codes[n, j] = the entry of the row's codebook closest to
// W[n, j*vec .. j*vec+vec) in squared Euclidean distance.  This is the assignment step of a
// vector quantiser, the step before the GEMM path (the reference only ever multiplies random codes,
// bench.py:84).
//
// The arithmetic is fixed so that the result is reproducible bit for bit: operands are widened to
// fp32, the distance is accumulated element by element in vector order with a fused multiply-add
// (acc = fma(d, d, acc), d = w - c), entry 0 starts as the best and a later entry replaces it only
// when its distance is strictly smaller (ties keep the lowest index; a NaN distance never wins).
//
// The rows of one codebook are contiguous in W and in the codes, so a codebook's block is walked as
// a flat array of vectors.  Two kernels compute the rule:
//
//   * encode_scan_kernel, for tables that fit the LDS whole: the matrix cores score every vector against every
//     entry (|c|^2 / 2 - w.c orders the entries as the distance does), the vector unit only keeps the best and the
//     second best of groups of eight scores, and the entries of the best group are scored once more one by one.  Where
//     another entry comes within what the rounding of a score can hide, the rule itself decides, on all entries.
//   * encode_b_kernel, for the rest: the rule on every entry.  A workgroup keeps a chunk of the codebook in the LDS as
//     fp32; all lanes read the same entry at a time (a broadcast), each thread scores four vectors against it.
#include "vq_encode.h"

#include <type_traits>

namespace vq {

namespace {

constexpr int kEncThreads = 256;
constexpr int kEncPerThread = 4;                 // vectors per thread
constexpr int kEncChunkFloats = 16384;           // fp32 codebook chunk in the LDS: 64 KB

template <int VEC, typename CodeT>
__global__ __launch_bounds__(kEncThreads) void encode_b_kernel(const half_t *__restrict__ w,
                                                               const half_t *__restrict__ cb,
                                                               CodeT *__restrict__ codes, int64_t vectors_per_cb,
                                                               int entries, int wgs_per_cb)
{
    __shared__ __align__(16) float table[kEncChunkFloats];
    constexpr int kChunkEntries = kEncChunkFloats / VEC;
    const int g = blockIdx.x / wgs_per_cb, part = blockIdx.x % wgs_per_cb;
    const half_t *wg_w = w + (int64_t)g * vectors_per_cb * VEC;
    CodeT *wg_codes = codes + (int64_t)g * vectors_per_cb;
    const half_t *book = cb + (int64_t)g * entries * VEC;

    for (int64_t base = (int64_t)part * kEncThreads * kEncPerThread; base < vectors_per_cb;
         base += (int64_t)wgs_per_cb * kEncThreads * kEncPerThread) {
        float v[kEncPerThread][VEC];
        float best[kEncPerThread];
        uint32_t arg[kEncPerThread];
#pragma unroll
        for (int u = 0; u < kEncPerThread; u++) {
            const int64_t idx = base + u * kEncThreads + threadIdx.x;
            const int64_t src = idx < vectors_per_cb ? idx : vectors_per_cb - 1;
#pragma unroll
            for (int t = 0; t < VEC; t++) v[u][t] = (float)wg_w[src * VEC + t];
            best[u] = 0.f;
            arg[u] = 0;
        }
        for (int e0 = 0; e0 < entries; e0 += kChunkEntries) {
            const int n_e = entries - e0 < kChunkEntries ? entries - e0 : kChunkEntries;
            __syncthreads();  // the previous chunk has been read by every thread
            for (int i = threadIdx.x; i < n_e * VEC; i += kEncThreads) table[i] = (float)book[(int64_t)e0 * VEC + i];
            __syncthreads();
            for (int e = 0; e < n_e; e++) {
                float c[VEC];
#pragma unroll
                for (int t = 0; t < VEC; t++) c[t] = table[e * VEC + t];
#pragma unroll
                for (int u = 0; u < kEncPerThread; u++) {
                    float acc = 0.f;
#pragma unroll
                    for (int t = 0; t < VEC; t++) {
                        const float d = v[u][t] - c[t];
                        acc = __builtin_fmaf(d, d, acc);
                    }
                    // entry 0 is taken as it is; later entries must be strictly closer
                    const bool take = (e0 + e == 0) || acc < best[u];
                    best[u] = take ? acc : best[u];
                    arg[u] = take ? (uint32_t)(e0 + e) : arg[u];
                }
            }
        }
#pragma unroll
        for (int u = 0; u < kEncPerThread; u++) {
            const int64_t idx = base + u * kEncThreads + threadIdx.x;
            if (idx < vectors_per_cb) wg_codes[idx] = (CodeT)arg[u];
        }
    }
}


// ---- matrix-core scan -------------------------------------------------------------------------
// What bounds it: the vector unit.  The rule costs 2 * vec + 2 vector instructions per vector and entry; a score costs
// the matrix pipe 1/32 of a cycle (v_mfma_f32_32x32x8_f16: 32 entries by 32 vectors, vec <= 8 of its k in use) and the
// vector unit one instruction: of a group of eight scores four to fold them to their minimum and four to keep the best
// two groups (0.75 in groups of sixteen).  4096 x 4096, 8-vectors, 256 entries: 230 -> 32 us.
//
// A wave takes 128 vectors as four batches of 32 (64 as two, where there are too few for a workgroup on every other unit), so that an entry tile read from the LDS (its halves and its
// half norms) meets four MFMAs.  A lane of the result holds 16 scores of one vector - two groups of eight entries, or one -, and
// the lane 32 further on the other 16.
// Scores per group: a larger one costs the scan less and the rule more; they meet at about this many entries.
constexpr int kScanWideGroupEntries = 768;

// bytes of the scan's table: whole tiles of 32 entries, an entry left out after every 256 bytes, in whole 16-byte steps
__host__ __device__ inline int scan_table_bytes(int entries, int vec)
{
    const int padded = (entries + 31) / 32 * 32;
    return ((padded + padded / (128 / vec)) * vec * 2 + 15) & ~15;
}

// Exact distance by the rule, elements in vector order; `c_neg` are the entry's halves with their signs flipped.
template <int DW>
__device__ __forceinline__ float rule_distance(const uint32_t (&w)[DW], const uint32_t (&c_neg)[DW])
{
    float acc = 0.f;
#pragma unroll
    for (int i = 0; i < DW; i++) {
        const half2_t a = __builtin_bit_cast(half2_t, w[i]), b = __builtin_bit_cast(half2_t, c_neg[i]);
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const float d = (float)a[t] + (float)b[t];
            acc = __builtin_fmaf(d, d, acc);
        }
    }
    return acc;
}

__device__ __forceinline__ float dot2(uint32_t a, uint32_t b, float c)
{
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(half2_t, a), __builtin_bit_cast(half2_t, b), c, false);
}

// two halves with both zeros as one (-0 + 0 is 0)
__device__ __forceinline__ uint32_t one_zero(uint32_t v) { return __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, v) + half2_t{}); }

template <int DW>
__device__ __forceinline__ void read_entry(const uint32_t *table, int e, uint32_t (&c)[DW])
{
    typedef uint32_t entry_t __attribute__((ext_vector_type(DW)));
    if constexpr (DW == 1) {
        c[0] = table[e];
    } else {
        const entry_t v = *reinterpret_cast<const entry_t *>(table + e * DW);
#pragma unroll
        for (int i = 0; i < DW; i++) c[i] = v[i];
    }
}

// Of two values per lane: .lo holds a of the lower 32 lanes followed by b of the lower lanes, .hi a of the upper lanes followed
// by b of the upper lanes.
struct HalfWaves {
    uint32_t lo, hi;
};
__device__ __forceinline__ HalfWaves swap_half_waves(uint32_t a, uint32_t b)
{
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    return HalfWaves{r[0], r[1]};
}

// LDS: entries padded to whole tiles of 32: halves with flipped signs, then |c|^2 / 2 (infinity behind the last entry),
// then with SUMS the sums of the vectors assigned to each entry and their number, [entry][VEC + 1], then n_buckets words.
//
// SUMS (a Lloyd iteration): every vector is added to its entry's sums, its distance to the workgroup's error, and
// both leave as the workgroup's row of `partials`: entries * (VEC + 1) sums and counts, then the error.  The sums are kept in
// double: an LDS addition of doubles takes a fifth of the time of one of floats on this device (2.1 M vectors of 8 elements:
// 19 against 99 us), and is exact for weights of any usual range.  kErrorOnly: the last assignment, whose sums nothing reads (44.2 -> 38.7 us;
// as a flag of the one kernel it cost every assignment half a microsecond).
enum ScanKeeps { kCodesOnly, kErrorOnly, kSums };

template <int VEC, typename CodeT, int GROUP, ScanKeeps KEEPS, int kScanBatches>
__global__ __launch_bounds__(kScanThreads) void encode_scan_kernel(const half_t *__restrict__ w, const half_t *__restrict__ cb,
                                                                   CodeT *__restrict__ codes, int64_t vectors_per_cb, int entries,
                                                                   int wgs_per_cb, float *__restrict__ partials, int bucket_off,
                                                                   int n_buckets)
{
    extern __shared__ __align__(16) uint8_t smem[];
    __shared__ float reduce[kScanThreads / 64];
    constexpr bool ACCUMULATE = KEEPS != kCodesOnly, SUMS = KEEPS == kSums;
    constexpr int DW = VEC / 2;                       // dwords of a vector
    constexpr int kScanVectors = 32 * kScanBatches;   // of a wave
    // An entry's place in the table: one is left out after every 256 bytes of them, or the entries of all best groups, which
    // start at multiples of sixteen entries, would lie in the same few banks.
    constexpr int kRow = 128 / VEC;
    auto at = [](int e) { return e + e / kRow; };
    constexpr int kGroups = 16 / GROUP, kQuads = GROUP / 4;  // groups of a lane's scores; runs of four entries in a group
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, h = lane >> 5;         // vector of a batch, and which half of K (and of the rows) the lane holds
    const int n_tiles = (entries + 31) / 32;
    uint32_t *table = reinterpret_cast<uint32_t *>(smem);                         // [n_tiles * 32][DW]
    float *norms = reinterpret_cast<float *>(smem + scan_table_bytes(entries, VEC));
    double *sums = reinterpret_cast<double *>(norms + n_tiles * 32);
    uint32_t *bucket = reinterpret_cast<uint32_t *>(smem + bucket_off);
    const int g = blockIdx.x / wgs_per_cb, part = blockIdx.x % wgs_per_cb;
    const half_t *wg_w = w + (int64_t)g * vectors_per_cb * VEC;
    CodeT *wg_codes = codes + (int64_t)g * vectors_per_cb;

    // table, half norms, whether all of them are finite (else every vector of the codebook is decided by the rule)
    bool book_finite;
    {
        // An entry that equals an earlier one is never chosen, but beside it no vector would be clear below, and a vector by the rule
        // takes as long as twenty others: it gets an infinite norm.  The entries' hashes deal them out to buckets, and an entry looks
        // at the first one in its bucket.  (What meets another entry there, and so stays, costs time, not the result.)  A codebook
        // half of whose entries equal the other half, 4096 x 4096 8-vectors: 749 -> 125 us, two equal ones and half of the weights
        // that value 435 -> 40; none equal 41.3 and 41.2.
        auto bucket_of = [&](const uint32_t (&c)[DW]) {
            uint32_t h = 0;
#pragma unroll
            for (int i = 0; i < DW; i++) {
                const uint32_t v = one_zero(c[i]);
                h ^= i ? v << (7 * i) | v >> (32 - 7 * i) : v;
            }
            return (int)__umulhi(h * 0x9e3779b1u, (uint32_t)n_buckets);
        };
        float largest = 0.f;
        const uint32_t *book = reinterpret_cast<const uint32_t *>(cb + (int64_t)g * entries * VEC);
        uint32_t own[DW];   // the thread's first entry, on its way while the buckets are cleared
        auto load = [&](int e) {
#pragma unroll
            for (int i = 0; i < DW; i++) own[i] = book[(int64_t)min(e, entries - 1) * DW + i];
#pragma unroll
            for (int i = 0; i < DW; i++) own[i] = (e < entries ? own[i] : 0u) ^ 0x80008000u;
        };
        load(tid);
        for (int i = tid; i < n_buckets; i += kScanThreads) bucket[i] = ~0u;
        if (n_buckets) __syncthreads();
        for (int e = tid; e < n_tiles * 32; e += kScanThreads) {
            if (e != tid) load(e);
            float n2 = 0.f;
            uint32_t c[DW];
#pragma unroll
            for (int i = 0; i < DW; i++) {
                const half2_t f = __builtin_bit_cast(half2_t, own[i]);
                n2 = __builtin_fmaf((float)f[0], (float)f[0], n2);
                n2 = __builtin_fmaf((float)f[1], (float)f[1], n2);
                table[at(e) * DW + i] = c[i] = own[i];
            }
            norms[e] = e < entries ? 0.5f * n2 : __builtin_inff();
            largest = n2 < __builtin_inff() ? fmaxf(largest, n2) : __builtin_inff();
            if (n_buckets && e < entries) atomicMin(&bucket[bucket_of(c)], (uint32_t)e);
        }
        if constexpr (SUMS)
            for (int i = tid; i < entries * (VEC + 1); i += kScanThreads) sums[i] = 0.0;
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) largest = fmaxf(largest, __shfl_xor(largest, d));
        if (lane == 0) reduce[wave] = largest;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kScanThreads / 64; i++) largest = fmaxf(largest, reduce[i]);
        book_finite = largest < __builtin_inff();
        if (n_buckets) {
            for (int e = tid; e < entries; e += kScanThreads) {
                uint32_t c[DW], other[DW];
                read_entry<DW>(table, at(e), c);
                const int first = (int)bucket[bucket_of(c)];
                read_entry<DW>(table, at(first), other);
                uint32_t differ = first < e ? 0u : 1u;
#pragma unroll
                for (int i = 0; i < DW; i++) differ |= one_zero(c[i]) ^ one_zero(other[i]);
                if (!differ) norms[e] = __builtin_inff();
            }
            __syncthreads();
        }
    }

    // Infinities the compiler takes for any numbers: a minimum that starts from one folds two scores per instruction, and
    // the median with the other is a minimum, without an instruction to quiet what might be a signalling NaN.
    float above = __builtin_inff(), below = -__builtin_inff();
    asm volatile("" : "+v"(above), "+v"(below));
    float error = 0.f;
    const int64_t step = (int64_t)wgs_per_cb * (kScanThreads / 64) * kScanVectors;
    for (int64_t base = ((int64_t)part * (kScanThreads / 64) + wave) * kScanVectors; base < vectors_per_cb; base += step) {
        // the vectors: lane (col, h) holds elements 4h .. 4h+3 of its vector in each batch (nothing where vec ends before)
        half4_t b[kScanBatches];
        float m1[kScanBatches], m2[kScanBatches];
        int best[kScanBatches];
#pragma unroll
        for (int u = 0; u < kScanBatches; u++) {
            const int64_t idx = min(base + u * 32 + col, vectors_per_cb - 1);
            const half_t *src = wg_w + idx * VEC + (VEC == 8 ? 4 * h : 0);
            b[u] = half4_t{};
            if (VEC == 8 || h == 0) {
                if constexpr (VEC == 2) {
                    const half2_t v = *reinterpret_cast<const half2_t *>(src);
                    b[u] = half4_t{v[0], v[1], (half_t)0.f, (half_t)0.f};
                } else {
                    b[u] = *reinterpret_cast<const half4_t *>(src);
                }
            }
            m1[u] = m2[u] = __builtin_inff();
            best[u] = 0;
        }
        for (int t = 0; t < n_tiles; t++) {
            half4_t a = {};
            {
                const uint32_t *src = table + at(t * 32 + col) * DW + (VEC == 8 ? 2 * h : 0);
                if (VEC == 8 || h == 0) {
                    if constexpr (VEC == 2) {
                        const half2_t v = __builtin_bit_cast(half2_t, src[0]);
                        a = half4_t{v[0], v[1], (half_t)0.f, (half_t)0.f};
                    } else {
                        a = *reinterpret_cast<const half4_t *>(src);
                    }
                }
            }
            float16_t c;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const float4_t v = *reinterpret_cast<const float4_t *>(norms + t * 32 + 8 * q + 4 * h);
#pragma unroll
                for (int i = 0; i < 4; i++) c[4 * q + i] = v[i];
            }
#pragma unroll
            for (int u = 0; u < kScanBatches; u++) {
                const float16_t s = __builtin_amdgcn_mfma_f32_32x32x8f16(a, b[u], c, 0, 0, 0);
#pragma unroll
                for (int gr = 0; gr < kGroups; gr++) {
                    float x = above;
#pragma unroll
                    for (int i = 0; i < GROUP; i++) x = fminf(x, s[gr * GROUP + i]);
                    best[u] = x < m1[u] ? kGroups * t + gr : best[u];
                    m2[u] = __builtin_amdgcn_fmed3f(m1[u], m2[u], x);
                    m1[u] = __builtin_amdgcn_fmed3f(m1[u], x, below);
                }
            }
        }
        // Two batches at a time, a vector per lane: lane l takes vector l of the pair.  One swap of half waves brings a lane
        // what its vector's two lanes hold: .lo of the rows (and elements) of half 0, .hi of half 1.
#pragma unroll
        for (int u = 0; u < kScanBatches; u += 2) {
            uint32_t full[DW];  // the vector, in element order
            {
                const uint2_t v0 = __builtin_bit_cast(uint2_t, b[u]), v1 = __builtin_bit_cast(uint2_t, b[u + 1]);
                const HalfWaves p0 = swap_half_waves(v0[0], v1[0]);
                full[0] = p0.lo;
                if constexpr (VEC >= 4) {
                    const HalfWaves p1 = swap_half_waves(v0[1], v1[1]);
                    full[1] = p1.lo;
                    if constexpr (VEC == 8) {
                        full[2] = p0.hi;
                        full[3] = p1.hi;
                    }
                }
            }
            float w2 = 0.f;
#pragma unroll
            for (int i = 0; i < DW; i++) w2 = dot2(full[i], full[i], w2);
            const HalfWaves s1 = swap_half_waves(__builtin_bit_cast(uint32_t, m1[u]), __builtin_bit_cast(uint32_t, m1[u + 1]));
            const HalfWaves s2 = swap_half_waves(__builtin_bit_cast(uint32_t, m2[u]), __builtin_bit_cast(uint32_t, m2[u + 1]));
            const HalfWaves sb = swap_half_waves((uint32_t)best[u], (uint32_t)best[u + 1]);
            const float lo1 = __builtin_bit_cast(float, s1.lo), hi1 = __builtin_bit_cast(float, s1.hi);
            const bool lower = !(hi1 < lo1);  // the best group is among the rows of half 0
            const int group = lower ? (int)sb.lo : (int)sb.hi;
            const float next = fminf(fmaxf(lo1, hi1), fminf(__builtin_bit_cast(float, s2.lo), __builtin_bit_cast(float, s2.hi)));
            // the scores of the group's entries once more, now one by one
            const int e0 = (group / kGroups) * 32 + (group % kGroups) * 16 + (lower ? 0 : 4);
            float first = above, second = above;
            int e_best = 0;
#pragma unroll
            for (int q = 0; q < kQuads; q++) {
                const float4_t norm = *reinterpret_cast<const float4_t *>(norms + e0 + 8 * q);
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    uint32_t c[DW];
                    read_entry<DW>(table, at(e0 + 8 * q) + i, c);
                    float x = norm[i];
#pragma unroll
                    for (int k = 0; k < DW; k++) x = dot2(c[k], full[k], x);
                    e_best = x < first ? e0 + 8 * q + i : e_best;
                    second = __builtin_amdgcn_fmed3f(first, second, x);
                    first = __builtin_amdgcn_fmed3f(first, x, below);
                }
            }
            // What rounding can hide.  With u = 2^-24: a score (nine exact terms, summed) is off by at most 24 u (|w||c| + |c|^2 / 2)
            // <= 24 u (|w|^2 / 2 + |c|^2), the rule's distance by 10 u of itself.  Whatever entry the rule would choose is no
            // further from w than the first one here, so that entry and the first both have |c| <= |w| + sqrt(D) with
            // D = |w|^2 + 2 first, |c|^2 <= 4 (|w|^2 + first).  Two scores and two halved distances: at most
            // u (228 |w|^2 + 216 first) < 2^-16 (|w|^2 + first).  (Not clear either where anything is not finite.)
            const float hidden = 1.52587890625e-5f * (w2 + first);
            const bool clear = book_finite && fminf(next, second) - first > hidden;
            // vectors that this does not decide: the rule on every entry, all lanes on one vector
            for (uint64_t todo = __ballot(!clear); todo; todo &= todo - 1) {
                const int v = __builtin_ctzll(todo);
                uint32_t one[DW], c[DW];
#pragma unroll
                for (int i = 0; i < DW; i++) one[i] = __builtin_amdgcn_readlane(full[i], v);
                read_entry<DW>(table, 0, c);
                float d0 = rule_distance<DW>(one, c);  // entry 0 is taken as it is
                int e_min = 0;
                for (int e = lane; e < entries; e += 64) {
                    read_entry<DW>(table, at(e), c);
                    const float d = rule_distance<DW>(one, c);
                    const bool take = d < d0;
                    d0 = take ? d : d0;
                    e_min = take ? e : e_min;
                }
#pragma unroll
                for (int s = 32; s >= 1; s >>= 1) {
                    const float od = __shfl_xor(d0, s);
                    const int oe = __shfl_xor(e_min, s);
                    const bool other = od < d0 || (od == d0 && oe < e_min);
                    d0 = other ? od : d0;
                    e_min = other ? oe : e_min;
                }
                e_best = lane == v ? e_min : e_best;
            }
            const int64_t idx = base + u * 32 + lane;
            if (idx < vectors_per_cb) {
                wg_codes[idx] = (CodeT)e_best;
                if constexpr (ACCUMULATE) {
                    uint32_t c[DW];
                    read_entry<DW>(table, at(e_best), c);
                    error += rule_distance<DW>(full, c);
                    if constexpr (SUMS) {
                        double *sum = sums + e_best * (VEC + 1);
#pragma unroll
                        for (int i = 0; i < DW; i++) {
                            const half2_t v = __builtin_bit_cast(half2_t, full[i]);
                            lds_add(sum + 2 * i, (double)(float)v[0]);
                            lds_add(sum + 2 * i + 1, (double)(float)v[1]);
                        }
                        lds_add(sum + VEC, 1.0);
                    }
                }
            }
        }
    }
    if constexpr (ACCUMULATE) {
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) error += __shfl_xor(error, d);
        __syncthreads();  // every sum is in, and every thread has read `reduce`
        if (lane == 0) reduce[wave] = error;
        __syncthreads();
        float *row = partials + (int64_t)blockIdx.x * lloyd_row(entries, VEC);
        if constexpr (SUMS)
            for (int i = tid; i < entries * (VEC + 1); i += kScanThreads) row[i] = (float)sums[i];
        if (tid == 0) {
            float e = 0.f;
            for (int i = 0; i < kScanThreads / 64; i++) e += reduce[i];
            row[entries * (VEC + 1)] = e;
        }
    }
}

size_t scan_lds_bytes(const ProblemB &p, bool accumulate)
{
    const size_t padded = ((size_t)p.entries + 31) / 32 * 32;
    return scan_table_bytes(p.entries, p.vec) + padded * 4 + (accumulate ? (size_t)p.entries * (p.vec + 1) * 8 : 0);
}

constexpr size_t kScanLdsTwoPerUnit = 72 * 1024, kScanLds = 128 * 1024;

// Buckets for finding equal entries: four per entry where the LDS has room that neither keeps a second workgroup off the unit nor the
// codebook off this kernel; none where not even one per two entries fits.
int scan_buckets(const ProblemB &p, bool accumulate)
{
    const size_t bytes = scan_lds_bytes(p, accumulate), room = ((bytes <= kScanLdsTwoPerUnit ? kScanLdsTwoPerUnit : kScanLds) - bytes) / 4;
    const size_t want = 4 * (size_t)p.entries;
    return room >= want ? (int)want : 2 * room >= (size_t)p.entries ? (int)room : 0;
}

// Batches of a wave and workgroups per codebook: as many as are resident together (two of eight waves per unit while the LDS
// allows), none without work.
struct ScanPlan {
    int batches, wgs_per_cb;
};
ScanPlan scan_plan(const ProblemB &p, bool accumulate)
{
    const int64_t vectors = (int64_t)p.rows_per_cb * (p.K / p.vec);
    const int per_cu = scan_lds_bytes(p, accumulate) <= kScanLdsTwoPerUnit ? 2 : 1;
    const int64_t want = ((int64_t)device_cu_count() * per_cu + p.n_codebooks - 1) / p.n_codebooks;
    auto have = [&](int batches) { return (vectors + kScanThreads / 2 * batches - 1) / (kScanThreads / 2 * batches); };
    const int batches = have(4) * p.n_codebooks * 2 <= device_cu_count() ? 2 : 4;
    return {batches, (int)(want < have(batches) ? want : have(batches))};
}

bool scan_supports(const half_t *w, const ProblemB &p, bool accumulate)
{
    const uintptr_t align = p.vec * 2 < 8 ? p.vec * 2 : 8;
    return ((uintptr_t)w & (align - 1)) == 0 && ((uintptr_t)p.cb & 3) == 0 && scan_lds_bytes(p, accumulate) <= kScanLds;
}

template <int VEC, typename CodeT, ScanKeeps KEEPS>
hipError_t launch_scan(const half_t *w, const ProblemB &p, void *codes_out, float *partials, hipStream_t s)
{
    const int64_t vectors_per_cb = (int64_t)p.rows_per_cb * (p.K / VEC);
    if (vectors_per_cb == 0) return hipSuccess;
    constexpr bool accumulate = KEEPS != kCodesOnly;   // (the last assignment in the same workgroups as the others)
    const ScanPlan plan = scan_plan(p, accumulate);
    const size_t smem = scan_lds_bytes(p, accumulate);
    const int buckets = scan_buckets(p, accumulate);
    const bool narrow = p.entries < kScanWideGroupEntries;
    auto kern = plan.batches == 4 ? (narrow ? encode_scan_kernel<VEC, CodeT, 8, KEEPS, 4> : encode_scan_kernel<VEC, CodeT, 16, KEEPS, 4>)
                                  : (narrow ? encode_scan_kernel<VEC, CodeT, 8, KEEPS, 2> : encode_scan_kernel<VEC, CodeT, 16, KEEPS, 2>);
    return launch_kernel(kern, dim3((unsigned)(plan.wgs_per_cb * p.n_codebooks)), dim3(kScanThreads), smem + 4 * (size_t)buckets, s, w, p.cb,
                       static_cast<CodeT *>(codes_out), vectors_per_cb, p.entries, plan.wgs_per_cb, partials, (int)smem, buckets);
}

template <int VEC, typename CodeT>
hipError_t encode_b_typed(const half_t *w, const ProblemB &p, void *codes_out, hipStream_t s)
{
    if (scan_supports(w, p, false)) return launch_scan<VEC, CodeT, kCodesOnly>(w, p, codes_out, nullptr, s);
    const int64_t vectors_per_cb = (int64_t)p.rows_per_cb * (p.K / VEC);
    if (vectors_per_cb == 0) return hipSuccess;
    // enough workgroups per codebook to fill the device a few times over, none without work
    const int64_t want = ((int64_t)device_cu_count() * 8 + p.n_codebooks - 1) / p.n_codebooks;
    const int64_t have = (vectors_per_cb + kEncThreads * kEncPerThread - 1) / (kEncThreads * kEncPerThread);
    const int wgs_per_cb = (int)(want < have ? want : have);
    return launch_kernel((encode_b_kernel<VEC, CodeT>), dim3((unsigned)(wgs_per_cb * p.n_codebooks)), dim3(kEncThreads), 0, s, w,
                       p.cb, static_cast<CodeT *>(codes_out), vectors_per_cb, p.entries, wgs_per_cb);
}

}  // namespace

bool encode_supports(const ProblemB &p) { return p.vec == 2 || p.vec == 4 || p.vec == 8; }

hipError_t launch_encode_b(const half_t *w, const ProblemB &p, void *codes_out, hipStream_t s)
{
    if (!encode_supports(p)) return hipErrorInvalidValue;
    const bool u8 = p.code_bits == 8;
    switch (p.vec) {
    case 8: return u8 ? encode_b_typed<8, uint8_t>(w, p, codes_out, s) : encode_b_typed<8, uint16_t>(w, p, codes_out, s);
    case 4: return u8 ? encode_b_typed<4, uint8_t>(w, p, codes_out, s) : encode_b_typed<4, uint16_t>(w, p, codes_out, s);
    default: return u8 ? encode_b_typed<2, uint8_t>(w, p, codes_out, s) : encode_b_typed<2, uint16_t>(w, p, codes_out, s);
    }
}

bool lloyd_supports(const ProblemB &p) { return encode_supports(p) && scan_lds_bytes(p, true) <= kScanLds; }

int lloyd_assign_rows(const ProblemB &p) { return scan_plan(p, true).wgs_per_cb; }

hipError_t launch_lloyd_assign(const half_t *w, const ProblemB &p, void *codes_out, float *partials, bool sums, hipStream_t s)
{
    if (!lloyd_supports(p) || !scan_supports(w, p, true)) return hipErrorInvalidValue;
    auto launch = [&](auto vec, auto code) {
        typedef decltype(code) CodeT;
        return sums ? launch_scan<vec(), CodeT, kSums>(w, p, codes_out, partials, s) : launch_scan<vec(), CodeT, kErrorOnly>(w, p, codes_out, partials, s);
    };
    auto with_code = [&](auto vec) { return p.code_bits == 8 ? launch(vec, uint8_t{}) : launch(vec, uint16_t{}); };
    using std::integral_constant;
    switch (p.vec) {
    case 8: return with_code(integral_constant<int, 8>{});
    case 4: return with_code(integral_constant<int, 4>{});
    default: return with_code(integral_constant<int, 2>{});
    }
}

}  // namespace vq
