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
// vector unit 12.5 instructions per 16: of each group of eight scores four to fold them to their minimum and one to put the group's number
// into its low bits, then five per two tiles that keep the best group and the second best (10.5 per 16 in groups of sixteen).  All of them
// take 4.2 cycles here; an MFMA adds 8 to the 52 of the fold of its results while other waves fold, of its own 32.  What a 4096 x
// 4096 weight takes in 8-vectors with 256 entries: 28.9 us (the second best kept after every tile, 13 per 16, 29.5; with a comparison and
// a selection for the group's number, 16 per 16 scores, 36; by the rule 230), of which a tile of 32 entries is 1.8, the pass per vector
// behind the scan 9, table and launch 4.
//
// A wave takes 128 vectors as four batches of 32 (64 as two, where there are too few for a workgroup on every other unit), so that an entry tile read from the LDS (its halves and its
// half norms) meets four MFMAs.  A lane of the result holds 16 scores of one vector - two groups of eight entries, or one -, and
// the lane 32 further on the other 16.
//
// The half norms: as the MFMA's accumulators, 16 numbers a lane out of the LDS per tile, or (NORMS_IN_K) as products too, in the half of K
// that a vector leaves unused (8-vectors: of the MFMA with 16 of K): as a sum of halves times powers of two, which are the same for
// every vector.  What an LDS read writes into registers is not free to the vector unit: 16 cycles of a 4-vectors' tile and batch.
// Scores per group: a larger one costs the scan less and the rule more; they meet at about this many entries.
constexpr int kScanWideGroupEntries = 768;

// The low bits of a score that hold a number: which of a run of groups it is the minimum of, which entry of a group it is of.
constexpr uint32_t kRunMask = 15;
constexpr float kHidden = 0x1.3p-16f, kHiddenManyParts = 0x1.9p-16f;  // derived in the kernel
constexpr float kNumbered = 0x1p-18f;   // by which the number can move a score, and as much again for the rounding of what is made of it
// Instead of the half norm of an entry that is never chosen, and the score that nothing has yet: far from any real one, and
// finite with a number in its low bits.
constexpr float kFar = 0x1p127f;

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

__device__ __forceinline__ float min3(float a, float b, float c)
{
    // (as an instruction: the compiler would quiet operands that integer operations made)
    float r;
    asm("v_min3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

// `score` with a number in the low bits
__device__ __forceinline__ float numbered(float score, uint32_t number)
{
    return __builtin_bit_cast(float, (__builtin_bit_cast(uint32_t, score) & ~kRunMask) | number);
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

// LDS: entries padded to whole tiles of 32: halves with flipped signs, then with NORMS_IN_K the parts of |c|^2 / 2 likewise, then |c|^2 / 2
// (kFar behind the last entry; not beside parts in groups of sixteen, which are scored again by the parts), then with SUMS the sums of the vectors assigned to each entry and their number, [entry][VEC + 1], then n_buckets words.
//
// SUMS (a Lloyd iteration): every vector is added to its entry's sums, its distance to the workgroup's error, and
// both leave as the workgroup's row of `partials`: entries * (VEC + 1) sums and counts, then the error.  The sums are kept in
// double: an LDS addition of doubles takes a fifth of the time of one of floats on this device (2.1 M vectors of 8 elements:
// 19 against 99 us), and is exact for weights of any usual range.  kErrorOnly: the last assignment, whose sums nothing reads (44.2 -> 38.7 us;
// as a flag of the one kernel it cost every assignment half a microsecond).
enum ScanKeeps { kCodesOnly, kErrorOnly, kSums };

template <int VEC, typename CodeT, int GROUP, ScanKeeps KEEPS, int kScanBatches, bool NORMS_IN_K, int THREADS>
__global__ __launch_bounds__(THREADS, 4) void encode_scan_kernel(const half_t *__restrict__ w, const half_t *__restrict__ cb,
                                                                   CodeT *__restrict__ codes, int64_t vectors_per_cb, int entries,
                                                                   int wgs_per_cb, float *__restrict__ partials, int bucket_off,
                                                                   int n_buckets)
{
    extern __shared__ __align__(16) uint8_t smem[];
    __shared__ float reduce[THREADS / 64];
    constexpr bool ACCUMULATE = KEEPS != kCodesOnly, SUMS = KEEPS == kSums;
    constexpr int DW = VEC / 2;                       // dwords of a vector
    constexpr int kScanVectors = 32 * kScanBatches;   // of a wave
    // An entry's place in the table: one is left out after every 256 bytes of them, or the entries of all best groups, which
    // start at multiples of sixteen entries, would lie in the same few banks.
    constexpr int kRow = 128 / VEC;
    auto at = [](int e) { return e + e / kRow; };
    constexpr int kGroups = 16 / GROUP, kQuads = GROUP / 4;  // groups of a lane's scores; runs of four entries in a group
    constexpr int kRunTiles = (kRunMask + 1) / kGroups;      // tiles of a run of groups
    constexpr bool kWideK = NORMS_IN_K && VEC == 8;          // sixteen of K per MFMA: the vector and the norm's parts
    constexpr bool kNormTable = !NORMS_IN_K || GROUP == 8;   // the half norms lie in the LDS as floats
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, h = lane >> 5;         // vector of a batch, and which half of K (and of the rows) the lane holds
    const int n_tiles = (entries + 31) / 32;
    uint32_t *table = reinterpret_cast<uint32_t *>(smem);                         // [n_tiles * 32][DW]
    uint32_t *parts = table + scan_table_bytes(entries, VEC) / 4;                 // with NORMS_IN_K, as the table
    float *norms = reinterpret_cast<float *>(parts + (NORMS_IN_K ? scan_table_bytes(entries, VEC) / 4 : 0));
    double *sums = reinterpret_cast<double *>(norms + (kNormTable ? n_tiles * 32 : 0));
    uint32_t *bucket = reinterpret_cast<uint32_t *>(smem + bucket_off);
    const int g = blockIdx.x / wgs_per_cb, part = blockIdx.x % wgs_per_cb;
    const half_t *wg_w = w + (int64_t)g * vectors_per_cb * VEC;
    CodeT *wg_codes = codes + (int64_t)g * vectors_per_cb;

    const int64_t step = (int64_t)wgs_per_cb * (THREADS / 64) * kScanVectors;
    // a vector per lane, two batches of them at a time
    typedef uint32_t dwords_of_vector_t __attribute__((ext_vector_type(DW)));
    typedef dwords_of_vector_t vector_t __attribute__((aligned(DW < 2 ? 4 : 8)));
    auto load_vectors = [&](int64_t base, vector_t (&v)[kScanBatches / 2]) {
        const vector_t *from = reinterpret_cast<const vector_t *>(wg_w + base * VEC);
        const uint32_t last = (uint32_t)min(vectors_per_cb - 1 - base, (int64_t)kScanVectors);
#pragma unroll
        for (int u = 0; u < kScanBatches / 2; u++) v[u] = from[min((uint32_t)(u * 64 + lane), last)];
    };
    vector_t coming[kScanBatches / 2];
    int64_t base = ((int64_t)part * (THREADS / 64) + wave) * kScanVectors;
    if (base < vectors_per_cb) load_vectors(base, coming);

    // table, half norms, whether all of them are finite (else every vector of the codebook is decided by the rule)
    bool book_finite;
    float slack = 0.f, hides = kHidden;   // by which the parts of a half norm can miss it; what rounding can hide, as a share
    half8_t scales{};                  // what the parts are multiplied by
    {
        // An entry that equals an earlier one is never chosen, but beside it no vector would be clear below, and a vector by the rule
        // takes as long as twenty others: its norm becomes kFar.  The entries' hashes deal them out to buckets, and an entry looks
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
        for (int i = tid; i < n_buckets; i += THREADS) bucket[i] = ~0u;
        if (n_buckets) __syncthreads();
        for (int e = tid; e < n_tiles * 32; e += THREADS) {
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
            if constexpr (kNormTable) norms[e] = e < entries ? 0.5f * n2 : kFar;
            largest = n2 < __builtin_inff() ? fmaxf(largest, n2) : __builtin_inff();
            if (n_buckets && e < entries) atomicMin(&bucket[bucket_of(c)], (uint32_t)e);
        }
        if constexpr (SUMS)
            for (int i = tid; i < entries * (VEC + 1); i += THREADS) sums[i] = 0.0;
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) largest = fmaxf(largest, __shfl_xor(largest, d));
        if (lane == 0) reduce[wave] = largest;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < THREADS / 64; i++) largest = fmaxf(largest, reduce[i]);
        book_finite = largest < __builtin_inff();
        if constexpr (NORMS_IN_K) {
            // |c|^2 / 2 as a sum of halves times powers of two: kTop parts at the scale that the largest needs (all but the first only for
            // codebooks of norms beyond 2^31), then two for what halves leave out, 11 bits further down each.
            constexpr int kParts = VEC == 8 ? 8 : 4, kTop = kParts - 2;
            const int shift = min(max((int)(__builtin_bit_cast(uint32_t, largest) >> 23) - 127 - 15, -2), 15);
            const float scale = __builtin_bit_cast(float, (uint32_t)(shift + 127) << 23), unscale = __builtin_bit_cast(float, (uint32_t)(127 - shift) << 23);
            book_finite = book_finite && 0.5f * largest <= kTop * 65504.f * scale;
            slack = 0x1p-44f * scale;
            if (VEC == 8 && 0.5f * largest > 65504.f * scale) hides = kHiddenManyParts;
#pragma unroll
            for (int i = 0; i < kParts; i++) scales[i] = (half_t)(i < kTop ? scale : i == kTop ? scale * 0x1p-11f : scale * 0x1p-22f);
            for (int e = tid; e < n_tiles * 32; e += THREADS) {
                uint32_t c[DW];
                read_entry<DW>(table, at(e), c);
                float left = 0.f;
#pragma unroll
                for (int i = 0; i < DW; i++) {
                    const half2_t f = __builtin_bit_cast(half2_t, c[i]);
                    left = __builtin_fmaf((float)f[0], (float)f[0], left);
                    left = __builtin_fmaf((float)f[1], (float)f[1], left);
                }
                bool never = e >= entries;
                if (n_buckets && !never) {
                    const int first = (int)bucket[bucket_of(c)];
                    uint32_t other[DW];
                    read_entry<DW>(table, at(first), other);
                    uint32_t differ = first < e ? 0u : 1u;
#pragma unroll
                    for (int i = 0; i < DW; i++) differ |= one_zero(c[i]) ^ one_zero(other[i]);
                    never = !differ;
                }
                if constexpr (kNormTable)
                    if (never) norms[e] = kFar;
                left = never ? kFar : 0.5f * left;
                half_t part[kParts];
                bool full = true;
#pragma unroll
                for (int i = 0; i < kTop; i++) {
                    const float q = full ? left * unscale : 0.f;
                    full = q > 65504.f;
                    part[i] = (half_t)fminf(q, 65504.f);
                    left = __builtin_fmaf(-(float)part[i], scale, left);
                }
                part[kTop] = never ? (half_t)0.f : (half_t)(left * unscale * 0x1p11f);
                left = __builtin_fmaf(-(float)part[kTop], scale * 0x1p-11f, left);
                part[kTop + 1] = never ? (half_t)0.f : (half_t)(left * unscale * 0x1p22f);
#pragma unroll
                for (int i = 0; i < DW; i++) parts[at(e) * DW + i] = __builtin_bit_cast(uint32_t, half2_t{part[2 * i], part[2 * i + 1]});
            }
            __syncthreads();
        } else
        if (n_buckets) {
            for (int e = tid; e < entries; e += THREADS) {
                uint32_t c[DW], other[DW];
                read_entry<DW>(table, at(e), c);
                const int first = (int)bucket[bucket_of(c)];
                read_entry<DW>(table, at(first), other);
                uint32_t differ = first < e ? 0u : 1u;
#pragma unroll
                for (int i = 0; i < DW; i++) differ |= one_zero(c[i]) ^ one_zero(other[i]);
                if (!differ) norms[e] = kFar;
            }
            __syncthreads();
        }
    }

    // Infinities the compiler takes for any numbers: a minimum that starts from one folds two scores per instruction, and
    // the median with the other is a minimum, without an instruction to quiet what might be a signalling NaN.
    float above = __builtin_inff(), below = -__builtin_inff();
    asm volatile("" : "+v"(above), "+v"(below));
    float error = 0.f;
    // a tile's entries as the matrix cores take them: the lower half wave the first half of K, the upper one the other
    typedef std::conditional_t<kWideK, half8_t, half4_t> operand_t;
    const uint32_t *a_from = (NORMS_IN_K && h ? parts : table) + at(col) * DW + (!NORMS_IN_K && VEC == 8 ? 2 * h : 0);
    auto load_tile = [&](int t) {
        if constexpr (VEC == 2) {
            operand_t a = {};
            const half2_t v = __builtin_bit_cast(half2_t, table[at(t * 32 + col)]);
            if (h == 0) a = half4_t{v[0], v[1], (half_t)0.f, (half_t)0.f};
            return a;
        } else {
            const operand_t a = *reinterpret_cast<const operand_t *>(a_from + t * (32 + 32 / kRow) * DW);
            return NORMS_IN_K || VEC == 8 || h == 0 ? a : operand_t{};
        }
    };
    auto load_norms = [&](int t, float16_t &c) {
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const float4_t v = *reinterpret_cast<const float4_t *>(norms + t * 32 + 8 * q + 4 * h);
#pragma unroll
            for (int i = 0; i < 4; i++) c[4 * q + i] = v[i];
        }
    };
    auto multiply = [&](operand_t a, operand_t b, const float16_t &c) {
        if constexpr (kWideK)
            return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
        else
            return __builtin_amdgcn_mfma_f32_32x32x8f16(a, b, c, 0, 0, 0);
    };
    const int quarter = (int)((vectors_per_cb + 4 * step - 1) / (4 * step));
    for (int turn = 0; base < vectors_per_cb; base += step, turn++) {
        // A SIMD issues for its oldest wave first, which would leave the youngest alone at the end, nobody covering its waits: a
        // wave's priority falls by one with every quarter of its vectors (8-vectors 33.1 -> 30.5 us, 4-vectors 52 -> 47).
        if (turn == 0)
            __builtin_amdgcn_s_setprio(3);
        else if (turn == quarter)
            __builtin_amdgcn_s_setprio(2);
        else if (turn == 2 * quarter)
            __builtin_amdgcn_s_setprio(1);
        else if (turn == 3 * quarter)
            __builtin_amdgcn_s_setprio(0);
        vector_t own[kScanBatches / 2];
        operand_t b[kScanBatches];
        float m1[kScanBatches], m2[kScanBatches];      // of this run of groups, with the group's number in the low bits
        float all1[kScanBatches], all2[kScanBatches];  // of all runs
        int best[kScanBatches];                        // the run that all1 is of
#pragma unroll
        for (int u = 0; u < kScanBatches; u += 2) {
            own[u / 2] = coming[u / 2];
            // One swap of half waves: .lo the lower lanes' dwords followed by what the upper half wave holds, .hi the upper lanes' likewise
            if constexpr (NORMS_IN_K) {
                typedef uint32_t dwords_t __attribute__((ext_vector_type(sizeof(operand_t) / 4)));
                dwords_t lo, hi;
#pragma unroll
                for (int i = 0; i < DW; i++) {
                    const HalfWaves r = swap_half_waves(own[u / 2][i], __builtin_bit_cast(uint32_t, half2_t{scales[2 * i], scales[2 * i + 1]}));
                    lo[i] = r.lo;
                    hi[i] = r.hi;
                }
                b[u] = __builtin_bit_cast(operand_t, lo);
                b[u + 1] = __builtin_bit_cast(operand_t, hi);
            } else {
                // lanes (col, h): elements 4h .. 4h+3 of the vector (nothing where vec ends before)
                uint2_t lo = {}, hi = {};
#pragma unroll
                for (int i = 0; i < (VEC == 2 ? 1 : 2); i++) {
                    const HalfWaves r = swap_half_waves(own[u / 2][i], VEC == 8 ? own[u / 2][(i + 2) % DW] : 0u);
                    lo[i] = r.lo;
                    hi[i] = r.hi;
                }
                b[u] = __builtin_bit_cast(operand_t, lo);
                b[u + 1] = __builtin_bit_cast(operand_t, hi);
            }
        }
#pragma unroll
        for (int u = 0; u < kScanBatches; u++) {
            m1[u] = m2[u] = all1[u] = all2[u] = kFar;
            best[u] = 0;
        }
        load_vectors(base + step < vectors_per_cb ? base + step : base, coming);
        operand_t ahead{};
        if constexpr (NORMS_IN_K) ahead = load_tile(0);
        for (int t0 = 0, run = 0; t0 < n_tiles; t0 += kRunTiles, run++) {
            const int t1 = min(t0 + kRunTiles, n_tiles);
            // one tile: the best and the second best of its groups and of m1's, the one kept in m1, the other returned
            auto scan_tile = [&](int t, float (&second)[kScanBatches]) {
                uint32_t number[2] = {(uint32_t)((t - t0) * kGroups), (uint32_t)((t - t0) * kGroups + 1)};
                asm("" : "+s"(number[0]), "+s"(number[1]));
                operand_t a;
                float16_t c = {};
                if constexpr (NORMS_IN_K) {
                    a = ahead;
                    ahead = load_tile(min(t + 1, n_tiles - 1));
                } else {
                    a = load_tile(t);
                    load_norms(t, c);
                }
#pragma unroll
                for (int u = 0; u < kScanBatches; u++) {
                    const float16_t s = multiply(a, b[u], c);
                    float x[kGroups];
#pragma unroll
                    for (int gr = 0; gr < kGroups; gr++) {
                        float f = above;
#pragma unroll
                        for (int i = 0; i < GROUP; i++) f = fminf(f, s[gr * GROUP + i]);
                        x[gr] = numbered(f, number[gr]);
                    }
                    if constexpr (kGroups == 2) {
                        second[u] = __builtin_amdgcn_fmed3f(m1[u], x[0], x[1]);
                        m1[u] = min3(m1[u], x[0], x[1]);
                    } else {
                        second[u] = __builtin_amdgcn_fmed3f(m1[u], x[0], above);
                        m1[u] = __builtin_amdgcn_fmed3f(m1[u], x[0], below);
                    }
                }
            };
            int t = t0;
            float second0[kScanBatches], second1[kScanBatches];
            for (; t + 1 < t1; t += 2) {
                scan_tile(t, second0);
                scan_tile(t + 1, second1);
#pragma unroll
                for (int u = 0; u < kScanBatches; u++) m2[u] = min3(m2[u], second0[u], second1[u]);
            }
            if (t < t1) {
                scan_tile(t, second0);
#pragma unroll
                for (int u = 0; u < kScanBatches; u++) m2[u] = __builtin_amdgcn_fmed3f(m2[u], second0[u], below);
            }
            if (t1 == n_tiles && run == 0) break;   // all there is
#pragma unroll
            for (int u = 0; u < kScanBatches; u++) {
                best[u] = m1[u] < all1[u] ? run : best[u];
                all2[u] = min3(all2[u], m2[u], __builtin_amdgcn_fmed3f(m1[u], all1[u], above));
                all1[u] = __builtin_amdgcn_fmed3f(m1[u], all1[u], below);
                m1[u] = m2[u] = kFar;
            }
        }
        if (n_tiles > kRunTiles) {
#pragma unroll
            for (int u = 0; u < kScanBatches; u++) {
                m1[u] = all1[u];
                m2[u] = all2[u];
            }
        }
        // Two batches at a time, a vector per lane: lane l takes vector l of the pair.  One swap of half waves brings a lane
        // what its vector's two lanes hold: .lo of the rows of half 0, .hi of half 1.
#pragma unroll
        for (int u = 0; u < kScanBatches; u += 2) {
            uint32_t full[DW];  // the vector
#pragma unroll
            for (int i = 0; i < DW; i++) full[i] = own[u / 2][i];
            float w2 = 0.f;
#pragma unroll
            for (int i = 0; i < DW; i++) w2 = dot2(full[i], full[i], w2);
            const HalfWaves s1 = swap_half_waves(__builtin_bit_cast(uint32_t, m1[u]), __builtin_bit_cast(uint32_t, m1[u + 1]));
            const HalfWaves s2 = swap_half_waves(__builtin_bit_cast(uint32_t, m2[u]), __builtin_bit_cast(uint32_t, m2[u + 1]));
            const HalfWaves sb = swap_half_waves((uint32_t)best[u], (uint32_t)best[u + 1]);
            const float lo1 = __builtin_bit_cast(float, s1.lo), hi1 = __builtin_bit_cast(float, s1.hi);
            const bool lower = !(hi1 < lo1);  // the best group is among the rows of half 0
            const uint32_t group = (lower ? sb.lo : sb.hi) * (kRunMask + 1) + ((lower ? s1.lo : s1.hi) & kRunMask);
            const float next = min3(__builtin_amdgcn_fmed3f(lo1, hi1, above), __builtin_bit_cast(float, s2.lo), __builtin_bit_cast(float, s2.hi));
            // the scores of the group's entries once more, now one by one, with the entry's number in the group in the low bits
            const uint32_t e0 = group * (32 / kGroups) + (lower ? 0u : 4u);
            const uint32_t *entry = table + at(e0) * DW, *entry_parts = parts + at(e0) * DW;
            float first = kFar, second = kFar;
#pragma unroll
            for (int q = 0; q < kQuads; q++) {
                constexpr int kPerQ = 8;
                const int at_q = kPerQ * q + kPerQ * q / kRow;
                float x[4];
                if constexpr (kNormTable) {
                    const float4_t norm = *reinterpret_cast<const float4_t *>(norms + e0 + kPerQ * q);
#pragma unroll
                    for (int i = 0; i < 4; i++) x[i] = norm[i];
                }
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    uint32_t e[DW];
                    if constexpr (!kNormTable) {
                        read_entry<DW>(entry_parts, at_q + i, e);
                        x[i] = 0.f;
#pragma unroll
                        for (int k = 0; k < DW; k++) x[i] = dot2(e[k], __builtin_bit_cast(uint32_t, half2_t{scales[2 * k], scales[2 * k + 1]}), x[i]);
                    }
                    read_entry<DW>(entry, at_q + i, e);
#pragma unroll
                    for (int k = 0; k < DW; k++) x[i] = dot2(e[k], full[k], x[i]);
                    x[i] = numbered(x[i], 4 * q + i);
                }
                const float s01 = __builtin_amdgcn_fmed3f(first, x[0], x[1]);
                first = min3(first, x[0], x[1]);
                const float s23 = __builtin_amdgcn_fmed3f(first, x[2], x[3]);
                first = min3(first, x[2], x[3]);
                second = min3(second, s01, s23);
            }
            const uint32_t in_group = __builtin_bit_cast(uint32_t, first) & kRunMask;
            int e_best = (int)(e0 + in_group + (in_group & ~3u));
            // What rounding can hide.  With u = 2^-24: a score is off by at most E u (|w||c| + |c|^2 / 2) <= E u (|w|^2 / 2 + |c|^2), the
            // rule's distance by 10 u of itself.  (E = 28: 8 for the norm and 2 for each addition of up to eleven exact terms; 38 where
            // the largest norm takes more than one part of the first scale, up to sixteen terms.)  Whatever entry the rule would choose
            // is no further from w than the first one here, so that entry and the first both have |c| <= |w| + sqrt(D) with
            // D = |w|^2 + 2 first, |c|^2 <= 4 (|w|^2 + first).  Two scores and two halved distances: at most
            // u ((9 E + 12) |w|^2 + (8 E + 24) first).  The number in the low bits of the first score moves it by 15 * 2^-23 of itself,
            // at most 30 u (|w|^2 + first) (as first >= -|w|^2 / 2), so 294 u < kHidden (or 384 u < kHiddenManyParts) of |w|^2 + first; the
            // number in those of the others moves them by 2^-19 of themselves.  (Not clear either where anything is not finite.)
            const float other = __builtin_amdgcn_fmed3f(next, second, below);
            const float hidden = __builtin_fmaf(hides, w2 + first, slack);
            const bool clear = book_finite && __builtin_fmaf(-kNumbered, __builtin_fabsf(other), other) - first > hidden;
            // vectors that this does not decide: the rule on every entry, all lanes on one vector
            // (Distances compare as their bits do: none is negative, and a NaN is above all.)
            for (uint64_t todo = __ballot(!clear); todo; todo &= todo - 1) {
                const int v = __builtin_ctzll(todo);
                uint32_t one[DW], c[DW];
#pragma unroll
                for (int i = 0; i < DW; i++) one[i] = __builtin_amdgcn_readlane(full[i], v);
                int e_min = min(lane, entries - 1);
                read_entry<DW>(table, at(e_min), c);
                uint32_t d_min = __builtin_bit_cast(uint32_t, rule_distance<DW>(one, c));
                const bool entry_0_is_nan = (__builtin_amdgcn_readfirstlane(d_min) & 0x7fffffffu) > 0x7f800000u;  // and taken as it is
                for (int e = lane + 64; e < entries; e += 64) {
                    read_entry<DW>(table, at(e), c);
                    const uint32_t d = __builtin_bit_cast(uint32_t, rule_distance<DW>(one, c));
                    e_min = d < d_min ? e : e_min;
                    d_min = min(d, d_min);
                }
                uint32_t least = d_min;
#define VQ_LEAST(control) least = min(least, (uint32_t)__builtin_amdgcn_update_dpp((int)least, (int)least, control, 0xf, 0xf, false))
                VQ_LEAST(0x128);  // rows of sixteen lanes, rotated by 8, 4, 2 and 1
                VQ_LEAST(0x124);
                VQ_LEAST(0x122);
                VQ_LEAST(0x121);
#undef VQ_LEAST
                least = min(min((uint32_t)__builtin_amdgcn_readlane(least, 0), (uint32_t)__builtin_amdgcn_readlane(least, 16)),
                            min((uint32_t)__builtin_amdgcn_readlane(least, 32), (uint32_t)__builtin_amdgcn_readlane(least, 48)));
                int e_first = entries;
                for (uint64_t at_least = __ballot(d_min == least); at_least; at_least &= at_least - 1)
                    e_first = min(e_first, (int)__builtin_amdgcn_readlane(e_min, __builtin_ctzll(at_least)));
                e_best = lane == v ? (entry_0_is_nan ? 0 : e_first) : e_best;
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
            for (int i = tid; i < entries * (VEC + 1); i += THREADS) row[i] = (float)sums[i];
        if (tid == 0) {
            float e = 0.f;
            for (int i = 0; i < THREADS / 64; i++) e += reduce[i];
            row[entries * (VEC + 1)] = e;
        }
    }
}

size_t scan_lds_bytes(const ProblemB &p, bool accumulate, bool norms_in_k = false)
{
    const size_t padded = ((size_t)p.entries + 31) / 32 * 32, table = scan_table_bytes(p.entries, p.vec);
    const size_t norms = norms_in_k && p.entries >= kScanWideGroupEntries ? 0 : padded * 4;
    return table + (norms_in_k ? table : 0) + norms + (accumulate ? (size_t)p.entries * (p.vec + 1) * 8 : 0);
}

// (two workgroups and their few static bytes in 160 KB)
constexpr size_t kScanLdsTwoPerUnit = 79 * 1024, kScanLds = 128 * 1024;

// Threads of a workgroup, batches of a wave, workgroups per codebook: as many as are resident together - two of eight waves per
// unit, or one of sixteen where every unit has work for it and two do not fit (4096 x 4096 in 8-vectors: 5000 entries 376 -> 338 us; a
// Lloyd iteration's sums of 1000 entries 101.6 -> 85) or leave sums behind, which the update has to read (256 entries 33.8 -> 32.7; 32
// entries, whose additions meet, 28.9 -> 29.6) -, none without work.  The same for every assignment of a Lloyd iteration.
struct ScanPlan {
    int threads, batches, wgs_per_cb;
};
ScanPlan scan_plan(const ProblemB &p, bool accumulate)
{
    const int64_t vectors = (int64_t)p.rows_per_cb * (p.K / p.vec), cus = device_cu_count();
    const bool two = scan_lds_bytes(p, accumulate) <= kScanLdsTwoPerUnit;
    const bool wide = (!two || (accumulate && p.entries >= 128)) && vectors * p.n_codebooks >= cus * (kScanWideThreads / 64) * 128;
    const int threads = wide ? kScanWideThreads : kScanThreads, per_cu = wide || !two ? 1 : 2;
    const int64_t want = (cus * per_cu + p.n_codebooks - 1) / p.n_codebooks;
    auto have = [&](int batches) { return (vectors + threads / 2 * batches - 1) / (threads / 2 * batches); };
    const int batches = have(4) * p.n_codebooks * 2 <= cus ? 2 : 4;
    return {threads, batches, (int)(want < have(batches) ? want : have(batches))};
}

// Half norms as parts of K: of 4-vectors wherever two workgroups still share a unit (no MFMA more, and a quarter of the LDS reads: 4096 x
// 4096 with 256 entries 57 -> 48 us, with 4096 entries 523 -> 447), of 8-vectors, whose MFMA is the longer one then, only beside the
// LDS additions of a Lloyd iteration (35.5 -> 34.0; codes alone 29.5 -> 30.5) and not for waves of two batches, whose launches are
// mostly prologue (512 x 512: 6.7 -> 6.9).
bool scan_norms_in_k(const ProblemB &p, bool accumulate, bool sums, int batches)
{
    return (p.vec == 4 || (p.vec == 8 && sums && batches == 4)) && scan_lds_bytes(p, accumulate, true) <= kScanLdsTwoPerUnit;
}

// Buckets for finding equal entries: four per entry where the LDS has room that neither keeps a second workgroup off the unit nor the
// codebook off this kernel; none where not even one per two entries fits.
int scan_buckets(size_t bytes, int entries)
{
    const size_t room = ((bytes <= kScanLdsTwoPerUnit ? kScanLdsTwoPerUnit : kScanLds) - bytes) / 4, want = 4 * (size_t)entries;
    return room >= want ? (int)want : 2 * room >= (size_t)entries ? (int)room : 0;
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
    const bool in_k = scan_norms_in_k(p, accumulate, KEEPS == kSums, plan.batches), narrow = p.entries < kScanWideGroupEntries;
    const size_t smem = scan_lds_bytes(p, accumulate, in_k);
    const int buckets = scan_buckets(smem, p.entries);
    auto launch = [&](auto threads, auto batches, auto norms_in_k) {
        auto go = [&](auto kern) {
            return launch_kernel(kern, dim3((unsigned)(plan.wgs_per_cb * p.n_codebooks)), dim3(threads()), smem + 4 * (size_t)buckets, s, w, p.cb,
                                 static_cast<CodeT *>(codes_out), vectors_per_cb, p.entries, plan.wgs_per_cb, partials, (int)smem, buckets);
        };
        if (narrow) return go(encode_scan_kernel<VEC, CodeT, 8, KEEPS, batches(), norms_in_k(), threads()>);
        return go(encode_scan_kernel<VEC, CodeT, 16, KEEPS, batches(), norms_in_k(), threads()>);
    };
    using std::integral_constant;
    using four = integral_constant<int, 4>;
    using two = integral_constant<int, 2>;
    using wide = integral_constant<int, kScanWideThreads>;
    using usual = integral_constant<int, kScanThreads>;
    const bool wide_wg = plan.threads == kScanWideThreads;
    if constexpr (VEC == 4 || (VEC == 8 && KEEPS == kSums))
        if (in_k) {
            if constexpr (accumulate)
                if (wide_wg) return launch(wide{}, four{}, std::true_type{});
            if constexpr (VEC == 4)
                if (plan.batches == 2) return launch(usual{}, two{}, std::true_type{});
            return launch(usual{}, four{}, std::true_type{});
        }
    if (wide_wg) return launch(wide{}, four{}, std::false_type{});
    return plan.batches == 4 ? launch(usual{}, four{}, std::false_type{}) : launch(usual{}, two{}, std::false_type{});
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
