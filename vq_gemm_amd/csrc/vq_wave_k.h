// Products whose tiles of the large kernels are fewer than the compute units: a workgroup takes a small tile of Y
// (16 to 96 rows by 16 to 128 columns) and its waves, eight in nearly all tiles, deal K out among themselves.
//
//   NN:        y[M,N] = x[M,K] . w[K,N], fp16 w
//   geometry A: out[M, 2*Nc] = x[M,K] . W_dec, W_dec[k, 2n + r] = codebook[n/4][w[k,n]][r] (reference
//               strategy_2/bsz512/src.cu:163-176, bench.py:46-56)
//   geometry B: y[M,N] = x[M,K] . W^T, W given as codes [N, K/vec] and codebooks
//
// Every wave multiplies the whole tile for its own k: units of 32 k go round the waves.  What a wave stages through the
// LDS only it reads, so nothing in the loop waits for another wave - no barrier, only the wave's own loads - and an operand
// of a wave serves the whole height (width) of the tile, where waves that share out a tile of this size would read every
// operand once per wave.  Units in flight: 100 to 150 KB per compute unit, what it takes to keep the memory busy from few
// workgroups.  At the end the waves' partial tiles are added up through the LDS, in the order of the waves, in fp32, and
// rounded once.  Geometry A's tiles of 64 x 64 and more are vq_wave_k_a.hip's.
//
// What bounds it: with few tiles the launch, the latency of the first units and the sum over the waves (together about
// 4 us); with many the LDS, which carries each unit in and out once.
//
//   * X lies in the LDS in rows of 64 or 128 bytes, XOR-swizzled (wave_x_swizzle).
//   * fp16 W lies as k-rows and is read with the transposing ds_read_b64_tr_b16.  Rows of W that are no multiple of 16
//     bytes (N % 8 != 0, or a pointer aligned to 2 bytes) cannot be loaded into the LDS directly: they go through registers.
//   * Codes of geometry A lie as k-rows of bytes; ds_read_b64_tr_b8 hands a lane the eight codes of its code column, and
//     the eight 4-byte gathers behind them are the operands of two pieces, the even and the odd columns of Y: no
//     dequantised tile is written to the LDS and read back.
//   * Codes of geometry B lie as 16-byte chunks of their rows; a lane reads those of both steps of a unit at once - it takes the
//     sixteen k from 16*kg on, eight a step, and X in the same order - and gathers its operands from the codebooks.
#pragma once

#include "vq_prefill_common.h"

#include <algorithm>
#include <type_traits>

namespace vq {

namespace {

constexpr int kStepK = 32;                // k of one MFMA step
constexpr int kCopiesBytes = 64 * 1024;   // a table of copies: a row of banks for each of 256 entries, or half of one for each of 512

// What W is and how a unit of it is laid out.  S: MFMA steps of a unit.
struct WaveDense {       // fp16 [K,N], rows of whole 16-byte chunks
    static constexpr int S = 1;
    static constexpr bool kDense = true, kAnyN = false, kA = false, kB = false, kCopies = false;
    static constexpr int VEC = 0, CSZ = 2;
};
struct WaveDenseAnyN {   // fp16 [K,N], any N, elements aligned to 2 bytes
    static constexpr int S = 1;
    static constexpr bool kDense = false, kAnyN = true, kA = false, kB = false, kCopies = false;
    static constexpr int VEC = 0, CSZ = 2;
};
struct WaveA {           // geometry A
    static constexpr int S = 1;
    static constexpr bool kDense = false, kAnyN = false, kA = true, kB = false, kCopies = false;
    static constexpr int VEC = 2, CSZ = 1;
};
// COPIES: the table holds one codebook of at most 256 entries, each as often as fills a row of the 64 banks (16 copies of
// an 8-vector, 32 of a 4-vector), and a lane gathers its own copy: no two lanes of a gather meet in a bank.  16-bit codes: of at
// most 512 entries, each half as often; two lanes meet where their entries lie in the same half of a row.
template <int VEC_, typename CodeT_, int S_, bool COPIES_ = false>
struct WaveB {           // geometry B
    static constexpr bool kCopies = COPIES_;
    static constexpr int kCopyRow = sizeof(CodeT_) == 1 ? 256 : 128, kCopyEntries = kCopiesBytes / kCopyRow;
    static constexpr int S = S_;
    static constexpr bool kDense = false, kAnyN = false, kA = false, kB = true;
    static constexpr int VEC = VEC_, CSZ = (int)sizeof(CodeT_);
};

// Waves of a workgroup: two on every SIMD, one's MFMAs beside the other's reads; four on every SIMD for
// the smallest tile on a table of copies, whose waves wait for one another's reads least (M = 16, K = 11008, N = 4096 9.2 -> 8.5 us; twice
// as wide a tile gains nothing from it, 9.7, and loses at K = 4096, 6.0 -> 6.7).
template <class P>
constexpr int wave_count(int mp, int np) { return P::kB && P::kCopies && mp * np == 1 ? 16 : 8; }

// Rows of pieces whose partial sums, `per_row` KB of them each, fit the LDS together: the most that divide the tile's.
constexpr int pass_rows(int mp, int per_row)
{
    int rows = mp;
    while (rows > 1 && (mp % rows != 0 || rows * per_row > 160)) rows--;
    return rows;
}

// MP x NP pieces of 16 x 16: the tile.
template <class P, int MP, int NP>
struct WaveKCfg {
    static constexpr int kWaves = wave_count<P>(MP, NP);
    static constexpr int S = P::S, kUnitK = S * kStepK;
    static constexpr int TM = MP * 16, TN = NP * 16;
    static constexpr int kXBytes = S * MP * 1024;
    // 16-byte chunks of a row of W in a unit - a k-row, or for geometry B a row of codes, whose chunks lie TN * 16 apart -
    // and the direct loads of a unit (64 chunks each)
    static constexpr int kRows = P::kB ? TN : kUnitK;
    static constexpr int kCodeBytes = P::kB ? kUnitK / P::VEC * P::CSZ : 0;                // of a row and unit: 4, 8, 16 or 32
    static constexpr int kRowChunks = P::kB ? (kCodeBytes + 15) / 16 : P::kA ? NP / 2 : P::kDense ? 2 * NP : 2 * NP + 1;
    static constexpr int kWLoads = (kRows * kRowChunks + 63) / 64;
    static constexpr int kUnitBytes = kXBytes + kWLoads * 1024;
    static constexpr int kLoads = S * MP + kWLoads;                                        // direct loads of a wave and unit
    static constexpr int kBooks = P::kA ? TN / 8 * 1024 : 0;                                 // bytes of codebooks known here
    static constexpr int kRoom = 160 * 1024 - (P::kCopies ? kCopiesBytes : P::kB ? (P::CSZ == 2 ? 33 : 5) * 1024 : kBooks);
    static constexpr int kFit = kRoom / (kWaves * kUnitBytes);
    static constexpr int D = kFit > 6 ? 6 : kFit;                                           // units in the LDS per wave
    static constexpr int kRing = kWaves * D * kUnitBytes;
    static constexpr int kPassMP = pass_rows(MP, NP * kWaves);                              // rows of pieces summed in one pass
    static constexpr int kSumBytes = kWaves * kPassMP * NP * 1024;
    static constexpr bool kExists = D >= 2;   // the LDS holds two units of every wave
    static_assert(D * kLoads < 64 && kPassMP >= 1 && MP % kPassMP == 0 && kSumBytes <= 160 * 1024, "counts of loads, passes of the sum");
    // (`books` bytes of codebooks, copied in steps of a wave load)
    static constexpr size_t lds_bytes(size_t books)
    {
        const size_t use = kRing + (P::kCopies ? (size_t)kCopiesBytes : copied_bytes(books));
        return use > (size_t)kSumBytes ? use : (size_t)kSumBytes;
    }
};

// X in a unit lies in rows of 64 bytes, four to a 256-byte bank row (one step), or of 128 bytes, two to a bank row (two steps), the
// chunks of a bank row XOR-swizzled with a function of its number.  A 16-byte read serves sixteen lanes at a time, not in their
// order but lanes 0-3, 12-15, 20-23 and 24-27, then 4-11, 16-19 and 28-31 (and the upper half wave alike): rows r16 of one chunk column
// and of the next together.  With these functions they fall into sixteen different chunks of the bank row: 4 cycles a read,
// where the bank row's own number makes it 8.
template <int S>
__device__ __forceinline__ int wave_x_swizzle(int bank_row)
{
    return S == 2 ? (bank_row & 1) | ((bank_row >> 2) & 1) * 6 : -bank_row & 3;
}

// Byte offset of chunk cc (16 bytes) of row `row`.
template <int S>
__device__ __forceinline__ int wave_x_offset(int row, int cc)
{
    const int bank_row = S == 2 ? row >> 1 : row >> 2;
    const int pos = (S == 2 ? ((row & 1) << 3) | cc : ((row & 3) << 2) | cc) ^ wave_x_swizzle<S>(bank_row);
    return (bank_row * 16 + pos) * 16;
}

// Rows of fp16 W: the XOR on the chunk index of k-row `k`, such that the eight rows x 32 bytes a half wave of a transposing
// read touches - four from k-row 8*kg on, for two kg - fall into different banks.
template <int NP>
__device__ __forceinline__ int wave_w_swizzle(int k)
{
    static_assert(NP == 2 || NP == 4, "32 or 64 columns");
    return NP == 4 ? ((k >> 1) & 1) * 2 + ((k >> 3) & 1) * 4 : ((k >> 3) & 1) * 2;
}

struct WaveKArgs {
    const half_t *x;
    const void *w;         // fp16 W, or codes
    const half_t *cb;
    half_t *y;
    const half_t *bias;
    int M, K, N;
    int k_x;               // columns of X: K, or K / stages where X repeats along K
    int tiles_m, tiles_n;
    int entries, rows_per_cb, books;   // (geometry B) books: codebooks of a tile
    int gated;
    int by_rows;           // consecutive tiles lie along the rows of tiles (wave_k_by_rows)
};

template <class P, int MP, int NP>
__global__ __launch_bounds__(wave_count<P>(MP, NP) * 64, wave_count<P>(MP, NP) / 4) void wave_k_kernel(const WaveKArgs a)
{
    typedef WaveKCfg<P, MP, NP> C;
    static_assert(C::kExists, "a tile the LDS holds");
    constexpr int D = C::D, S = C::S, kWaves = C::kWaves, kUnitK = C::kUnitK, kRowChunks = C::kRowChunks;
    extern __shared__ __align__(16) uint8_t smem[];
    const int M = a.M, K = a.K, N = a.N, k_x = P::kB ? a.k_x : a.K;
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int r16 = lane & 15, kg = lane >> 4;

    // Workgroup ids are dealt round-robin to the 8 XCDs: an XCD takes consecutive tiles, by rows or by columns.
    const int n_wg = a.tiles_m * a.tiles_n, xcd = blockIdx.x & 7;
    const int tile = xcd * (n_wg >> 3) + min(xcd, n_wg & 7) + ((int)blockIdx.x >> 3);
    const int along = a.by_rows ? a.tiles_n : a.tiles_m, line = tile / along, at_line = tile - line * along;
    const int tm = a.by_rows ? line : at_line, tn = a.by_rows ? at_line : line;
    const int m0 = tm * C::TM, n0 = tn * C::TN;
    const int n_all = K / kUnitK;
    const int n_unit = (n_all - wave + kWaves - 1) / kWaves;  // of this wave: wave, wave + kWaves, ...
    const uint32_t ring = (uint32_t)wave * (D * C::kUnitBytes);
    constexpr int kBookBase = C::kRing;

    // ---- global -> LDS --------------------------------------------------------------------------
    uint32_t x_voff[S * MP];
#pragma unroll
    for (int i = 0; i < S * MP; i++) {
        const int slot = i * 64 + lane;
        const int bank_row = slot >> 4;
        const int pos = (slot & 15) ^ wave_x_swizzle<S>(bank_row);
        const int row = S == 2 ? 2 * bank_row + (pos >> 3) : 4 * bank_row + (pos >> 2), cc = pos & (4 * S - 1);
        x_voff[i] = (uint32_t)(((int64_t)(min(m0 + row, M - 1) - m0) * k_x + cc * 8) * 2);
    }
    // bytes of a row of w, and its tile's first byte in it (geometry B: rows are rows of codes, the tile's first is n0)
    const int64_t w_row = P::kB ? (int64_t)(K / (P::kB ? P::VEC : 1)) * P::CSZ : P::kA ? N / 2 : (int64_t)N * 2;
    const int64_t w_col = P::kB ? 0 : P::kA ? n0 / 2 : (int64_t)n0 * 2;
    // (kAnyN) bytes from the granule of 16 that holds the tile's first element to that element: the same for every unit,
    // which lie 64 * N bytes apart
    const int w_skew = P::kAnyN ? (int)((reinterpret_cast<uintptr_t>(a.w) + (uintptr_t)w_col) & 15) : 0;
    uint32_t w_voff[C::kWLoads];
#pragma unroll
    for (int i = 0; i < C::kWLoads; i++) {
        const int slot = min(i * 64 + lane, C::kRows * kRowChunks - 1);   // (lanes beyond the unit: its last chunk again)
        if constexpr (P::kB) {
            const int c = slot / C::kRows, row = slot % C::kRows;
            w_voff[i] = (uint32_t)((int64_t)min(row, N - 1 - n0) * w_row + c * 16);
        } else {
            const int k = slot / kRowChunks, c = slot % kRowChunks;
            if constexpr (P::kAnyN) {
                // the granules that hold the row's columns, up to the one with its last (each holds a byte of the row, so it
                // lies in the same page as the row), from the tile's first granule on
                const int64_t first = (k * w_row + w_skew) & ~(int64_t)15;
                const int64_t last = (k * w_row + w_skew + (int64_t)min(C::TN, N - n0) * 2 - 1) & ~(int64_t)15;
                w_voff[i] = (uint32_t)min(first + c * 16, last);
            } else {
                const int cs = P::kDense ? c ^ wave_w_swizzle<NP>(k) : c;
                w_voff[i] = (uint32_t)(k * w_row + min(w_col + cs * 16, w_row - 16) - w_col);
            }
        }
    }
    // (geometry B, fewer than sixteen bytes of codes per row and unit: the sixteen around them are loaded, from a multiple of
    // eight on and inside the row)
    constexpr bool kPartChunk = P::kB && C::kCodeBytes < 16;
    auto code_skip = [&](int u) {   // bytes from where unit u's load begins to its codes
        const int at = (u * kWaves + wave) * C::kCodeBytes;
        return kPartChunk ? at - min(at & ~7, (int)w_row - 16) : 0;
    };
    const int64_t w_unit = P::kB ? C::kCodeBytes : kUnitK * w_row;     // bytes from unit to unit
    const half_t *x_tile = a.x + (int64_t)m0 * k_x;
    // (an X that repeats along K: modulo its columns, by a loop; where a codebook entry is on its way without a branch.  That everywhere
    // cost the kernel for 4-vectors with 16-bit codes 2 %: M = 16, K = 4096, N = 11008 8.08 -> 8.25 us.)
    int x_at = wave * kUnitK, x_step = kWaves * kUnitK;
    if constexpr (P::kB) {
        while (x_at >= k_x) x_at -= k_x;
        if constexpr (P::kCopies)
            while (x_step >= k_x) x_step -= k_x;
    }
    const uint8_t *w_ahead = static_cast<const uint8_t *>(a.w) + (P::kB ? (int64_t)n0 * w_row : w_col - w_skew) + wave * w_unit;
    auto issue = [&](int buf, int u) {
        const uint32_t at = ring + buf * C::kUnitBytes;
        const uint8_t *src = w_ahead - code_skip(u);
#pragma unroll
        for (int i = 0; i < C::kWLoads; i++) load_to_lds_16(at + C::kXBytes + i * 1024, w_voff[i], src);
#pragma unroll
        for (int i = 0; i < S * MP; i++) load_to_lds_16(at + i * 1024, x_voff[i], x_tile + x_at);
        w_ahead += kWaves * w_unit;
        x_at += x_step;
        if constexpr (P::kCopies) x_at = (int)min((uint32_t)x_at, (uint32_t)(x_at - k_x));
        else if constexpr (P::kB)
            while (x_at >= k_x) x_at -= k_x;
    };

    // ---- operands -------------------------------------------------------------------------------
    // Chunk of X of step s: natural order, or (geometry B in units of two steps) 2*kg + s - a lane then finds the codes of both steps side by side.
    uint32_t x_rd[S == 2 ? 2 : 1][2];   // [step][parity of the piece]: + piece * 1 KB (two steps: + piece pair * 4 KB)
#pragma unroll
    for (int s = 0; s < S; s++)
#pragma unroll
        for (int par = 0; par < 2; par++) x_rd[s][par] = ring + wave_x_offset<S>((S == 2 ? par * 16 : 0) + r16, P::kB && S == 2 ? 2 * kg + s : 4 * s + kg);
    uint32_t w_rd[P::kAnyN ? 8 : P::kA ? NP / 2 : NP];
    if constexpr (P::kA) {
        // source lane (kg, s = r16) of the transposing read supplies k-row kg*8 + s/2, codes 8*(s%2) .. +7 of a group of 16
#pragma unroll
        for (int q = 0; q < NP / 2; q++) w_rd[q] = ring + C::kXBytes + (kg * 8 + (r16 >> 1)) * (kRowChunks * 16) + q * 16 + (r16 & 1) * 8;
    } else if constexpr (P::kAnyN) {
        // element by element: column r16 of a piece in k-rows kg*8 .. +7, each with its own offset from its first granule
#pragma unroll
        for (int t = 0; t < 8; t++) {
            const int k = kg * 8 + t;
            w_rd[t] = ring + C::kXBytes + k * (kRowChunks * 16) + (uint32_t)((k * w_row + w_skew) & 15) + r16 * 2;
        }
    } else if constexpr (P::kDense) {
        // source lane (kg, s = r16) supplies k-row kg*8 + h*4 + s/4, columns piece*16 + 4*(s%4) .. +3
        // (four k-rows on, and 32: the same XOR)
        const int k = kg * 8 + (r16 >> 2);
#pragma unroll
        for (int j = 0; j < NP; j++)
            w_rd[j] = ring + C::kXBytes + k * (kRowChunks * 16) + (r16 & 1) * 8 + ((2 * j + ((r16 & 3) >> 1)) ^ wave_w_swizzle<NP>(k)) * 16;
    } else {
        // codebook of the piece's row, or the lane's copy in it
        const int g_first = n0 / a.rows_per_cb;
#pragma unroll
        for (int j = 0; j < NP; j++)
            if constexpr (P::kCopies) w_rd[j] = kBookBase + (uint32_t)(lane * (P::VEC * 2) & (P::kCopyRow - 1));
            else w_rd[j] = kBookBase + (uint32_t)((min(n0 + j * 16 + r16, N - 1) / a.rows_per_cb - g_first) * a.entries * (P::VEC * 2));
    }
    const uint32_t code_rd = ring + C::kXBytes + (C::kCodeBytes == 32 ? (kg >> 1) * (C::kRows * 16) + (kg & 1) * 8 : kg * (C::kCodeBytes / 4)) + r16 * 16;
    typedef short short4_t __attribute__((__vector_size__(4 * sizeof(short))));
    typedef int int2v_t __attribute__((__vector_size__(2 * sizeof(int))));
    typedef __attribute__((address_space(3))) short4_t lds_short4_t;
    typedef __attribute__((address_space(3))) int2v_t lds_int2_t;
    half8_t xs[2][MP], ws[2][NP];
    int2v_t code_a[P::kA ? NP / 2 : 1];
    uint32_t code_b[P::kB ? NP : 1][C::kCodeBytes == 32 ? 2 : 1];   // of both steps of a unit
    auto read_x = [&](int set, int buf, int s) {
#pragma unroll
        for (int i = 0; i < MP; i++)
            xs[set][i] = *reinterpret_cast<const half8_t *>(smem + x_rd[s][i & 1] + buf * C::kUnitBytes + (S == 2 ? (i >> 1) * 4096 : i * 1024));
    };
    // W operands of step s of the unit in `buf`; geometry A and B: its codes first (B: of all its steps; skip: code_skip)
    auto read_codes = [&](int buf, int skip) {
        if constexpr (P::kA) {
#pragma unroll
            for (int q = 0; q < NP / 2; q++)
                code_a[q] = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_int2_t *)(smem + w_rd[q] + buf * C::kUnitBytes));
        } else if constexpr (P::kB) {
            const uint8_t *src = smem + code_rd + buf * C::kUnitBytes + skip;
#pragma unroll
            for (int j = 0; j < NP; j++) {
                if constexpr (C::kCodeBytes == 4) {
                    code_b[j][0] = src[j * 256];
                } else if constexpr (C::kCodeBytes == 8) {
                    code_b[j][0] = *reinterpret_cast<const uint16_t *>(src + j * 256);
                } else if constexpr (C::kCodeBytes == 16) {
                    code_b[j][0] = *reinterpret_cast<const uint32_t *>(src + j * 256);
                } else {
                    const uint2_t v = *reinterpret_cast<const uint2_t *>(src + j * 256);
                    code_b[j][0] = v[0];
                    code_b[j][1] = v[1];
                }
            }
        }
    };
    auto read_w = [&](int set, int buf, int s) {
        if constexpr (P::kA) {
#pragma unroll
            for (int q = 0; q < NP / 2; q++) {
                const uint32_t book = kBookBase + (q * 4 + (r16 >> 2)) * 1024;
                uint32_t g[8];
#pragma unroll
                for (int t = 0; t < 8; t++) {
                    const uint32_t c = ((uint32_t)code_a[q][t >> 2] >> (8 * (t & 3))) & 0xffu;
                    g[t] = *reinterpret_cast<const uint32_t *>(smem + book + c * 4);
                }
                uint4_t even, odd;
#pragma unroll
                for (int t = 0; t < 4; t++) {
                    even[t] = __builtin_amdgcn_perm(g[2 * t + 1], g[2 * t], 0x05040100);
                    odd[t] = __builtin_amdgcn_perm(g[2 * t + 1], g[2 * t], 0x07060302);
                }
                ws[set][2 * q] = __builtin_bit_cast(half8_t, even);
                ws[set][2 * q + 1] = __builtin_bit_cast(half8_t, odd);
            }
        } else if constexpr (P::kB) {
            constexpr int kEntry = []() constexpr {   // bytes from entry to entry
                if constexpr (P::kCopies) return P::kCopyRow;
                else return P::VEC * 2;
            }();
#pragma unroll
            for (int j = 0; j < NP; j++) {
                if constexpr (P::VEC == 8) {
                    const uint32_t c = P::CSZ == 1 ? (code_b[j][0] >> (8 * s)) & 0xffu : (code_b[j][0] >> (16 * s)) & 0xffffu;
                    ws[set][j] = *reinterpret_cast<const half8_t *>(smem + w_rd[j] + c * kEntry);
                } else {
                    const uint32_t pair = P::CSZ == 1 ? (code_b[j][0] >> (16 * s)) & 0xffffu : code_b[j][C::kCodeBytes == 32 ? s : 0];
                    const uint32_t c_lo = P::CSZ == 1 ? pair & 0xffu : pair & 0xffffu, c_hi = P::CSZ == 1 ? pair >> 8 : pair >> 16;
                    const half4_t lo = *reinterpret_cast<const half4_t *>(smem + w_rd[j] + c_lo * kEntry);
                    const half4_t hi = *reinterpret_cast<const half4_t *>(smem + w_rd[j] + c_hi * kEntry);
                    ws[set][j] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
                }
            }
        } else if constexpr (P::kAnyN) {
#pragma unroll
            for (int j = 0; j < NP; j++)
#pragma unroll
                for (int t = 0; t < 8; t++) ws[set][j][t] = *reinterpret_cast<const half_t *>(smem + w_rd[t] + buf * C::kUnitBytes + j * 32);
        } else {
#pragma unroll
            for (int j = 0; j < NP; j++) {
                const uint8_t *src = smem + w_rd[j] + buf * C::kUnitBytes + s * (32 * kRowChunks * 16);
                const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_t *)src);
                const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_t *)(src + 4 * kRowChunks * 16));
                ws[set][j] = __builtin_shufflevector(__builtin_bit_cast(half4_t, lo), __builtin_bit_cast(half4_t, hi), 0, 1, 2, 3, 4, 5, 6, 7);
            }
        }
    };

    float4_t acc[NP][MP];
#pragma unroll
    for (int j = 0; j < NP; j++)
#pragma unroll
        for (int i = 0; i < MP; i++) acc[j][i] = float4_t{0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](int set) {
#pragma unroll
        for (int j = 0; j < NP; j++)
#pragma unroll
            for (int i = 0; i < MP; i++) acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ws[set][j], xs[set][i], acc[j][i], 0, 0, 0);
    };

    // ---- codebooks, first units -------------------------------------------------------------------
    if constexpr (!P::kCopies && (P::kA || P::kB)) {
        const int book_bytes = P::kA ? 1024 : a.entries * (P::VEC * 2);
        const int g_first = P::kA ? n0 / 8 : n0 / a.rows_per_cb;
        const int n16 = (P::kA ? C::TN / 8 : a.books) * book_bytes / 16;
        const int n_books = P::kA ? N / 8 : (N + a.rows_per_cb - 1) / a.rows_per_cb;
        const int last16 = (int)((int64_t)(n_books - g_first) * book_bytes / 16) - 1;   // past the last codebook: its last 16 bytes again
        const uint8_t *src = reinterpret_cast<const uint8_t *>(a.cb) + (int64_t)g_first * book_bytes;
        for (int i0 = wave * 64; i0 < n16; i0 += kWaves * 64)
            load_to_lds_16(kBookBase + i0 * 16, (uint32_t)min(i0 + lane, last16) * 16u, src);
    }
    if constexpr (P::kCopies) {
        // The thread's entry comes by a load into registers, beside the others the first to be back.  The compiler does not count it: nothing
        // but the units' loads, no branch, lies between it and the wait (the build looks at that), and where there are
        // fewer units it goes last.
        static_assert(P::VEC == 8 || P::VEC == 4, "entries of 16 or 8 bytes");
        typedef uint32_t entry_t __attribute__((ext_vector_type(P::VEC / 2)));
        const half_t *src = a.cb + ((int64_t)(n0 / a.rows_per_cb) * a.entries + min(tid & (P::kCopyEntries - 1), a.entries - 1)) * P::VEC;
        entry_t entry;
        auto load_entry = [&]() {
            if constexpr (P::VEC == 8) asm volatile("global_load_dwordx4 %0, %1, off" : "=&v"(entry) : "v"(src) : "memory");
            else asm volatile("global_load_dwordx2 %0, %1, off" : "=&v"(entry) : "v"(src) : "memory");
        };
        // two threads an entry (four of sixteen waves; half of that for 512 entries), four or eight pieces of 16 bytes each, neighbouring entries
        // in another order
        auto write_copies = [&]() {
            asm volatile("" : "+v"(entry));
            constexpr int kPer = kWaves * 64 / P::kCopyEntries, kPieces = P::kCopyRow / 16 / kPer;
            static_assert(kPer >= 1 && kPer <= 4 && (kPieces == 4 || kPieces == 8), "threads an entry");
            const uint4_t piece = {entry[0], entry[1], entry[P::VEC == 8 ? 2 : 0], entry[P::VEC == 8 ? 3 : 1]};
            const uint32_t at = kBookBase + (tid & (P::kCopyEntries - 1)) * P::kCopyRow + tid / P::kCopyEntries * (kPieces * 16) + (tid & (kPieces - 1)) * 16;
#pragma unroll
            for (int i = 0; i < kPieces; i++) *reinterpret_cast<uint4_t *>(smem + (at ^ (i * 16))) = piece;
        };
        if (n_unit >= D) {
            load_entry();
#pragma unroll
            for (int d = 0; d < D; d++) issue(d, d);
            wait_vmcnt<D * C::kLoads>();
            write_copies();
        } else {
#pragma unroll
            for (int d = 0; d < D; d++)
                if (d < n_unit) issue(d, d);
            load_entry();
            wait_vmcnt<0>();
            write_copies();
        }
        __syncthreads();
    } else {
#pragma unroll
        for (int d = 0; d < D; d++)
            if (d < n_unit) issue(d, d);
    }
    if constexpr (!P::kCopies && (P::kA || P::kB)) {
        // (the codebooks are the oldest loads of the waves that brought them)
        if (n_unit >= D) wait_vmcnt<D * C::kLoads>();
        else wait_vmcnt<0>();
        __syncthreads();
    }

    // ---- the wave's units ---------------------------------------------------------------------------
    // While a step multiplies one register set, the operands of the next are read into the other.  A unit's buffer is free
    // as soon as its last reads are through: unit u + D is loaded there.
    if (n_unit > 0) {
        if (n_unit > D - 1) wait_vmcnt<(D - 1) * C::kLoads>();
        else wait_vmcnt<0>();
        asm volatile("" ::: "memory");
        read_codes(0, code_skip(0));
        read_x(0, 0, 0);
        read_w(0, 0, 0);
        int buf = 0;
        // the last step of unit u, in register set `set`
        auto last_step = [&](auto set_const, int u) {
            constexpr int set = decltype(set_const)::value;
            const int next = buf + 1 == D ? 0 : buf + 1;
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            if (u + D < n_unit) {
                issue(buf, u + D);
                wait_vmcnt<(D - 1) * C::kLoads>();
            } else {
                wait_vmcnt<0>();
            }
            asm volatile("" ::: "memory");
            if (u + 1 < n_unit) {
                read_codes(next, code_skip(u + 1));
                read_x(set ^ 1, next, 0);
                read_w(set ^ 1, next, 0);
            }
            multiply(set);
            buf = next;
        };
        if constexpr (S == 2) {
            for (int u = 0; u < n_unit; u++) {
                read_x(1, buf, 1);
                read_w(1, buf, 1);
                multiply(0);
                last_step(std::integral_constant<int, 1>{}, u);
            }
        } else {
            int u = 0;
            for (; u + 1 < n_unit; u += 2) {
                last_step(std::integral_constant<int, 0>{}, u);
                last_step(std::integral_constant<int, 1>{}, u + 1);
            }
            if (u < n_unit) last_step(std::integral_constant<int, 0>{}, u);
        }
    }

    // ---- the sum over the waves ---------------------------------------------------------------------
    // A piece is 1 KB, float4 by lane; a wave takes pairs of pieces of a row of pieces.
    constexpr int PM = C::kPassMP, H = NP % 2 == 0 ? 2 : 1, kPairs = PM * NP / H;
#pragma unroll
    for (int pass = 0; pass < MP / PM; pass++) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < PM; i++)
#pragma unroll
            for (int j = 0; j < NP; j++)
                *reinterpret_cast<float4_t *>(smem + ((wave * PM + i) * NP + j) * 1024 + lane * 16) = acc[j][pass * PM + i];
        __syncthreads();
        for (int pair = wave; pair < kPairs; pair += kWaves) {
            const int i = pair / (NP / H), q = pair % (NP / H);
            const int m = m0 + (pass * PM + i) * 16 + r16;
            float4_t sum[H];
#pragma unroll
            for (int h = 0; h < H; h++) {
                const uint8_t *src = smem + (i * NP + H * q + h) * 1024 + lane * 16;
                sum[h] = *reinterpret_cast<const float4_t *>(src);
#pragma unroll
                for (int v = 1; v < kWaves; v++) sum[h] += *reinterpret_cast<const float4_t *>(src + v * (PM * NP * 1024));
            }
            if (m >= M) continue;
            if constexpr (P::kA) {
                // the even columns and the odd ones: eight columns in a row
                const int n = n0 + q * 32 + kg * 8;
                half8_t v;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    v[2 * e] = (half_t)sum[0][e];
                    v[2 * e + 1] = (half_t)sum[1][e];
                }
                if (n < N) __builtin_memcpy(a.y + (int64_t)m * N + n, &v, 16);
            } else {
                int n = n0 + H * q * 16 + kg * 4, end = N;
                if (P::kB && a.bias) {
#pragma unroll
                    for (int h = 0; h < H; h++)
#pragma unroll
                        for (int e = 0; e < 4; e++) sum[h][e] += (float)a.bias[min(n + h * 16 + e, N - 1)];
                }
                const bool gated = P::kB && H == 2 && a.gated;
                if constexpr (H == 2)
                    if (gated) {
#pragma unroll
                        for (int e = 0; e < 4; e++) sum[0][e] = silu_f32(sum[0][e]) * sum[1][e];
                        n = n0 / 2 + q * 16 + kg * 4;
                        end = N / 2;
                    }
                half_t *row = a.y + (int64_t)m * end;
#pragma unroll
                for (int h = 0; h < H; h++) {
                    if (h == 1 && gated) break;
                    const half4_t v = {(half_t)sum[h][0], (half_t)sum[h][1], (half_t)sum[h][2], (half_t)sum[h][3]};
                    if (n + h * 16 + 4 <= end) {
                        __builtin_memcpy(row + n + h * 16, &v, 8);
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; e++)
                            if (n + h * 16 + e < end) row[n + h * 16 + e] = v[e];
                    }
                }
            }
        }
    }
}

// Whether an XCD, whose L2 is its own, takes its consecutive tiles along the rows of tiles or down the columns: the way that brings it
// fewer bytes of X and W, `x_row` and `w_col` of them a tile and k.  Down the columns always, as it was, every XCD read all of X: with
// this and the swizzle of X 150 shapes of M 65 to 2000 take 0.963 of their time, M = 1555, K = 1664, N = 656 15.0 us -> 10.6.
inline int wave_k_by_rows(int tiles_m, int tiles_n, double x_row, double w_col)
{
    const int tiles = (tiles_m * tiles_n + 7) / 8;
    auto bytes = [&](int along, double b_along, double b_across) { return std::min(along, tiles) * b_along + (tiles + along - 1) / along * b_across; };
    return bytes(tiles_n, w_col, x_row) < bytes(tiles_m, x_row, w_col) ? 1 : 0;
}

template <class P, int MP, int NP>
hipError_t launch_tile(WaveKArgs a, hipStream_t s)
{
    typedef WaveKCfg<P, MP, NP> C;
    a.tiles_m = (a.M + C::TM - 1) / C::TM;
    a.tiles_n = (a.N + C::TN - 1) / C::TN;
    // (geometry A by columns: a tile takes 16 or 32 bytes of a row of codes, and those beside it the rest of the line; so fp16 W, whose
    // tiles bring as much of it as of X: M = 1306, K = 3712, N = 1280 34.5 us, by rows 36.5)
    a.by_rows = P::kB ? wave_k_by_rows(a.tiles_m, a.tiles_n, C::TM * 2.0, C::TN * (double)P::CSZ / (P::kB ? P::VEC : 1)) : 0;
    const size_t lds = C::lds_bytes(P::kB ? (size_t)a.books * a.entries * P::VEC * 2 : C::kBooks);
    if (lds > 160 * 1024) return hipErrorInvalidValue;
    return launch_kernel(wave_k_kernel<P, MP, NP>, dim3((unsigned)(a.tiles_m * a.tiles_n)), dim3(C::kWaves * 64), lds, s, a);
}

// What a tile of mp x np pieces (10 * mp + np) costs, fitted to measurements: microseconds besides its units of 32 k (their
// first latency, the sum over the waves, the stores), cycles per unit on an idle device, how many more when every compute
// unit works, and by which share a unit takes longer with every doubling of X beyond 2 MB (geometry B).
struct WaveKTile {
    int tile = 0;
    double fixed_us = 0.0, idle_clk = 0.0, busy_clk = 0.0, wait = 0.05;
};

// Microseconds a launch is expected to take (a tenth off, either way): the tiles go over the compute units in rounds.
// wait: how much longer a unit takes than fitted.
inline double wave_k_tile_cost_us(const WaveKTile &t, int M, int K, int N, double bytes, double wait = 1.0)
{
    const int cus = device_cu_count(), tm = t.tile / 10 * 16, tn = t.tile % 10 * 16;
    const int64_t tiles = (int64_t)((M + tm - 1) / tm) * ((N + tn - 1) / tn);
    const int64_t rounds = (tiles + cus - 1) / cus;
    const double busy = (double)tiles / (double)(rounds * cus);
    const double tiles_us = (double)rounds * (t.fixed_us + (K / (double)kStepK) * (t.idle_clk + t.busy_clk * busy) * wait / 2100.0);
    const double memory_us = bytes / 4e6;
    return 2.0 + (tiles_us > memory_us ? tiles_us : memory_us);
}

struct WaveKPlan {
    int mp, np;
    double cost_us;
    bool wide = false;   // (geometry A) the kernel of vq_wave_k_a.hip
};

// whole units of K, rows of X in whole 16-byte chunks, offsets within 32 bits
inline bool wave_k_shape(const half_t *x, int M, int K, int N)
{
    return M >= 1 && N >= 1 && K >= kStepK && K % kStepK == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0 && (int64_t)128 * K * 2 < (int64_t)1 << 31 &&
           (int64_t)N * 2 * 64 < (int64_t)1 << 31;
}

}  // namespace

}  // namespace vq
