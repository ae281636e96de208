// Geometry A in the larger tiles of the wave-K scheme (vq_wave_k.h): K is dealt out to the four waves of a workgroup, each
// multiplies the whole tile for its own k, and the four partial tiles are added up at the end.
//
// What bounds it: the LDS, next to the matrix cores and, when every unit works, the L2.  With one wave on a SIMD nothing hides a
// wait but the wave itself, so that everything a step needs is dealt out between the MFMAs of the steps before it:
//
//   * A code makes two halves of W by one 4-byte gather.  64 of them in random banks take 6.8 cycles, and in distinct ones 2: the table
//     in the LDS has a row of the 64 banks for every code, with two copies of each of a pair's four codebooks for every lane of a
//     half wave (or one, and then 4 cycles), 64 KB whatever the tile's width.  A row and the lane's word in it make the
//     address by one v_perm.  The gathers of step s + 1 go out one by one while step s multiplies.
//   * Even and odd columns of Y are two pieces; the halves are put in order (v_perm, two instructions a pair of codes) one pair of pieces
//     ahead of its MFMAs.
//   * X, 16 cycles a KB into the LDS and 4 out of it, is read into registers in the last third (half) of the step before and leaves its
//     buffer free as the step begins: two steps of X in the LDS are one and a third on its way and one in use.
//   * Tiles of an XCD lie along the rows of tiles or down the columns, whichever brings it fewer bytes (wave_k_by_rows).
//
// 128 x 96, one tile alone: 0.53 us a step (48 MFMAs, 0.33 us by themselves) where the common kernel took 0.78.  M = 2048, K = 4096,
// Nc = 640: 38.6 -> 30.8 us; M = 1192, K = 2752, Nc = 480: 22.0 -> 14.3; M = 3925, K = 8128, Nc = 352: 88 -> 60.
// X straight from memory into the operands' registers, around the LDS, was measured first: a lane's 16 bytes lie in another row than
// its neighbours', 64 lines a load, 44 us.  X through registers into the LDS (ds_write): 37.
#include "vq_wave_k.h"

namespace vq {

namespace {

template <int MP, int NP>
struct WaveACfg {
    static constexpr int kWaves = 4, Q = NP / 2;
    static constexpr int TM = MP * 16, TN = NP * 16;
    static constexpr int kRowBytes = NP * 8;                                      // codes of a k-row
    static constexpr int kCodeLoads = (kStepK * kRowBytes + 1023) / 1024;         // direct loads of a step's codes
    static constexpr int kXBytes = MP * 1024, kCodeBytes = kCodeLoads * 1024;
    static constexpr int DC = 4;                                                  // steps of codes in the LDS per wave; two of X
    static constexpr int kTable = 256 * 256, kXBase = kTable, kCodeBase = kXBase + kWaves * 2 * kXBytes;
    static constexpr int kPassMP = pass_rows(MP, NP * kWaves);
    static constexpr int kSumBytes = kWaves * kPassMP * NP * 1024;
    static constexpr int kUse = kCodeBase + kWaves * DC * kCodeBytes;
    static constexpr int kLdsBytes = kUse > kSumBytes ? kUse : kSumBytes;
    static_assert((NP == 4 || NP == 6) && MP * NP <= 64 && kLdsBytes <= 160 * 1024, "pairs of pieces, accumulators in the AGPRs");
    // the table: the words of pair q in a row, from word first(q) on, two copies of each of the pair's four codebooks for every
    // lane of a quarter wave that gathers from it, or one
    static constexpr int words(int q) { return NP == 4 || q == 0 ? 32 : 16; }
    static constexpr int first(int q) { return q == 0 ? 0 : first(q - 1) + words(q - 1); }
};

template <int MP, int NP>
__global__ __launch_bounds__(256, 1) void wave_k_a_kernel(const half_t *__restrict__ x, const uint8_t *__restrict__ w, const half_t *__restrict__ cb,
                                                          half_t *__restrict__ y, int M, int K, int N, int tiles_m, int tiles_n, int by_rows)
{
    typedef WaveACfg<MP, NP> C;
    constexpr int Q = C::Q, kWaves = C::kWaves, kRowBytes = C::kRowBytes, DC = C::DC;
    extern __shared__ __align__(16) uint8_t smem[];
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int r16 = lane & 15, kg = lane >> 4;

    const int n_wg = tiles_m * tiles_n, xcd = blockIdx.x & 7;
    const int tile = xcd * (n_wg >> 3) + min(xcd, n_wg & 7) + ((int)blockIdx.x >> 3);
    const int along = by_rows ? tiles_n : tiles_m, line = tile / along, at_line = tile - line * along;
    const int tm = by_rows ? line : at_line, tn = by_rows ? at_line : line;
    const int m0 = tm * C::TM, n0 = tn * C::TN;
    const int n_step = (K / kStepK - wave + kWaves - 1) / kWaves;   // of this wave: wave, wave + kWaves, ...
    const uint32_t x_ring = C::kXBase + (uint32_t)wave * (2 * C::kXBytes), code_ring = C::kCodeBase + (uint32_t)wave * (DC * C::kCodeBytes);
    const int row_w = N / 2;

    // ---- the table's words, on their way ----------------------------------------------------------------
    // (a wave writes four rows at a time, lane by lane sixteen bytes: four words of one codebook)
    uint32_t words[16];
    {
        const int chunk = r16, q = NP == 4 ? chunk >> 3 : chunk < 8 ? 0 : (chunk >> 2) - 1;
        const int book = min(n0 / 8 + q * 4 + (chunk & 3), N / 8 - 1);   // (columns past the last: that one's codebook again)
        const uint32_t *src = reinterpret_cast<const uint32_t *>(cb) + (int64_t)book * 256 + wave * 64 + kg;
#pragma unroll
        for (int r = 0; r < 16; r++) words[r] = src[r * 4];
    }

    // ---- global -> LDS: codes; global -> registers -> LDS: X ---------------------------------------------
    uint32_t w_voff[C::kCodeLoads], x_voff[MP];
#pragma unroll
    for (int i = 0; i < C::kCodeLoads; i++) {
        const int slot = min(i * 64 + lane, kStepK * kRowBytes / 16 - 1), k = slot / (kRowBytes / 16), c = slot % (kRowBytes / 16);
        w_voff[i] = (uint32_t)(k * row_w + min(n0 / 2 + c * 16, row_w - 16) - n0 / 2);   // (columns past the last: that one's again)
    }
#pragma unroll
    for (int i = 0; i < MP; i++) {
        const int slot = i * 64 + lane, bank_row = slot >> 4, pos = (slot & 15) ^ wave_x_swizzle<1>(bank_row);
        x_voff[i] = (uint32_t)(((int64_t)(min(m0 + 4 * bank_row + (pos >> 2), M - 1) - m0) * K + (pos & 3) * 8) * 2);
    }
    const uint8_t *w_tile = w + n0 / 2;
    const uint8_t *x_tile = reinterpret_cast<const uint8_t *>(x + (int64_t)m0 * K);
    // (steps past the wave's last: that one again, into what nothing reads any more)
    auto k_of = [&](int t) { return (min(t, n_step - 1) * kWaves + wave) * kStepK; };
    auto issue_x = [&](int set, int i, const uint8_t *src) { load_to_lds_16(x_ring + set * C::kXBytes + i * 1024, x_voff[i], src); };
    auto issue_codes = [&](int i, uint32_t slot, const uint8_t *src) { load_to_lds_16(code_ring + slot * C::kCodeBytes + i * 1024, w_voff[i], src); };

    half8_t xs[2][MP];
    uint32_t raw[Q][8], code[Q][2];       // gathered pairs of halves, and the codes of the step behind theirs
    uint4_t ws[NP];
    typedef int int2v_t __attribute__((__vector_size__(2 * sizeof(int))));
    typedef __attribute__((address_space(3))) int2v_t lds_int2_t;
    typedef __attribute__((address_space(3))) const uint32_t lds_uint_t;
    // source lane (kg, s = r16) of the transposing read supplies k-row kg*8 + s/2, codes 8*(s%2) .. +7 of a group of 16
    const uint32_t code_rd = code_ring + (kg * 8 + (r16 >> 1)) * kRowBytes + (r16 & 1) * 8;
    const uint32_t x_rd = x_ring + wave_x_offset<1>(r16, kg);
    auto read_codes = [&](int q, uint32_t slot) {
        const int2v_t v = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_int2_t *)(smem + code_rd + slot * C::kCodeBytes + q * 16));
        code[q][0] = (uint32_t)v[0];
        code[q][1] = (uint32_t)v[1];
    };
    auto read_x = [&](int set, int i) { xs[set][i] = *reinterpret_cast<const half8_t *>(smem + x_rd + set * C::kXBytes + i * 1024); };
    // row of the code, word of the lane: one instruction
    const uint32_t word32 = (lane & 31) * 4, word16 = r16 * 4;
    auto gather = [&](int q, int t) {
        const uint32_t at = __builtin_amdgcn_perm(code[q][t >> 2], C::words(q) == 32 ? word32 : word16, 0x0c0c0400u + ((t & 3) << 8));
        raw[q][t] = *(lds_uint_t *)(at + C::first(q) * 4);
    };
    auto order = [&](int q, int t) {   // dword t / 2 of the even columns' operand, of the odd ones'
        ws[2 * q + (t & 1)][t >> 1] = __builtin_amdgcn_perm(raw[q][(t | 1)], raw[q][t & ~1], t & 1 ? 0x07060302 : 0x05040100);
    };

    float4_t acc[NP][MP];
#pragma unroll
    for (int j = 0; j < NP; j++)
#pragma unroll
        for (int i = 0; i < MP; i++) acc[j][i] = float4_t{0.f, 0.f, 0.f, 0.f};

    // ---- first steps --------------------------------------------------------------------------------------
    if (n_step > 0) {
#pragma unroll
        for (int d = 0; d < DC; d++) {
            const uint8_t *src = w_tile + (int64_t)k_of(d) * row_w;
#pragma unroll
            for (int i = 0; i < C::kCodeLoads; i++) issue_codes(i, d, src);
        }
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int i = 0; i < MP; i++) issue_x(t, i, x_tile + (int64_t)k_of(t) * 2);
    }
#pragma unroll
    for (int r = 0; r < 16; r++) *reinterpret_cast<uint4_t *>(smem + (wave * 64 + r * 4) * 256 + lane * 16) = uint4_t{words[r], words[r], words[r], words[r]};
    wait_vmcnt<0>();
    __syncthreads();

    if (n_step > 0) {
#pragma unroll
        for (int q = 0; q < Q; q++) read_codes(q, 0);
#pragma unroll
        for (int i = 0; i < MP; i++) read_x(0, i);
#pragma unroll
        for (int q = 0; q < Q; q++) {
#pragma unroll
            for (int t = 0; t < 8; t++) gather(q, t);
            read_codes(q, 1);
        }
#pragma unroll
        for (int t = 0; t < 8; t++) order(0, t);
        uint32_t c_slot = 0;   // of this step's codes
        // one step: its MFMAs pair of pieces by pair of pieces, and between them what the steps behind it need
        auto step = [&](auto set_const, int u) {
            constexpr int set = decltype(set_const)::value, kLater = MP >= 8 ? 1 : 0;   // (between the gathers)
            const uint32_t c_next2 = (c_slot + 2) % DC;
            const uint8_t *x_src = x_tile + (int64_t)k_of(u + 2) * 2, *w_src = w_tile + (int64_t)k_of(u + DC) * row_w;
#pragma unroll
            for (int q = 0; q < Q; q++) {
                asm volatile("s_nop 1" ::: "memory");
#pragma unroll
                for (int n = 0; n < 2 * MP; n++) {
                    const int i = n >> 1, h = n & 1;
                    __builtin_amdgcn_sched_barrier(0);
                    mfma_in_place(acc[2 * q + h][i], __builtin_bit_cast(half8_t, ws[2 * q + h]), xs[set][i]);
                    __builtin_amdgcn_sched_barrier(0);
                    // the next step's gathers of this pair, then the codes of the step behind that
#pragma unroll
                    for (int t = n * 8 / (2 * MP); t < (n + 1) * 8 / (2 * MP); t++) gather(q, t);
                    // X of the step behind the next and the codes of the fourth: this step's X is in the registers piece by piece
                    if (q == 0 && h == 1) issue_x(set, i, x_src);
                    if (q == 0 && n >= 2 * MP - C::kCodeLoads) issue_codes(n - 2 * MP + C::kCodeLoads, c_slot, w_src);
                    if (q == 0 && n == 2 * MP - 1) {
                        wait_vmcnt<2 * (MP + C::kCodeLoads)>();   // the codes of step u + 2 have landed
                        asm volatile("" ::: "memory");
                    }
                    if (q == Q - 2 && n == 2 * MP - 1) {
                        wait_vmcnt<MP + C::kCodeLoads>();         // X of the next step has
                        asm volatile("" ::: "memory");
                    }
                    if (n == 2 * MP - 1) read_codes(q, c_next2);
                    // the next pair's operands: of this step, or of the next one
#pragma unroll
                    for (int t = (n + kLater) * 8 / (2 * MP); t < (n + kLater + 1) * 8 / (2 * MP); t++)
                        if (t < 8) order(q + 1 < Q ? q + 1 : 0, t);
                    if (q == Q - 1 && h == 0) read_x(set ^ 1, i);
                }
            }
            c_slot = (c_slot + 1) % DC;
        };
        int u = 0;
        for (; u + 1 < n_step; u += 2) {
            step(std::integral_constant<int, 0>{}, u);
            step(std::integral_constant<int, 1>{}, u + 1);
        }
        if (u < n_step) step(std::integral_constant<int, 0>{}, u);
    }
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");   // the last MFMAs have left the pipe
    hold_accumulators(acc);
    wait_vmcnt<0>();                                      // nothing is on its way into the LDS any more

    // ---- the sum over the waves: a piece is 1 KB, float4 by lane; a wave takes pairs of pieces of a row of pieces
    constexpr int PM = C::kPassMP;
#pragma unroll
    for (int pass = 0; pass < MP / PM; pass++) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < PM; i++)
#pragma unroll
            for (int j = 0; j < NP; j++)
                *reinterpret_cast<float4_t *>(smem + ((wave * PM + i) * NP + j) * 1024 + lane * 16) = acc[j][pass * PM + i];
        __syncthreads();
        for (int pair = wave; pair < PM * Q; pair += kWaves) {
            const int i = pair / Q, q = pair % Q;
            const int m = m0 + (pass * PM + i) * 16 + r16, n = n0 + q * 32 + kg * 8;
            float4_t sum[2];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const uint8_t *src = smem + (i * NP + 2 * q + h) * 1024 + lane * 16;
                sum[h] = *reinterpret_cast<const float4_t *>(src);
#pragma unroll
                for (int v = 1; v < kWaves; v++) sum[h] += *reinterpret_cast<const float4_t *>(src + v * (PM * NP * 1024));
            }
            // the even columns and the odd ones: eight columns in a row
            half8_t v;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                v[2 * e] = (half_t)sum[0][e];
                v[2 * e + 1] = (half_t)sum[1][e];
            }
            if (m < M && n < N) __builtin_memcpy(y + (int64_t)m * N + n, &v, 16);
        }
    }
}

}  // namespace

hipError_t launch_wave_k_a_wide(const ProblemA &p, int tile, hipStream_t s)
{
    auto launch = [&](auto mp, auto np) {
        typedef WaveACfg<mp(), np()> C;
        const int N = 2 * p.Nc, tiles_m = (p.M + C::TM - 1) / C::TM, tiles_n = (N + C::TN - 1) / C::TN;
        return launch_kernel(wave_k_a_kernel<mp(), np()>, dim3((unsigned)(tiles_m * tiles_n)), dim3(256), C::kLdsBytes, s, p.x, p.w, p.cb, p.y, p.M, p.K, N, tiles_m, tiles_n,
                             wave_k_by_rows(tiles_m, tiles_n, C::TM * 2.0, C::TN * 0.5));
    };
    using std::integral_constant;
    switch (tile) {
    case 44: return launch(integral_constant<int, 4>{}, integral_constant<int, 4>{});
    case 64: return launch(integral_constant<int, 6>{}, integral_constant<int, 4>{});
    case 66: return launch(integral_constant<int, 6>{}, integral_constant<int, 6>{});
    case 84: return launch(integral_constant<int, 8>{}, integral_constant<int, 4>{});
    case 86: return launch(integral_constant<int, 8>{}, integral_constant<int, 6>{});
    default: return hipErrorInvalidValue;
    }
}

}  // namespace vq
