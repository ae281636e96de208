// Prefill kernel with tiles of 128, 160, 192 or 224 rows by 128 columns, one workgroup to a compute unit: between the heights of
// the other tiles (128 and 256) a band of rows that is not full costs as much as one that is, and with the 128x128 tile of
// vq_prefill_small.hip two workgroups share a unit's LDS, which bounds it.
//
// What bounds this one is the LDS too: a step of 32 k reads MP + 4 KB of operands per wave for 4 * MP MFMAs, and what the four
// waves read, the direct loads write and the codes take is 390 cycles where the MFMAs of 128 rows are 256 (192 rows: 484 to 384).
// With 8-bit codes and one codebook to a tile the LDS holds the codebook as a table of copies - half a row of the 64 banks per
// entry, 8 copies of an 8-vector or 16 of a 4-vector, every lane gathering its own - in which few gathers meet in a bank; whole
// rows (64 KB) gained no more.  More stages of X ahead than three gained nothing, two cost a fifth.
// 64 tiles of 128 rows, K = 4096: 29.2 us (128x128 two to a unit) -> 27.1; M = 320, K = 4096, N = 11008 (two tiles of 160 rows by 86):
// 46.5 -> 32.1, with 16-bit codes of 512 8-vectors 50.0 -> 35.6, of 4096 4-vectors 76.5 -> 41.0; M = 640, K = N = 8192 94.6 -> 74.8.
//
// The frame is vq_prefill_small.hip's: 256 threads (2x2 waves), MP*16 x 64 per wave, X (whole 128-byte lines) and code tiles
// global -> LDS directly, three stages ahead, accumulators pinned in the AGPRs, every MFMA fenced and everything else dealt
// out between them, an operand of W gathered whole; one barrier per stage.  K in multiples of 64 (HALF: 8-vectors with 8-bit
// codes, a last code tile of one stage).  The sums are those of the other tiles, in the same order: the same bits.
#include "vq_prefill_common.h"

#include <cmath>
#include <type_traits>

namespace vq {

namespace {

constexpr int MNP = 4, MBN = 2 * MNP * 16;   // pieces of a wave and columns of a tile
constexpr int kMidEntries = 256, kCopyRow = 128;   // entries of a table of copies, and the bytes of copies of each
constexpr int kMidStages = 4;                  // X stages in the LDS

template <int VEC, typename CodeT, int MP_>
struct MidCfg {
    typedef PrefillCfg<VEC, CodeT> C;
    static constexpr int MP = MP_, NS = kMidStages, D = NS - 1;
    static constexpr int BM = 2 * MP * 16, WM = MP * 16;
    static constexpr int kStage = BM * kStageK * 2;
    static constexpr int NC = C::STAGES == 1 ? NS : (NS - 1) / 2 + 2;   // code tiles in the LDS
    static constexpr int kTile = C::CH * MBN * 16;                      // [chunk][row][16 bytes]
    static constexpr int kCodeBase = NS * kStage, kTable = kCodeBase + NC * kTile;
    static_assert(kMidEntries * VEC * 2 <= kStage, "a stage holds the plain copy of the codebook");
};

template <int VEC, typename CodeT, int MP, bool COPIES, bool HALF>
__global__ __launch_bounds__(kThreads, 1) void prefill_mid_kernel(const half_t *__restrict__ x, const CodeT *__restrict__ codes,
                                                                  const half_t *__restrict__ cb, half_t *__restrict__ y,
                                                                  const half_t *__restrict__ bias, int M, int K, int N, int entries,
                                                                  int rows_per_cb, int tiles_m, int tiles_n, int books, int gated)
{
    typedef MidCfg<VEC, CodeT, MP> G;
    typedef PrefillCfg<VEC, CodeT> C;
    constexpr int NS = G::NS, D = G::D, NC = G::NC;
    extern __shared__ __align__(16) uint8_t smem[];
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int wm = wave >> 1, wn = wave & 1;
    const int r16 = lane & 15, kg = lane >> 4;
    const int J = K / VEC;

    // Workgroup ids are dealt round-robin to the 8 XCDs: an XCD takes consecutive tiles, those over the same columns of Y next to
    // each other.
    const int n_wg = tiles_m * tiles_n, xcd = blockIdx.x & 7;
    const int wg = xcd * (n_wg >> 3) + min(xcd, n_wg & 7) + ((int)blockIdx.x >> 3);
    const int tm = wg % tiles_m, tn = wg / tiles_m;
    const int m0 = tm * G::BM, n0 = tn * MBN;
    const int n_super = (K + C::K_SUPER - 1) / C::K_SUPER;
    const int n_stage = n_super * C::STAGES - (HALF ? 1 : 0);

    // ---- staging: global -> LDS directly (as in prefill_small_kernel) -----------------------------
    uint32_t x_voff[MP];
#pragma unroll
    for (int i = 0; i < MP; i++) {
        const int slot = (4 * i + wave) * 64 + lane;
        const int bank_row = slot >> 4;
        const int v = (slot & 15) ^ (bank_row & 15);
        const int row = 2 * bank_row + (v >> 3), cc = v & 7;
        x_voff[i] = (uint32_t)(((int64_t)(min(m0 + row, M - 1) - m0) * K + cc * 8) * 2);
    }
    const half_t *x_tile = x + (int64_t)m0 * K;
    auto issue_x = [&](int i, int buf, const half_t *xb) { load_to_lds_16(buf * G::kStage + (4 * i + wave) * 1024, x_voff[i], xb); };
    const uint8_t *code_tile = reinterpret_cast<const uint8_t *>(codes + (int64_t)n0 * J);
    const uint32_t code_voff = (uint32_t)(min(wn * 64 + lane, N - 1 - n0) * J * C::CSZ);
    constexpr int kSuperBytes = C::K_SUPER / VEC * C::CSZ;   // of one row's codes per code tile
    auto code_at = [&](int i) { return code_tile + (int64_t)min(i, n_super - 1) * kSuperBytes - (HALF && i >= n_super - 1 ? 8 : 0); };
    auto issue_codes = [&](int c, int cbuf, const uint8_t *cbase) {
        load_to_lds_16(G::kCodeBase + cbuf * G::kTile + c * (MBN * 16) + wn * 1024, code_voff + c * 16, cbase);
    };
    const half_t *x_ahead = x_tile + min(D, n_stage - 1) * kStageK;
    const uint8_t *c_ahead = code_at(D / C::STAGES);

    float4_t acc[MNP][MP];
#pragma unroll
    for (int j = 0; j < MNP; j++)
#pragma unroll
        for (int i = 0; i < MP; i++) acc[j][i] = float4_t{0.f, 0.f, 0.f, 0.f};

    // ---- operand reads ------------------------------------------------------------------------
    int x_rd[2][2];
#pragma unroll
    for (int par = 0; par < 2; par++)
#pragma unroll
        for (int s = 0; s < 2; s++) x_rd[par][s] = x_offset(wm * G::WM + par * 16 + r16, s * 4 + kg);
    const uint32_t code_rd = G::kCodeBase + (wn * 64 + r16) * 16 + kg * C::RB;
    constexpr uint32_t kEntry = COPIES ? kCopyRow : VEC * 2;   // bytes from entry to entry
    const int g_first = n0 / rows_per_cb;
    uint32_t book[MNP];   // the table of W row j*16 + r16 of the wave tile: its codebook, or the lane's copy
#pragma unroll
    for (int j = 0; j < MNP; j++)
        book[j] = G::kTable + (COPIES ? (uint32_t)(lane * (VEC * 2) & (kCopyRow - 1))
                                      : (uint32_t)((min(n0 + wn * 64 + j * 16 + r16, N - 1) / rows_per_cb - g_first) * entries * (VEC * 2)));

    half8_t wp[2][MNP], xp[2][MP];
    uint32_t cr[MNP];  // the codes behind the W pieces of the step whose gathers come next
    auto load_x1 = [&](int set, int i, int buf, int s) {
        xp[set][i] = *reinterpret_cast<const half8_t *>(smem + buf * G::kStage + x_rd[i & 1][s] + (i >> 1) * 4096);
    };
    auto load_c1 = [&](int j, int cbuf, int shift, int t, int s) {
        const int pos = (t % C::STAGES) * 2 * C::HALF + s * C::HALF;
        cr[j] = read_codes<C::RB>(smem + code_rd + cbuf * G::kTile + shift + (pos / 16) * (MBN * 16) + j * 256 + pos % 16);
    };
    auto load_w = [&](int set, int j) {
        if constexpr (VEC == 8) {
            wp[set][j] = *reinterpret_cast<const half8_t *>(smem + book[j] + cr[j] * kEntry);
        } else {
            static_assert(VEC == 4, "4- or 8-vectors");
            const uint32_t c_lo = cr[j] & (C::CSZ == 1 ? 0xffu : 0xffffu), c_hi = cr[j] >> (8 * C::CSZ);
            const half4_t lo = *reinterpret_cast<const half4_t *>(smem + book[j] + c_lo * kEntry);
            const half4_t hi = *reinterpret_cast<const half4_t *>(smem + book[j] + c_hi * kEntry);
            wp[set][j] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        }
    };

    // ---- prologue: the codebooks, stages 0..D-1 -----------------------------------------------------
    // Loads complete in the order they were issued, so one count serves all of them.
    auto loads_of = [](int stage_mod) constexpr { return MP + (stage_mod % C::STAGES == 0 ? C::CH : 0); };
    {
        // (copies: a plain one first, into the last X buffer, which is free until stage 0 issues the loads of stage D)
        const uint8_t *src = reinterpret_cast<const uint8_t *>(cb + (int64_t)g_first * entries * VEC);
        const int n16 = books * entries * (VEC * 2) / 16, dst = COPIES ? D * G::kStage : G::kTable;
        const int last16 = (int)((int64_t)((N + rows_per_cb - 1) / rows_per_cb - g_first) * entries * (VEC * 2) / 16) - 1;   // past the last codebook: its last 16 bytes again
        for (int i0 = wave * 64; i0 < n16; i0 += kThreads) load_to_lds_16(dst + i0 * 16, (uint32_t)min(i0 + lane, last16) * 16u, src);
    }
#pragma unroll
    for (int d = 0; d < D; d++) {
        if (d % C::STAGES == 0) {
#pragma unroll
            for (int c = 0; c < C::CH; c++) issue_codes(c, (d / C::STAGES) % NC, code_at(d / C::STAGES));
        }
#pragma unroll
        for (int i = 0; i < MP; i++) issue_x(i, d, x_tile + min(d, n_stage - 1) * kStageK);
    }
    {
        constexpr int in_flight = [&]() constexpr {
            int n = 0;
            for (int d = 1; d < D; d++) n += loads_of(d);
            return n;
        }();
        wait_vmcnt<in_flight>();   // the codebooks and stage 0 have landed
    }
    __syncthreads();
    if constexpr (COPIES) {
        // a thread an entry, its pieces of 16 bytes in an order that neighbouring entries do not share
        static_assert(kThreads == kMidEntries, "a thread an entry");
        const uint8_t *src = smem + D * G::kStage + min(tid, entries - 1) * (VEC * 2);
        uint4_t piece;
        if constexpr (VEC == 8) {
            piece = *reinterpret_cast<const uint4_t *>(src);
        } else {
            const uint2_t v = *reinterpret_cast<const uint2_t *>(src);
            piece = uint4_t{v[0], v[1], v[0], v[1]};
        }
        const uint32_t at = G::kTable + tid * kCopyRow + (tid * 16 & (kCopyRow - 1));
#pragma unroll
        for (int i = 0; i < kCopyRow / 16; i++) *reinterpret_cast<uint4_t *>(smem + (at ^ (i * 16))) = piece;
        __syncthreads();
    }

    int buf = 0, cbuf = 0;
    // step 0 of stage 0: all of its operands; then the codes of step 1
#pragma unroll
    for (int j = 0; j < MNP; j++) load_c1(j, cbuf, 0, 0, 0);
#pragma unroll
    for (int j = 0; j < MNP; j++) load_w(0, j);
#pragma unroll
    for (int i = 0; i < MP; i++) load_x1(0, i, buf, 0);
#pragma unroll
    for (int j = 0; j < MNP; j++) load_c1(j, cbuf, 0, 0, 1);

#define VQ_FENCE __builtin_amdgcn_sched_barrier(0)
    auto stage_body = [&](int super, auto t_const) {
        constexpr int t = decltype(t_const)::value;
        const int stage = super * C::STAGES + t;
        const int buf_next = buf + 1 == NS ? 0 : buf + 1;
        // the loads of stage+D go into the buffer stage-1 was read from
        const int tgt_buf = buf == 0 ? NS - 1 : buf - 1;
        constexpr bool tgt_codes = (t + D) % C::STAGES == 0;
        constexpr int d_super = (t + D) / C::STAGES;
        const int tgt_cbuf = (cbuf + d_super) % NC;
        constexpr bool same_super = t + 1 < C::STAGES;
        const int cbuf_n = same_super ? cbuf : (cbuf + 1 == NC ? 0 : cbuf + 1);
        constexpr int t_n = same_super ? t + 1 : 0;
        const int cshift_n = HALF && super + (same_super ? 0 : 1) >= n_super - 1 ? 8 : 0;
        // Publish stage+1: only what the stages behind it bring along may still be in flight.
        constexpr int in_flight = [&]() constexpr {
            int n = 0;
            for (int d = 2; d < D; d++) n += loads_of(t + d);
            return n;
        }();
        wait_vmcnt<in_flight>();
        __syncthreads();
        VQ_FENCE;
        // A step: 4 * MP MFMAs of set `step`; behind them one by one the gathers and X reads of the next step into the other set, the
        // codes of the step after that, and this step's share of the stage's global loads.
#pragma unroll
        for (int step = 0; step < 2; step++) {
            constexpr int first_half = (MP + 1) / 2;   // X loads of step 0
#pragma unroll
            for (int m = 0; m < MNP * MP; m++) {
                const int j = m / MP, i = m % MP;
                mfma_in_place(acc[j][i], wp[step][j], xp[step][i]);
                VQ_FENCE;
                if (m < MNP) {
                    load_w(step ^ 1, m);
                } else if (m < MNP + MP) {
                    if (step == 0) load_x1(1, m - MNP, buf, 1);
                    else load_x1(0, m - MNP, buf_next, 0);
                } else if (m < 2 * MNP + MP) {
                    if (step == 0) load_c1(m - MNP - MP, cbuf_n, cshift_n, t_n, 0);
                    else load_c1(m - MNP - MP, cbuf_n, cshift_n, t_n, 1);
                } else {
                    const int q = m - 2 * MNP - MP, n_x = step == 0 ? first_half : MP - first_half;
                    if (q < n_x) issue_x(step * first_half + q, tgt_buf, x_ahead);
                    else if (tgt_codes && q == first_half && step < C::CH) issue_codes(step, tgt_cbuf, c_ahead);
                }
                VQ_FENCE;
            }
            static_assert(MNP * MP > 2 * MNP + MP + first_half && C::CH <= 2, "a step has room for everything");
        }
        x_ahead += stage + D + 1 < n_stage ? kStageK : 0;
        if ((t + D + 1) % C::STAGES == 0) {
            const int next = (stage + D + 1) / C::STAGES;
            c_ahead += next < n_super ? (HALF && next == n_super - 1 ? kSuperBytes - 8 : kSuperBytes) : 0;
        }
        buf = buf_next;
    };
    const int n_whole = n_super - (HALF ? 1 : 0);  // (at least one)
    int super = 0;
    do {
        stage_body(super, std::integral_constant<int, 0>{});
        if constexpr (C::STAGES == 2) stage_body(super, std::integral_constant<int, 1>{});
        cbuf = cbuf + 1 == NC ? 0 : cbuf + 1;
    } while (++super < n_whole);
    if constexpr (HALF) {
        // (the MFMAs are opaque to the compiler: let them leave the pipe ahead of the peeled stage, where it may copy accumulators)
        asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
        VQ_FENCE;
        stage_body(n_super - 1, std::integral_constant<int, 0>{});
    }
#undef VQ_FENCE
    wait_vmcnt<0>();   // the clamped loads still in flight
    __syncthreads();
    // the last MFMAs must have left the pipe before the accumulators are read
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
    hold_accumulators(acc);

    // ---- epilogue: lane holds Y[m = i*16 + r16][n = j*16 + 4*kg + 0..3] of its wave tile -------------
    const int m_wave = m0 + wm * G::WM, n_wave = n0 + wn * 64;
    if (gated) {
        if (bias) store_gated<MNP, MP, true>(acc, y, bias, M, N, N, m_wave, n_wave, r16, kg);
        else store_gated<MNP, MP, false>(acc, y, bias, M, N, N, m_wave, n_wave, r16, kg);
        return;
    }
    auto epilogue = [&](auto has_bias_const) {
        constexpr bool HB = decltype(has_bias_const)::value;
        constexpr int kPitch = 144;  // 64 fp16 + 16 bytes: rows land in different banks
        uint8_t *stage_out = smem + wave * (G::WM * kPitch);
#pragma unroll
        for (int j = 0; j < MNP; j++) {
            float bj[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int n = n_wave + j * 16 + 4 * kg + e;
                bj[e] = HB && n < N ? (float)bias[n] : 0.f;
            }
#pragma unroll
            for (int i = 0; i < MP; i++)
                *reinterpret_cast<half4_t *>(stage_out + (i * 16 + r16) * kPitch + (j * 16 + 4 * kg) * 2) = round4<HB>(acc[j][i], bj);
        }
#pragma unroll
        for (int it = 0; it < G::WM / 8; it++) {
            const int row = it * 8 + (lane >> 3), c = lane & 7;
            const uint4_t v = *reinterpret_cast<const uint4_t *>(stage_out + row * kPitch + c * 16);
            const int m = m_wave + row, n = n_wave + c * 8;
            if (m < M) store_eight(y + (int64_t)m * N + n, v, N - n, (N & 7) == 0);
        }
    };
    if (bias) epilogue(std::true_type{});
    else epilogue(std::false_type{});
}

// 8-bit codes (at most 256 entries) and one codebook to a tile
template <typename CodeT>
bool mid_copies(const ProblemB &p)
{
    return sizeof(CodeT) == 1 && codebooks_per_tile(p, MBN) == 1;
}

template <int VEC, typename CodeT, int MP>
size_t mid_lds_bytes(const ProblemB &p)
{
    return MidCfg<VEC, CodeT, MP>::kTable + (mid_copies<CodeT>(p) ? (size_t)kMidEntries * kCopyRow : copied_bytes((size_t)codebooks_per_tile(p, MBN) * p.entries * VEC * 2));
}

template <int VEC, typename CodeT, int MP>
hipError_t launch_mid_typed(const ProblemB &p, hipStream_t s)
{
    typedef MidCfg<VEC, CodeT, MP> G;
    typedef PrefillCfg<VEC, CodeT> C;
    const size_t lds = mid_lds_bytes<VEC, CodeT, MP>(p);
    if (lds > kLdsLimit) return hipErrorInvalidValue;
    const int tiles_m = (p.M + G::BM - 1) / G::BM, tiles_n = (p.N + MBN - 1) / MBN;
    constexpr bool can_half = C::STAGES == 2, can_copy = sizeof(CodeT) == 1;
    const bool half = p.K % C::K_SUPER != 0, copies = mid_copies<CodeT>(p);
    auto kern = copies ? (half ? prefill_mid_kernel<VEC, CodeT, MP, can_copy, can_half> : prefill_mid_kernel<VEC, CodeT, MP, can_copy, false>)
                       : (half ? prefill_mid_kernel<VEC, CodeT, MP, false, can_half> : prefill_mid_kernel<VEC, CodeT, MP, false, false>);
    return launch_kernel(kern, dim3((unsigned)(tiles_m * tiles_n)), dim3(kThreads), lds, s, p.x, static_cast<const CodeT *>(p.codes), p.cb, p.y,
                         p.bias, p.M, p.K, p.N, p.entries, p.rows_per_cb, tiles_m, tiles_n, codebooks_per_tile(p, MBN), p.gated ? 1 : 0);
}

// calls f with the format's vector length and code type; false where there is none
template <class F>
bool with_mid_format(const ProblemB &p, F f)
{
    using std::integral_constant;
    const bool u8 = p.code_bits == 8;
    if (p.vec == 8) {
        if (u8) f(integral_constant<int, 8>{}, uint8_t{});
        else f(integral_constant<int, 8>{}, uint16_t{});
    } else if (p.vec == 4) {
        if (u8) f(integral_constant<int, 4>{}, uint8_t{});
        else f(integral_constant<int, 4>{}, uint16_t{});
    } else {
        return false;
    }
    return true;
}

}  // namespace

// whole code tiles along K (or a last one of one stage), a tile's offsets within 32 bits
bool prefill_mid_supports(const ProblemB &p)
{
    if (p.M < 1 || p.N < 1 || p.K < 1 || p.packed || p.k_x != p.K || ((size_t)p.entries * p.vec * 2) % 16 != 0) return false;
    bool ok = false;
    with_mid_format(p, [&](auto vec, auto code) {
        typedef decltype(code) CodeT;
        typedef PrefillCfg<vec(), CodeT> C;
        ok = p.K >= C::K_SUPER && (p.K % C::K_SUPER == 0 || (C::STAGES == 2 && prefill_k_ok<vec(), CodeT>(p.K))) &&
             (int64_t)MBN * (p.K / vec()) * (int64_t)sizeof(CodeT) < ((int64_t)1 << 31) && (int64_t)224 * p.K * 2 < ((int64_t)1 << 32) &&
             mid_lds_bytes<vec(), CodeT, 4>(p) <= kLdsLimit;
    });
    return ok;
}

// What a tile costs, fitted to 500 shapes of M 90 to 2500 (3 % off): microseconds besides its stages, a stage's on an idle
// device, how much more when every unit works, and by which share a stage takes longer with every doubling of X beyond 2 MB.
struct MidTile {
    double fixed_us, idle_us, busy_us, wait;
};
// [rows / 32 - 4] of 8-vectors and 4-vectors with a table of copies, and without (16-bit codes, several codebooks to a tile)
constexpr MidTile kMidTiles[4][4] = {{{3.1, 0.327, 0.083, 0.035}, {3.4, 0.377, 0.113, 0.022}, {4.0, 0.431, 0.128, 0.020}, {4.4, 0.491, 0.143, 0.018}},
                                     {{3.2, 0.437, 0.078, 0.011}, {3.6, 0.496, 0.082, 0.009}, {4.0, 0.553, 0.094, 0.014}, {4.3, 0.628, 0.115, 0.012}},
                                     {{2.8, 0.400, 0.075, 0.017}, {3.6, 0.446, 0.087, 0.017}, {4.0, 0.502, 0.111, 0.017}, {4.5, 0.566, 0.123, 0.015}},
                                     {{3.7, 0.444, 0.071, 0.018}, {4.1, 0.499, 0.082, 0.021}, {4.6, 0.589, 0.060, 0.028}, {5.1, 0.637, 0.078, 0.030}}};

// The tile that is expected to be fastest, and its time: a round over the units or two.  (In more rounds the heights no longer
// matter, and the large tiles spend less energy, which is what bounds a device at full work: of 48 shapes in three rounds and more
// a third were faster here, by 1 %; of 389 in one round 98 %, by 9 %, of 61 in two 64 %, by 6 %, and those are asked for 10 %.)
MidPlan prefill_mid_plan(const ProblemB &p)
{
    MidPlan best = {0, 1e30};
    if (!prefill_mid_supports(p)) return best;
    const int cus = device_cu_count(), forced = (int)tuning().prefill_mid_force;
    if (forced == 1) return best;
    const bool copies = p.code_bits == 8 && mid_copies<uint8_t>(p);
    const double octaves = std::fmin(3.0, std::fmax(0.0, std::log2(2.0 * p.M * p.K / 2e6)));
    const int tiles_n = (p.N + MBN - 1) / MBN;
    for (int h = 0; h < 4; h++) {
        const int rows = 128 + 32 * h;
        if (forced > 1 && rows != forced) continue;
        size_t lds = 0;
        with_mid_format(p, [&](auto vec, auto code) {
            typedef decltype(code) CodeT;
            lds = h == 0   ? mid_lds_bytes<vec(), CodeT, 4>(p)
                  : h == 1 ? mid_lds_bytes<vec(), CodeT, 5>(p)
                  : h == 2 ? mid_lds_bytes<vec(), CodeT, 6>(p)
                           : mid_lds_bytes<vec(), CodeT, 7>(p);
        });
        if (lds > kLdsLimit) continue;
        const int64_t tiles = (int64_t)((p.M + rows - 1) / rows) * tiles_n, full = tiles / cus, rem = tiles % cus;
        if (tiles > 2 * cus && forced <= 1) continue;
        const MidTile &t = kMidTiles[(p.vec == 8 ? 0 : 1) + (copies ? 0 : 2)][h];
        const double stages = p.K / 64.0 * (1.0 + t.wait * octaves);
        double us = 2.0 + (double)full * (t.fixed_us + stages * (t.idle_us + t.busy_us));
        if (rem) us += t.fixed_us + stages * (t.idle_us + t.busy_us * (double)rem / cus);
        if (tiles > cus) us *= 1.1;
        if (us < best.cost_us) best = {rows, us};
    }
    return best;
}

hipError_t launch_prefill_mid_b(const ProblemB &p, hipStream_t s, int rows)
{
    if (!prefill_mid_supports(p)) return hipErrorInvalidValue;
    hipError_t e = hipErrorInvalidValue;
    with_mid_format(p, [&](auto vec, auto code) {
        typedef decltype(code) CodeT;
        switch (rows) {
        case 128: e = launch_mid_typed<vec(), CodeT, 4>(p, s); break;
        case 160: e = launch_mid_typed<vec(), CodeT, 5>(p, s); break;
        case 192: e = launch_mid_typed<vec(), CodeT, 6>(p, s); break;
        case 224: e = launch_mid_typed<vec(), CodeT, 7>(p, s); break;
        default: break;
        }
    });
    return e;
}

}  // namespace vq
