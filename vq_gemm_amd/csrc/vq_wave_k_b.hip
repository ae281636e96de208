// The kernels of vq_wave_k.h for geometry B.
#include "vq_wave_k.h"

#include <cmath>

namespace vq {

namespace {

// A format, and what its kernels' units are: two steps of K - whole 128-byte lines of X, the codes of both steps in one
// read - where the LDS holds two such units of eight waves beside the codebooks, one step for the larger tiles and the
// larger tables.
template <int VEC_, typename CodeT_>
struct Format {
    static constexpr int VEC = VEC_, CSZ = (int)sizeof(CodeT_);
    template <int MP, int NP>
    using Wave = WaveB<VEC_, CodeT_, ((MP * NP > 16 || (CSZ == 2 && MP >= 4)) ? 1 : 2)>;
    // Tiles of up to 32 rows gather more than they read of X: with a table of copies, 64 KB of the LDS that their units leave,
    // the gathers' bank conflicts go, M = 128, K = N = 4096 9.5 -> 9.0 us, M = 16, K = 2048, N = 11008 6.7 -> 6.0, tiles of
    // 32 x 128 14.5 -> 12.0; 32 x 16 gathers too little, equal.  Taller ones read X twice as long as they gather and would keep half the units in flight: 64 x 64
    // with 32 KB of copies 13.7 -> 15.0.  16-bit codes of up to 512 entries (two stages of 256) in tiles wider than tall, with half as many
    // copies: M = 16, K = 4096, N = 11008 7.5 -> 6.8, M = 32, K = 4096, N = 11008 8.5 -> 8.35, tiles of 16 x 64 8.6 -> 7.4, 4-vectors
    // 2 to 7 %; 16 x 16 and 32 x 32 gather too little (M = 5, K = 8192, N = 4096 7.0 -> 7.5).
    template <int MP, int NP>
    static constexpr bool kHasCopies = MP <= 2 && (CSZ == 1 ? NP >= MP : NP > MP) && WaveKCfg<WaveB<VEC_, CodeT_, Wave<MP, NP>::S, true>, MP, NP>::kExists;
    template <int MP, int NP>
    using Copies = WaveB<VEC_, CodeT_, Wave<MP, NP>::S, true>;
};

// calls f with the pieces of the tile (10 * rows + columns), as types
template <class F>
void with_tile(int tile, F f)
{
    using std::integral_constant;
    switch (tile) {
    case 12: f(integral_constant<int, 1>{}, integral_constant<int, 2>{}); break;
    case 14: f(integral_constant<int, 1>{}, integral_constant<int, 4>{}); break;
    case 18: f(integral_constant<int, 1>{}, integral_constant<int, 8>{}); break;
    case 22: f(integral_constant<int, 2>{}, integral_constant<int, 2>{}); break;
    case 24: f(integral_constant<int, 2>{}, integral_constant<int, 4>{}); break;
    case 44: f(integral_constant<int, 4>{}, integral_constant<int, 4>{}); break;
    case 48: f(integral_constant<int, 4>{}, integral_constant<int, 8>{}); break;
    case 34: f(integral_constant<int, 3>{}, integral_constant<int, 4>{}); break;
    case 54: f(integral_constant<int, 5>{}, integral_constant<int, 4>{}); break;
    case 64: f(integral_constant<int, 6>{}, integral_constant<int, 4>{}); break;
    case 28: f(integral_constant<int, 2>{}, integral_constant<int, 8>{}); break;
    case 11: f(integral_constant<int, 1>{}, integral_constant<int, 1>{}); break;
    case 21: f(integral_constant<int, 2>{}, integral_constant<int, 1>{}); break;
    case 13: f(integral_constant<int, 1>{}, integral_constant<int, 3>{}); break;
    case 23: f(integral_constant<int, 2>{}, integral_constant<int, 3>{}); break;
    default: break;
    }
}

// Whether the tile's kernel with a table of copies serves the problem: at most as many entries, tiles that meet one codebook.
template <class F, int MP, int NP>
bool takes_copies(const ProblemB &p)
{
    // (16-bit codes, 16 rows: a longer K wants the units that the copies take the room of: M = 16, N = 11008, K = 8192 9.73 -> 9.15, 9216
    // 10.32 -> 10.27, 10240 12.4 -> 12.9, 16384 16.8 -> 17.4.)
    if constexpr (F::template kHasCopies<MP, NP>)
        return codebooks_per_tile(p, NP * 16) == 1 && p.entries <= F::template Copies<MP, NP>::kCopyEntries && (F::CSZ == 1 || MP > 1 || p.K <= 8192);
    return false;
}

template <class F>
bool fits(const ProblemB &p, int tile)
{
    bool ok = false;
    with_tile(tile, [&](auto mp, auto np) {
        typedef WaveKCfg<typename F::template Wave<mp(), np()>, mp(), np()> C;
        if constexpr (C::kExists) ok = C::lds_bytes((size_t)codebooks_per_tile(p, C::TN) * p.entries * p.vec * 2) <= 160 * 1024;
    });
    return ok;
}

// Costs of the tiles, by code size and vector length, fitted to 3200 launches, K 512 to 12288, 24 to 700 tiles: 1 to 6 % off; the tiles
// whose units are one step, 64 x 128, 80 x 64 and 96 x 64 - with 16-bit codes 64 x 64 too - 7 to 12 %, and 80 and 96 x 64, of which one
// launch in ten took half as long again, are set a tenth above their fit.
constexpr WaveKTile kTileCosts[2][2][15] = {
    {{{11, 1.5, 31, 10, 0.00}, {12, 2.2, 36, 12, 0.00}, {13, 1.8, 48, 11, 0.00}, {14, 2.4, 58, 17, 0.00}, {18, 3.3, 112, 19, 0.00}, {21, 1.6, 37, 11, 0.00}, {22, 2.4, 42, 16, 0.00},
      {23, 2.2, 49, 24, 0.00}, {24, 3.0, 62, 24, 0.00}, {28, 4.6, 107, 43, 0.02}, {34, 3.3, 75, 31, 0.05}, {44, 3.8, 90, 44, 0.06}, {48, 6.0, 132, 127, 0.27}, {54, 5.1, 108, 54, 0.06},
      {64, 4.8, 122, 67, 0.35}},
     {{11, 1.5, 29, 10, 0.00}, {12, 2.1, 40, 9, 0.00}, {13, 1.8, 51, 13, 0.04}, {14, 2.3, 62, 26, 0.00}, {18, 3.0, 120, 30, 0.00}, {21, 1.5, 37, 13, 0.01}, {22, 2.4, 41, 17, 0.24},
      {23, 2.2, 49, 27, 0.01}, {24, 2.9, 67, 32, 0.02}, {28, 4.3, 121, 60, 0.08}, {34, 3.3, 76, 33, 0.01}, {44, 3.6, 98, 42, 0.13}, {48, 6.8, 140, 102, 0.50}, {54, 5.4, 113, 47, 0.50},
      {64, 6.1, 117, 51, 0.50}}},
    {{{11, 1.5, 25, 9, 0.00}, {12, 2.1, 32, 13, 0.00}, {13, 1.8, 45, 12, 0.00}, {14, 2.4, 59, 17, 0.00}, {18, 3.2, 102, 41, 0.00}, {21, 1.6, 36, 11, 0.03}, {22, 2.4, 40, 16, 0.00},
      {23, 2.2, 48, 25, 0.08}, {24, 3.0, 60, 28, 0.01}, {28, 4.2, 110, 47, 0.08}, {34, 3.3, 72, 36, 0.07}, {44, 3.6, 80, 72, 0.11}, {48, 5.6, 149, 120, 0.26}, {54, 4.6, 110, 81, 0.50},
      {64, 4.8, 135, 64, 0.50}},
     // (no 32 x 128 and 48 x 64 here)
     {{11, 1.8, 29, 11, 0.00}, {12, 2.4, 42, 13, 0.00}, {13, 2.2, 50, 26, 0.00}, {14, 2.7, 69, 33, 0.18}, {18, 3.5, 136, 60, 0.00}, {21, 1.8, 41, 15, 0.03}, {22, 2.6, 51, 17, 0.19},
      {23, 2.2, 59, 39, 0.12}, {24, 3.0, 85, 38, 0.32}, {44, 3.4, 114, 51, 0.50}, {48, 5.6, 160, 178, 0.46}, {54, 5.1, 121, 52, 0.50}, {64, 5.8, 127, 90, 0.50}}}};
// with a table of copies
constexpr WaveKTile kCopiesCosts[2][9] = {
    {{11, 1.9, 25, 7, 0.00}, {12, 2.1, 33, 10, 0.00}, {13, 1.8, 36, 13, 0.00}, {14, 2.4, 42, 17, 0.00}, {18, 2.9, 65, 38, 0.03}, {22, 2.4, 42, 16, 0.00}, {23, 2.1, 43, 23, 0.00},
     {24, 2.8, 55, 22, 0.23}, {28, 3.8, 86, 60, 0.05}},
    {{11, 1.9, 24, 9, 0.01}, {12, 2.2, 30, 13, 0.00}, {13, 1.9, 38, 14, 0.00}, {14, 2.4, 48, 20, 0.00}, {18, 3.0, 78, 39, 0.00}, {22, 2.4, 38, 18, 0.00}, {23, 2.2, 45, 25, 0.02},
     {24, 2.9, 56, 30, 0.12}, {28, 3.8, 101, 47, 0.00}}};

template <class F>
WaveKPlan plan_b(const ProblemB &p)
{
    const int forced = (int)tuning().wave_k_force_tile;
    // An X that does not fit the 4 MB of an XCD's L2 beside the rest keeps the units waiting, the longer the larger it is, and most where
    // a unit of one step takes half a 128-byte line at a time.
    const double octaves = std::fmin(3.0, std::fmax(0.0, std::log2(2.0 * p.M * p.K / 2e6)));
    // Tiles of 64 x 64 in several rounds take another 30 % from 1500 rows on: M = 2168, K = 7808, N = 1024 takes 95 us, M = 3028, K = 11264,
    // N = 640 98 us, expected 64 without the two.
    const double wait_rows = 1.0 + 0.3 * (p.M < 1000 ? 0.0 : p.M > 1500 ? 1.0 : (p.M - 1000) / 500.0);
    const bool rounds = (int64_t)((p.M + 63) / 64) * ((p.N + 63) / 64) > device_cu_count();
    const double bytes = (double)p.K * p.N * F::CSZ / F::VEC + 2.0 * (double)p.M * (p.K + p.N);
    WaveKPlan best = {0, 0, 1e30};
    for (WaveKTile t : kTileCosts[F::CSZ - 1][F::VEC == 8 ? 0 : 1]) {
        if (forced > 0 && forced != t.tile) continue;
        if (!fits<F>(p, t.tile) || (p.gated && t.tile % 2 == 1)) continue;
        with_tile(t.tile, [&](auto mp, auto np) {
            if (F::CSZ == 2 || !takes_copies<F, mp(), np()>(p)) return;   // (16-bit codes: the tile as without copies, a little above its time)
            for (const WaveKTile &c : kCopiesCosts[F::VEC == 8 ? 0 : 1])
                if (c.tile == t.tile) t = c;
        });
        const double us = wave_k_tile_cost_us(t, p.M, p.K, p.N, bytes, (1.0 + t.wait * octaves) * (t.tile == 44 && rounds ? wait_rows : 1.0));
        if (us < best.cost_us) best = {t.tile / 10, t.tile % 10, us};
    }
    return best;
}

template <class F>
hipError_t launch_b(const ProblemB &p, hipStream_t s, int tile)
{
    if (tile == 0) {
        const WaveKPlan plan = plan_b<F>(p);
        tile = plan.mp * 10 + plan.np;
    }
    if (tile == 0) return hipErrorInvalidValue;   // (the one tile asked for does not fit)
    const WaveKArgs a = {p.x, p.codes, p.cb, p.y, p.bias, p.M, p.K, p.N, p.k_x, 0, 0, p.entries, p.rows_per_cb, codebooks_per_tile(p, tile % 10 * 16), p.gated ? 1 : 0};
    hipError_t e = hipErrorInvalidValue;
    with_tile(tile, [&](auto mp, auto np) {
        if constexpr (F::template kHasCopies<mp(), np()>)
            if (takes_copies<F, mp(), np()>(p)) {
                e = launch_tile<typename F::template Copies<mp(), np()>, mp(), np()>(a, s);
                return;
            }
        typedef typename F::template Wave<mp(), np()> P;
        if constexpr (WaveKCfg<P, mp(), np()>::kExists) e = launch_tile<P, mp(), np()>(a, s);
    });
    return e;
}

// calls f with the format's type; false where there is none
template <class F>
bool with_format(const ProblemB &p, F f)
{
    const bool u8 = p.code_bits == 8;
    if (p.vec == 8) {
        if (u8) f(Format<8, uint8_t>{});
        else f(Format<8, uint16_t>{});
    } else if (p.vec == 4) {
        if (u8) f(Format<4, uint8_t>{});
        else f(Format<4, uint16_t>{});
    } else {
        return false;
    }
    return true;
}

}  // namespace

bool wave_k_b_supports(const ProblemB &p)
{
    if (!wave_k_shape(p.x, p.M, p.K, p.N) || p.K % 64 != 0 || p.K < 128 || p.packed || p.k_x % 64 != 0) return false;
    if (((size_t)p.entries * p.vec * 2) % 16 != 0) return false;
    if ((int64_t)128 * (p.K / p.vec) * (p.code_bits / 8) >= (int64_t)1 << 31) return false;
    bool ok = false;
    with_format(p, [&](auto format) { ok = fits<decltype(format)>(p, 22); });
    return ok;
}

double wave_k_b_cost_us(const ProblemB &p)
{
    double t = 1e30;
    if (wave_k_b_supports(p)) with_format(p, [&](auto format) { t = plan_b<decltype(format)>(p).cost_us; });
    return t;
}

int wave_k_b_tile(const ProblemB &p)
{
    int tile = 0;
    with_format(p, [&](auto format) {
        const WaveKPlan plan = plan_b<decltype(format)>(p);
        tile = plan.mp * 10 + plan.np;
    });
    return tile;
}

// What the codes take to come out of HBM, at most 64 rows of X: the more of a row a unit of K brings (8, 16 or 32 bytes), the more are on
// their way - 2.0, 3.3 or 3.8 TB/s when every compute unit works, its share of that when some have no tile -, where the decode
// kernel, whose workgroups go on from tile to tile, draws up to 3.5 on any width.  (Without this 5 x 11648 x 27328, 159 MB of codes, 213
// units of 256 at work, was taken at 60.5 us where the decode kernel takes 45.8, 4 x 8448 x 26048 at 45.0, 35.1, and a gated
// 15 x 10112 x 20992 at 59.0, 43.1.  Over 236 shapes with 20 MB and more of codes the choice is 1.9 % from the better kernel, without 3.6;
// with the codes in the last-level cache, where the wave-K kernel stands better, 1.3 and 1.2.  There it would lose by more if this had to
// beat the decode kernel by the margin below too: 1.7 and 1.6.)
static double stream_us(const ProblemB &p, int tile)
{
    const int cus = device_cu_count(), tm = tile / 10 * 16, tn = tile % 10 * 16;
    const int64_t tiles = (int64_t)((p.M + tm - 1) / tm) * ((p.N + tn - 1) / tn), rounds = (tiles + cus - 1) / cus;
    const double bytes = (double)p.K * p.N / p.vec * (p.code_bits / 8) + 2.0 * (double)p.M * (p.K + p.N);
    const int brings = 64 / p.vec * (p.code_bits / 8);
    return 2.0 + bytes / (brings <= 8 ? 2.0e6 : brings <= 16 ? 3.3e6 : 3.8e6) * (double)(rounds * cus) / (double)tiles;
}

// The rule: whichever is expected to be faster.  Up to 64 rows of X the other is the decode path, whose model is as close as this
// one's (with these margins the choice is 1 to 3 % from the better one over 540 measured shapes); where that
// path would take its streaming or its general kernel it keeps up to 16 rows.  Above, the tiled kernels, by more than the models' error.
// (us, before -> now: M = 8, K = 640, N = 22912 23.8 -> 6.1; M = 44, K = 704, N = 21888, 4-vectors 32.3 -> 11.0; M = 100,
// K = 1408, N = 3500 11.9 -> 6.5; M = 256, K = N = 4096, 16-bit codes 26.5 -> 17.6; M = 451, K = 1152, N = 1376 18.2 -> 8.0.)
bool wave_k_b_preferred(const ProblemB &p, double t_other, double margin)
{
    const int force = (int)tuning().wave_k_force;
    if (force == 2 || !wave_k_b_supports(p)) return false;
    if (force == 1) return true;
    if (p.M <= 64) {
        const double t_decode = decode_slab_cost_us(p);
        // (the streaming kernel, up to 16 rows: over 34 of its shapes on codes out of HBM the tile expected to be fastest takes 0.85 of
        // its time up to K = 24576 - 16 x 11008 x 4096 11.9 us -> 8.9 - and over 7 from there on 1.03, 13 x 27520 x 2944 17.5 -> 20.2)
        if (t_decode > 1e29) return p.M > 16 || (p.K <= 24576 && decode_stream_preferred(p));
        // The gated decode kernels deal tiles in pairs, which their model does not see.  3 to 16 rows: over 425 shapes this line is 1.2 %
        // from the better kernel on codes out of HBM and 1.0 % on codes in the caches (0.92: 1.0 and 1.4, 0.97: 1.5 and 1.0); one and two rows of X, which the models know least (2 x 1024 x 576 3.0 us and 3.4), by more.
        return wave_k_b_cost_us(p) < (p.gated ? 1.15 : p.M <= 2 ? 0.85 : p.M <= 16 ? 0.94 : 0.97) * t_decode &&
               stream_us(p, wave_k_b_tile(p)) < (p.gated ? 1.15 : 1.0) * t_decode;
    }
    return wave_k_b_cost_us(p) < margin * t_other;
}

hipError_t launch_wave_k_b(const ProblemB &p, hipStream_t s, int tile)
{
    if (!wave_k_b_supports(p)) return hipErrorInvalidValue;
    hipError_t e = hipErrorInvalidValue;
    with_format(p, [&](auto format) { e = launch_b<decltype(format)>(p, s, tile); });
    return e;
}

}  // namespace vq
