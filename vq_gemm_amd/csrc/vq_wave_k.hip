// The kernels of vq_wave_k.h for the plain [K,N] GEMM and for geometry A.
#include "vq_wave_k.h"

namespace vq {

namespace {

enum WaveKind { kDense, kDenseAnyN, kGeometryA };

WaveKPlan wave_k_plan(int kind, int M, int K, int N)
{
    const int forced = (int)tuning().wave_k_force_tile;
    // Geometry A: over 450 shapes, M 20 to 4096, K 512 to 8192, N 512 to 8192, the tile chosen is 0.7 % from the fastest.  Numbered from
    // 100 on: the kernel of vq_wave_k_a.hip (3 to 6 % off; the others, which wait for memory more, 8 to 15 %).
    constexpr WaveKTile kTilesA[] = {{12, 1.6, 86, 27}, {22, 1.5, 96, 59}, {24, 2.4, 132, 47}, {42, 1.7, 102, 93}, {44, 2.6, 139, 96},
                                     {144, 3.4, 159, 47}, {164, 3.8, 188, 88}, {166, 5.3, 254, 94}, {184, 4.1, 205, 165}, {186, 7.0, 275, 133}};
    // (fp16 rows that straddle the memory's 128-byte lines cost a third more)
    constexpr WaveKTile kTilesDense[] = {{12, 1.6, 106, 13}, {22, 1.5, 137, 17}, {24, 1.5, 175, 10}, {42, 1.2, 167, 63}, {44, 1.8, 214, 45}};
    WaveKPlan best = {0, 0, 1e30};
    auto consider = [&](WaveKTile t) {
        const bool wide = t.tile > 100;
        if (forced > 0 && forced != t.tile && forced != t.tile % 100) return;
        t.tile %= 100;
        if (kind != kGeometryA && N % 64 != 0) t.idle_clk *= 1.38;
        const double us = wave_k_tile_cost_us(t, M, K, N, (double)K * N * (kind == kGeometryA ? 0.5 : 2.0) + 2.0 * (double)M * (K + N));
        if (us < best.cost_us) best = {t.tile / 10, t.tile % 10, us, wide};
    };
    if (kind == kGeometryA)
        for (const WaveKTile &t : kTilesA) consider(t);
    else
        for (const WaveKTile &t : kTilesDense) consider(t);
    return best;
}

template <class P>
hipError_t launch_wave_k(const WaveKArgs &a, const WaveKPlan &plan, hipStream_t s)
{
    switch (plan.mp * 10 + plan.np) {
    case 12: return launch_tile<P, 1, 2>(a, s);
    case 22: return launch_tile<P, 2, 2>(a, s);
    case 24: return launch_tile<P, 2, 4>(a, s);
    case 42: return launch_tile<P, 4, 2>(a, s);
    case 44: return launch_tile<P, 4, 4>(a, s);
    default: return hipErrorInvalidValue;
    }
}

bool dense_any_n(const half_t *w, int N) { return N % 8 != 0 || (reinterpret_cast<uintptr_t>(w) & 15) != 0; }

}  // namespace

bool gemm_wave_k_supports(const half_t *x, const half_t *w, int M, int K, int N)
{
    return wave_k_shape(x, M, K, N) && (reinterpret_cast<uintptr_t>(w) & 1) == 0;
}

double gemm_wave_k_cost_us(const half_t *w, int M, int K, int N) { return wave_k_plan(dense_any_n(w, N) ? kDenseAnyN : kDense, M, K, N).cost_us; }

hipError_t launch_gemm_wave_k(const half_t *x, const half_t *w, half_t *y, int M, int K, int N, hipStream_t s)
{
    if (!gemm_wave_k_supports(x, w, M, K, N)) return hipErrorInvalidValue;
    const WaveKArgs a = {x, w, nullptr, y, nullptr, M, K, N, K, 0, 0, 0, 1, 0, 0};
    if (dense_any_n(w, N)) return launch_wave_k<WaveDenseAnyN>(a, wave_k_plan(kDenseAnyN, M, K, N), s);
    return launch_wave_k<WaveDense>(a, wave_k_plan(kDense, M, K, N), s);
}

bool wave_k_a_supports(const ProblemA &p)
{
    return p.Nc >= 16 && p.Nc % 16 == 0 && wave_k_shape(p.x, p.M, p.K, 2 * p.Nc) && (reinterpret_cast<uintptr_t>(p.w) & 15) == 0 &&
           (reinterpret_cast<uintptr_t>(p.cb) & 15) == 0;
}

double wave_k_a_cost_us(const ProblemA &p) { return wave_k_plan(kGeometryA, p.M, p.K, 2 * p.Nc).cost_us; }

hipError_t launch_wave_k_a(const ProblemA &p, hipStream_t s)
{
    if (!wave_k_a_supports(p)) return hipErrorInvalidValue;
    const WaveKPlan plan = wave_k_plan(kGeometryA, p.M, p.K, 2 * p.Nc);
    if (plan.wide) return launch_wave_k_a_wide(p, plan.mp * 10 + plan.np, s);
    const WaveKArgs a = {p.x, p.w, p.cb, p.y, nullptr, p.M, p.K, 2 * p.Nc, p.K, 0, 0, 0, 1, 0, 0};
    return launch_wave_k<WaveA>(a, plan, s);
}

}  // namespace vq
