// gauss_rules.hpp -- which kernel the Gauss law and its projection take: plain
// C++, checked without a device.
#pragma once
#include <stdlib.h>
#include <string.h>

#include <initializer_list>

#include "limits.hpp"

namespace lqcd {

inline bool env_is(const char* name, const char* value)
{
    const char* env = getenv(name);
    return env && strcmp(env, value) == 0;
}

// workgroup tiles of the streamed kernels (k_gauss.hip)
struct GaussTiles {
    int a = 0, b = 0, C = 0;   // 0: no streamed tiling for this lattice
    int n1 = 0, n2 = 0;        // tiles along x_1, x_2
    int nblocks = 0;           // n1 n2 (L3 / C)
};

constexpr int kGaussHaloMax = kBlock;

// The streamed tiling of a D = 4 lattice, or a = 0 when it does not apply
// (or LQCD_GAUSS_TILES=0 pins the site walk): L0 divides 64 (whole x_0 rows
// per wavefront), a tile L0 x a x b of kBlock sites with the rows of a
// wavefront in one x_2 layer, a | L1, b | L2 and the smallest halo L0 (a + b);
// C | L3 the largest of 32, 16, .., 1 that leaves `target` workgroups or more and
// at most kMaxReduceBlocks: 512 (one round of two per CU), or half of the tiles
// where those are fewer than 1024, as C = 2 saves a quarter of the G evaluations
// (the 512 tiles of 16^3 x 32, us per step of C = 1 -> 2: f64 60.5 -> 50.2, f32 42.0 -> 38.4), but not
// below one workgroup per CU (the 256 tiles of 16^4, C = 1 -> 2: f64 29.3 -> 34.4).
inline GaussTiles gauss_tiles(const Geom& g)
{
    GaussTiles gt;
    if (g.dim != 4 || env_is("LQCD_GAUSS_TILES", "0")) return gt;
    const int L0 = g.extent[0], L1 = g.extent[1], L2 = g.extent[2], L3 = g.extent[3];
    if (L0 > 64 || 64 % L0 != 0) return gt;
    const int m = kBlock / L0, rpw = 64 / L0;
    int best_a = 0, best_b = 0;
    for (int a = rpw; a <= m; a += rpw) {
        if (m % a != 0) continue;
        const int b = m / a;
        if (L1 % a != 0 || L2 % b != 0) continue;
        if (L0 * (a + b) > kGaussHaloMax) continue;
        if (best_a == 0 || a + b < best_a + best_b) {
            best_a = a;
            best_b = b;
        }
    }
    if (best_a == 0) return gt;
    const int64_t tiles = (int64_t)(L1 / best_a) * (L2 / best_b);
    const int64_t all = tiles * L3;
    const int64_t half = all / 2 < 512 ? all / 2 : 512;
    const int64_t target = half > 256 ? half : all < 256 ? all : 256;
    int C = 0;
    for (int c : {32, 16, 8, 4, 2, 1})
        if (L3 % c == 0 && all / c >= target && all / c <= kMaxReduceBlocks) {
            C = c;
            break;
        }
    if (C == 0) return gt;
    gt.a = best_a;
    gt.b = best_b;
    gt.C = C;
    gt.n1 = L1 / best_a;
    gt.n2 = L2 / best_b;
    gt.nblocks = (int)(all / C);
    return gt;
}

// Whether the steps of the projection carry the transports U^+ E U of E along:
// small lattices, where the step is one round of memory latency and not the
// 1.1 - 1.7 KB per site that it moves: below 2^15 sites against the streamed
// tiles (f64, us per step: 16^2 x 8^2 19.0 -> 10.0, 8^4 16.4 -> 8.5;
// 16^3 x 8 f64 23.4 -> 16.3, but 16^4 f32 23.2 -> 25.4, 32^4 362 -> 502), and
// below 2^20 against the site walk, which evaluates up to D + 1 Gs per site
// one after the other (13x11x17x9 25.6 -> 13.5, 20x18x16x14 54.6 -> 33.2,
// 24^4 200 -> 167, 500^2 52.1 -> 36.3; 48^4 f32 2210 -> 2770).  Not in D = 3,
// where the site walk is level or ahead (8^3 7.9 / 7.9, 32^3 16.5 / 23.8, 48^3
// 35.5 / 38.5).  LQCD_GAUSS_TRANSPORTS=0 pins the steps without them (the
// streamed tiles, or the site walk that LQCD_GAUSS_TILES=0 pins), 1 those
// with them (not D = 3).
inline bool gauss_uses_transports(const Geom& g)
{
    if (g.dim == 3 || env_is("LQCD_GAUSS_TILES", "0") || env_is("LQCD_GAUSS_TRANSPORTS", "0")) return false;
    if (env_is("LQCD_GAUSS_TRANSPORTS", "1")) return true;
    return g.nsite < (gauss_tiles(g).a > 0 ? 1 << 15 : 1 << 20);
}

} // namespace lqcd
