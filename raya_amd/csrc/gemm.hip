// launch_gemm: the checks, the tile and the split of an NT GEMM (the kernel is in gemm_kernel.hpp).
#include <cmath>
#include <type_traits>

#include "gemm_kernel.hpp"

namespace raya {
namespace {

using namespace gemm;

constexpr int kUnits = 256;  // MI355X compute units

// What a tile's workgroups take, fitted to measured launches (K = 768 and 3072, 1 to 4,000
// workgroups, N(0, 1) operands): `fixed` us a launch, and per 768 of k `alone` us while each
// compute unit has at most one workgroup and `each` us per workgroup of a unit beyond that.
struct TileCost {
    int bm, bn, bk, threads;
    double fixed, alone, each;
};
template <class T>
constexpr TileCost tile_cost(double fixed, double alone, double each) {
    return {T::BM, T::BN, T::BK, T::THREADS, fixed, alone, each};
}
constexpr TileCost kTiles[] = {
    tile_cost<Tile256>(10.0, 95.0, 118.0),   tile_cost<Tile256x128>(8.0, 40.0, 63.0),
    tile_cost<Tile128>(9.0, 23.0, 37.0),     tile_cost<Tile64x128>(6.3, 16.0, 19.5),
    tile_cost<Tile64>(6.6, 9.2, 13.4),       tile_cost<Tile32>(7.5, 6.3, 10.0),
};
constexpr int kTileCount = sizeof kTiles / sizeof kTiles[0];

int64_t blocks_of(int64_t m, int64_t n, int bm, int bn, int act) {
    const int out_bn = act == RAYA_EPI_GEGLU ? bn / 2 : bn;
    return (m + bm - 1) / bm * ((n + out_bn - 1) / out_bn);
}
int64_t tiles_of(int tile, int m, int n, int act) { return blocks_of(m, n, kTiles[tile].bm, kTiles[tile].bn, act); }

// Outputs of more 128 x 128 blocks than this are refused (rows and columns then stay below 2^30, and
// the kernel's 32-bit row and column numbers cannot overflow); a launch has fewer than 2^32 threads.
constexpr int64_t kMaxBlocks = 0x7fffffff / 256, kMaxThreads = int64_t(1) << 32;
bool within_limits(int m, int n, int act) { return blocks_of(m, n, 128, 128, act) <= kMaxBlocks; }

struct GemmPlan {
    int tile, splits;
};

size_t partial_floats(const GemmPlan &p, int m, int n, int act) {
    return p.splits > 1 ? (size_t)tiles_of(p.tile, m, n, act) * p.splits * kTiles[p.tile].bm * kTiles[p.tile].bn : 0;
}

// The cheapest tile (and, within `room` floats of partials, split) by that measure, among those
// whose grid can be launched (within_limits: the 256 x 128 tile's can).  `whole`: only tiles whose
// slabs divide the depth (the row statistics' kernels do not pad).
GemmPlan plan_of(int m, int n, int k, int act, bool vec, bool whole, size_t room) {
    GemmPlan best{1, 1};
    double cost = 1e300;
    for (int t = 0; t < kTileCount; ++t) {
        const TileCost &c = kTiles[t];
        const bool pad = !vec || k % c.bk != 0;
        if (pad && (t == 0 || whole)) continue;
        const int64_t tiles = tiles_of(t, m, n, act);
        for (int s = 1; s <= 8; ++s) {
            if (tiles * s * c.threads >= kMaxThreads) break;
            if (s > 1 && (t == 0 || ((int64_t)k + c.bk - 1) / c.bk < 2 * s || partial_floats({t, s}, m, n, act) > room))
                break;
            const double r = (double)(tiles * s) / kUnits;
            // A last round that is not full runs faster than a full one, the less so the larger the tile.
            const double part = t == 0 ? 0.25 : 0.5;
            const double per = r <= 1.0 ? c.alone + 0.25 * r * (c.each - c.alone)
                                        : c.each * (part * r + (1.0 - part) * std::ceil(r));
            double us = c.fixed + per * k / (768.0 * s);
            // The summing launch: its own fixed cost and the partials written and read once each.
            if (s > 1) us += 5.0 + partial_floats({t, s}, m, n, act) * 8.0 / 3e6;
            if (us < cost) cost = us, best = {t, s};
        }
    }
    return best;
}

hipError_t launch(const GemmLaunch &g, hipStream_t stream) {
    constexpr int kNone = RAYA_EPI_NONE, kGeglu = RAYA_EPI_GEGLU;
    const int act = g.act;
    const bool norm = g.in_stats || g.in_chunks;
    if (norm || g.out_stats) {
        // Only the staged epilogue carries them (see GemmLaunch).
        const bool vec_out = (g.ldo & 3) == 0 && ((uintptr_t)g.out & 15) == 0 &&
                             (!g.residual || ((g.ldr & 3) == 0 && ((uintptr_t)g.residual & 15) == 0));
        if (!vec_out) return hipErrorInvalidValue;
        if (norm && (!g.colsum || (!g.in_stats && g.k % 64 != 0))) return hipErrorInvalidValue;
        if (g.out_stats && (act != kNone || g.n % 64 != 0)) return hipErrorInvalidValue;
    }
    if (g.rope_cos && (act != kNone || g.residual || g.rope_cols % kRopeHeadDim != 0 || g.rope_cols > g.n))
        return hipErrorInvalidValue;
    if (g.reduce || g.splits > 1) return hipErrorInvalidValue;  // launch_gemm's own fields
    if (!within_limits(g.m, g.n, act)) return hipErrorInvalidValue;
    const GemmPlan p = plan_of(g.m, g.n, g.k, act, aligned_rows(g), norm || g.out_stats,
                               g.partials ? g.partial_floats : 0);
    const int64_t tiles = tiles_of(p.tile, g.m, g.n, act);
    const auto with = [&](const GemmLaunch &l, int64_t grid, auto geglu) {
        constexpr bool G = decltype(geglu)::value;
        switch (p.tile) {
        case 0: return launch_tile<Tile256, G>(l, (unsigned)grid, stream);
        case 1: return launch_tile<Tile256x128, G>(l, (unsigned)grid, stream);
        case 2: return launch_tile<Tile128, G>(l, (unsigned)grid, stream);
        case 3: return launch_tile<Tile64x128, G>(l, (unsigned)grid, stream);
        case 4: return launch_tile<Tile64, G>(l, (unsigned)grid, stream);
        default: return launch_tile<Tile32, G>(l, (unsigned)grid, stream);
        }
    };
    const auto go = [&](const GemmLaunch &l, int64_t grid) {
        return act == kGeglu ? with(l, grid, std::true_type{}) : with(l, grid, std::false_type{});
    };
    GemmLaunch l = g;
    l.splits = p.splits;
    hipError_t e = go(l, tiles * p.splits);
    if (e != hipSuccess || p.splits == 1) return e;
    // Split-K: the partial tiles are complete when the first launch ends; one workgroup
    // per tile sums them and runs the epilogue.
    l.reduce = 1;
    return go(l, tiles);
}

}  // namespace

size_t gemm_partial_floats(int m, int n, int k, int act) {
    if (m <= 0 || n <= 0 || k <= 0 || !within_limits(m, n, act)) return 0;
    return partial_floats(plan_of(m, n, k, act, true, true, SIZE_MAX), m, n, act);
}

hipError_t launch_gemm(const GemmLaunch &g, hipStream_t stream) {
    if (g.m == 0 || g.n == 0) return hipSuccess;
    if (g.act < RAYA_EPI_NONE || g.act > RAYA_EPI_GEGLU) return hipErrorInvalidValue;
    return launch(g, stream);
}

}  // namespace raya

// The tile and split that launch_gemm takes, for the tests: {rows, weight rows, threads, splits, workgroups}
// of aligned (`vec`) or other operands, with `room` floats of partials.  0, or -1 where it refuses the size.
extern "C" int raya_gemm_plan(int m, int n, int k, int act, int vec, int whole, uint64_t room, int64_t *out) {
    using namespace raya;
    if (m <= 0 || n <= 0 || k < 0 || !within_limits(m, n, act)) return -1;
    const GemmPlan p = plan_of(m, n, k, act, vec != 0, whole != 0, room);
    const TileCost &t = kTiles[p.tile];
    const int64_t plan[5] = {t.bm, t.bn, t.threads, p.splits, tiles_of(p.tile, m, n, act) * p.splits};
    std::copy(plan, plan + 5, out);
    return 0;
}
