// Grid autotuner: columns per side, slabs per side, slabs per shape block and
// position columns per column.
//
// The time of the planner and the pair kernel on a grid, for uniform densities:
//   tests : every shape against the positions of the position columns within
//           reach of its block, in batches of 64 lanes (half a batch of every
//           item is idle);
//   runs  : once per block and position, the lane's pending histogram run ends;
//   bodies: the pairs whose column touches the domain of their shape (bins,
//           e+ and ex, the histogram);
//   wraps : tests whose separation takes the minimum image pair by pair, where a
//           block and a slab or column straddle half the box;
//   items : the column lookup and the planner's work per item;
//   blocks: the planner's and the scalar loads' work per shape block.
// Thin position columns cut tests and bodies near the edge of the domain and
// add items (at most 64 columns each); small blocks cut tests and add runs and
// items.  The areas that columns of width f cover around a block or a shape are
// those of the Minkowski sums (for a convex outline of area A and perimeter p
// on a square grid, on average A + (2/pi) p f + f^2).  The constants are a fit
// to eight grids of a million clustered positions (200,000 shapes, reach 20 by
// 60), 8.7 to 9.8 ms: within 3 %, the best grid 2 % from the one it picks.  Wraps
// and blocks are from 590 grids of sixteen counts in boxes of 75 to 500: without
// wraps, blocks as tall as the box won wherever pi_max is half of it (300,001
// positions, 100,003 weighted shapes in a box of 75 16.8 ms, now 14.7; 208,875
// and 59,553 6.9, now 6.0), without blocks, three shapes per block in thin samples
// (562,663 positions, 40,378 shapes in a box of 300 1.86 ms, now 1.61).  Against
// the best of the grids tried for each count the pick is 1 % behind in the median.
#include "mia_common.hpp"

#include <algorithm>
#include <cmath>
#include <mutex>
#include <tuple>

namespace mia {

namespace {

constexpr double kTestCost = 1.15e-12;   // s per tested (shape, position) pair
constexpr double kRunCost = 1.1e-12;     // s per tested (block, position) pair
constexpr double kBodyCost = 1.0e-12;    // s per pair of the columns that touch a shape's domain
constexpr double kWrapCost = 0.5e-12;    // s per tested pair with a wrap
constexpr double kItemCost = 1.5e-9;     // s per work item
constexpr double kBlockCost = 4.0e-9;    // s per shape block
constexpr int kBlockShapes = 64;
constexpr int kItemPositions = 8192;
constexpr int kMaxPosColumns = 4096;     // position columns per side (12-bit indices)

constexpr int kSearchSteps = 40;         // column and slab counts tried per axis, about

struct Choice {
    int ncj, nzj, G, m;
};

// Expected cost and work items of one grid.
double grid_cost(double L, int jk, const Choice &c, double R, double Z, bool rmu, double Ns, double Np,
                 double *items_out = nullptr) {
    const double pi = 3.14159265358979;
    const int nc = c.ncj * jk, nz = c.nzj * jk;
    const double cw = L / nc, h = L / nz * c.G, f = cw / c.m;
    const double rho = Np / (L * L * L);
    const double groups = (double)nc * nc * (nz / c.G);
    const double lam = Ns / groups;
    const double nblocks = groups * (1.0 - std::exp(-lam)) * std::max(1.0, lam / kBlockShapes);
    const double per_block = Ns / std::max(nblocks, 1e-300);
    // a block of few shapes is smaller than its cells
    const double shrink = per_block > 1.0 ? (per_block - 1.0) / (per_block + 1.0) : 0.0;
    const double bw = cw * shrink, bh = h * shrink;
    // position columns of width g around a square block of side w
    auto area = [&](double w, double g) {
        const double a = w * w + 4.0 * w * R + pi * R * R, p = 4.0 * w + 2.0 * pi * R;
        return std::min(L * L, a + 2.0 / pi * p * g + g * g);
    };
    // mean line-of-sight window over those columns
    const double win = std::min(L, (rmu ? 4.0 / 3.0 * R : 2.0 * Z) + bh);
    const double per_col = rho * f * f * win;
    const double tests = Ns * rho * area(bw, f) * win;
    const double columns = area(bw, f) / (f * f);
    const double cpi = std::max(1.0, std::min((double)kWave, kItemPositions / std::max(per_col, 1e-9)));
    // rectangles of one sub-box and shift class the reach falls into
    const double side = bw + 2.0 * R + f;
    const double sx = 1.0 + std::min(side, L) / (L / jk), sz = 1.0 + win / (L / jk) + win / L;
    const double rects = sx * sx * sz;
    const double items = nblocks * std::max(rects, 1.27 * columns * sz / cpi + 0.5 * rects);
    if (items_out) *items_out = items;
    const double idle = items * 32.0 * per_block;
    // the part of an axis's windows that straddles half the box: the block's and a
    // cell's extent (w) on either side, where the reach comes as far
    auto mixed = [&](double reach, double w) { return reach + w > L / 2.0 ? std::min(1.0, 2.0 * w / L) : 0.0; };
    const double straight = 1.0 - mixed(R, bw + f), wraps = 1.0 - (1.0 - mixed(rmu ? R : Z, bh + L / nz)) * straight * straight;
    return (kTestCost + kWrapCost * wraps) * (tests + idle) + kRunCost * (tests + idle) / std::max(per_block, 1.0) +
           kBodyCost * Ns * rho * area(0.0, f) * win + kItemCost * items + kBlockCost * nblocks;
}

std::mutex g_mu;
std::map<std::tuple<double, int, double, double, int, int64_t, int64_t>, Choice> g_cache;

// Position columns per column: the cheapest of 1 .. 8.
int best_m(double L, int jk, Choice c, double R, double Z, bool rmu, double Ns, double Np, double *cost) {
    int best = 1;
    double best_t = -1.0;
    for (c.m = 1; c.m <= 8; ++c.m) {
        const double n = (double)c.ncj * jk * c.m;
        if (c.m > 1 && (n > kMaxPosColumns || n * n * (c.nzj * jk + 1.0) > 8.0 * Np + 262144.0)) break;
        const double t = grid_cost(L, jk, c, R, Z, rmu, Ns, Np);
        if (best_t < 0 || t < best_t) {
            best_t = t;
            best = c.m;
        }
    }
    *cost = best_t;
    return best;
}

Choice search(double L, int jk, double R, double Z, bool rmu, int64_t ns, int64_t np) {
    auto key = std::make_tuple(L, jk, R, Z, (int)rmu, ns, np);
    {
        std::lock_guard<std::mutex> lk(g_mu);
        auto it = g_cache.find(key);
        if (it != g_cache.end()) return it->second;
    }
    const double Ns = (double)std::max<int64_t>(ns, 1), Np = (double)std::max<int64_t>(np, 1);
    const double span = L / jk;
    const double zr = rmu ? R : Z;
    // column widths in [R/12, R/2], slab heights in [zr/12, max(zr, R)/2], at most 512 per side
    int c0 = std::max(1, (int)std::floor(span / (R / 2.0)));
    int c1 = std::max(c0, std::min(512 / jk, (int)std::ceil(span / (R / 12.0))));
    int z0 = std::max(1, (int)std::floor(span / (std::max(zr, R) / 2.0)));
    int z1 = std::max(z0, std::min(512 / jk, (int)std::ceil(span / (zr / 12.0))));
    Choice best{c0, z0, 1, 1};
    double best_t = -1.0;
    // at most kSearchSteps counts per axis, evenly spaced in the logarithm (a
    // search over all of them took 0.1 s for a large box without jackknife)
    auto counts = [](int lo, int hi) {
        std::vector<int> v;
        for (int k = 0; k <= kSearchSteps; ++k) {
            const int x = hi - lo < kSearchSteps ? lo + k
                                                 : (int)std::lround(lo * std::pow((double)hi / lo, k / (double)kSearchSteps));
            if (x <= hi && (v.empty() || x > v.back())) v.push_back(x);
        }
        return v;
    };
    const std::vector<int> cs = counts(c0, c1), zs = counts(z0, z1);
    for (int ncj : cs)
        for (int nzj : zs)
            for (int G = 1; G <= 4 && G <= nzj; ++G) {
                if (nzj % G) continue;
                Choice c{ncj, nzj, G, 1};
                double t;
                c.m = best_m(L, jk, c, R, Z, rmu, Ns, Np, &t);
                if (best_t < 0 || t < best_t) {
                    best_t = t;
                    best = c;
                }
            }
    std::lock_guard<std::mutex> lk(g_mu);
    g_cache[key] = best;
    return best;
}

}  // namespace

// Expected work items (at most what the block capacity allows).
double estimate_items(const Grid &g, int G, int cpi, double reach_r, double reach_z, bool rmu, int64_t ns, int64_t np,
                      int64_t blk_cap) {
    if (ns <= 0 || np <= 0) return 0.0;
    const int jk = g.jk > 0 ? g.jk : 1;
    const double fw = g.cw / g.m;
    const double groups = (double)g.nc * g.nc * (g.nz / std::max(1, G));
    const double lam = (double)ns / groups;
    const double nblocks =
        std::min((double)blk_cap, groups * (1.0 - std::exp(-lam)) * std::max(1.0, lam / kBlockShapes) + 1.0);
    const double side = std::min(g.L, g.cw + 2.0 * reach_r + fw), win = std::min(g.L, 2.0 * reach_z + G * g.hz);
    const double sx = 1.0 + side / (g.L / jk) + side / g.L, sz = 1.0 + win / (g.L / jk) + win / g.L;
    const double cols = (side / fw + 1.0) * (side / fw + 1.0);
    return nblocks * sz * (cols / cpi + sx * sx);
}

Grid make_grid(const mia_sample &s, const mia_bins &bins, const mia_tuning *t) {
    Grid g;
    g.L = s.boxsize;
    g.half = s.boxsize / 2.0;
    g.los = s.los;
    int k = 0;
    int na[2];
    for (int c = 0; c < 3; ++c)
        if (c != s.los) na[k++] = c;
    g.ax_a = na[0];
    g.ax_b = na[1];
    g.jk = s.jk_per_side > 0 ? s.jk_per_side : 0;
    g.jk_sub = g.jk > 0 ? s.jk_sub : s.boxsize;
    const bool rmu = bins.mode == MIA_RMU;
    double reach_r = std::sqrt(bins.r2_edges[bins.n_r]);
    double reach_z = rmu ? reach_r
                         : std::fmax(std::fabs(bins.x2_edges[0]), std::fabs(bins.x2_edges[bins.n_2]));
    int jk_eff = g.jk > 0 ? g.jk : 1;
    double span = g.L / jk_eff;
    int ncj, nzj, G = 0;
    if (t && t->cell_shapes > 0) {
        // density rule: cubes holding ~cell_shapes shapes, within [reach/10, reach/2]
        double nobj = (double)(s.n_shape > 0 ? s.n_shape : std::max<int64_t>(s.n_pos, 1));
        double a = std::cbrt((double)t->cell_shapes * g.L * g.L * g.L / nobj);
        double cw_t = std::min(std::max(a, reach_r / 10.0), reach_r / 2.0);
        double hz_t = std::min(std::max(a, reach_z / 10.0), std::max(reach_z / 2.0, reach_r / 2.0));
        ncj = std::max(1, (int)std::lround(span / cw_t));
        nzj = std::max(1, (int)std::lround(span / hz_t));
    } else {
        Choice c = search(g.L, jk_eff, reach_r, reach_z, rmu, s.n_shape, s.n_pos);
        ncj = c.ncj;
        nzj = c.nzj;
        G = c.G;
    }
    if (t && t->columns_per_side > 0) ncj = std::max(1, t->columns_per_side / jk_eff);
    if (t && t->slabs_per_side > 0) nzj = std::max(1, t->slabs_per_side / jk_eff);
    while (ncj * jk_eff > 512 && ncj > 1) --ncj;
    while (nzj * jk_eff > 512 && nzj > 1) --nzj;
    g.ncj = ncj;
    g.nzj = nzj;
    g.nc = ncj * jk_eff;
    g.nz = nzj * jk_eff;
    g.cw = g.L / g.nc;
    g.hz = g.L / g.nz;
    g.margin = 1e-9 * g.L + 1e-12;
    {
        Choice c{ncj, nzj, G > 0 && nzj % G == 0 ? G : 1, 1};
        double t;
        g.m = best_m(g.L, jk_eff, c, reach_r, reach_z, rmu, (double)std::max<int64_t>(s.n_shape, 1),
                     (double)std::max<int64_t>(s.n_pos, 1), &t);
    }
    g.G = (G > 0 && nzj % G == 0) ? G : 0;
    return g;
}

}  // namespace mia
