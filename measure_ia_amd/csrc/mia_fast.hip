// Fast pair counter: cell-pair work items, LDS histograms.
//
// Replaces the per-shape KDTree loop and np.add.at scatter of the reference
// (src/measureia/measure_w_box_jk.py:386-461, measure_m_box_jk.py:403-487)
// with three steps on the device:
//   1. plan   : shapes of one column and a few line-of-sight slabs form a
//               block (<= 64 shapes, one jackknife region R_s).  Positions are
//               sorted by thinner columns.  A block's reach along each axis
//               falls into segments of one jackknife sub-box and one periodic
//               shift; a rectangle of two such segments and a line-of-sight
//               run have one position region R_p, and up to 64 columns of it
//               make a work item.  Items are counting-sorted by
//               (sample, R_s, R_p).
//   2. pairs  : a persistent grid takes contiguous runs of the sorted list,
//               balanced by estimated cost to a batch of 64 positions, then
//               claims tail chunks from a counter.  Each lane looks up the
//               positions of one column of an item; the wave then reads its
//               shape block through the scalar cache (one 64-byte record per
//               shape, wave-uniform) and streams the positions through
//               registers, 64 at a time.  Separations are the reference's own
//               FP64 differences, so r_p^2 (or r^2) and pi are compared exactly
//               with the host-bisected thresholds (an FP32 log2 only guesses
//               the bin); e+ and ex are FP64 (CDNA4 runs FP64 FMA at the rate
//               of non-packed FP32) and go into an LDS histogram (a wave's own, or shared by a workgroup) with
//               LDS atomics.  mu = pi/r is screened in FP32 and recomputed in
//               FP64 when it lies within a guard band of a bin edge; the
//               arccos NaN rule is likewise checked in FP64 for nearly
//               parallel pairs.
//   3. flush  : a histogram is added to the workspace's FP64
//               accumulators of the total and of tally[R_s] / tally[R_p]
//               only when the (R_s, R_p) key changes, i.e. a handful of times
//               per wave; k_finalize then writes the caller's outputs.  In
//               the deterministic mode the flushes go to per-wave slots that
//               k_finalize_det sums in a fixed order instead.
// Pair counts are integers (exact, order independent); the e+ sums are FP64
// throughout, so every bin carries only the rounding of FP64 additions.
#include "mia_common.hpp"

#include <hipcub/hipcub.hpp>

#include <cmath>
#include <memory>
#include <mutex>

namespace mia {

namespace {

constexpr int kMaxWavesPerBlock = 4;
constexpr int kThreads = kWave * kMaxWavesPerBlock;
constexpr size_t kPairStaticLds = 64;            // the pair kernel's own LDS words, at most
constexpr int kStatCopies = 32, kStatStride = 16;  // copies of the pair kernel's statistics, words apart
constexpr int kSharedBelow = 16;                 // private waves per CU below which histograms are shared
// A wave spills the 32-bit counts every 2^kSpillBits wave-iterations of 64 pairs at
// most, and looks after kRunBatches batches against 64 shapes: the four waves of a
// group add at most 4 * 64 * (2^23 + 2^22) < 2^32 pairs to a count in between.
constexpr int kSpillBits = 23, kRunBatches = 1 << 16;
constexpr int kSplitItems = 32;                  // items per group of four waves below which a claim is a quarter of an item
constexpr int kPairWavesPerSimd = 6;             // waves per SIMD the pair kernel's registers allow
constexpr int64_t kMaxKeysPerSample = 1 << 24;   // K^2 planner keys per sample (K regions)
constexpr double kSinExact = 1e-5;  // FP64 arccos-domain check when |sin phi| < 1e-5 |cos phi|

#define MIA_CONST __attribute__((address_space(4)))

struct Block {
    int32_t s0, ns;
    int32_t sample, rs;
};

// A work item pairs one shape block with the positions of up to kItemColumns
// consecutive position columns of one rectangle (columns within reach of the
// block, of one jackknife sub-box and one periodic shift class per axis), over
// one line-of-sight run of slabs.  The pair kernel looks the columns' positions
// up itself, one column per lane, so the plan holds no per-column record.
struct Item {
    int32_t blk;
    int32_t w;          // R_p | shift byte << 16: 2 bits per axis (a, b, l): 0 -> 0, 1 -> +L, 2 -> -L ;
                        // bit 6: per-pair wrap | line-of-sight class (3: mixed) << 24
    uint16_t ja, jb;    // first column of the rectangle
    uint16_t wb, nc;    // columns of the rectangle along b; columns of the item
    int32_t c0;         // the item's first column, counted row by row in the rectangle
    uint16_t k0, k1;    // slabs [k0, k1); k0 == nz: the columns' tails
    int32_t np;         // positions (k_item_cost)
    int32_t key;        // planner key over all samples
};
static_assert(sizeof(Item) == 32, "Item layout");
static_assert(sizeof(Block) == 16, "Block layout");

struct SampleDev {
    // sorted sample
    const double *prec;          // 4 doubles per position {a, b, l, w}, sorted order
    const double *srec;          // 8 doubles per shape, sorted order
    double L, half;
    int los, K, nbins, pad;
    // accumulators (workspace)
    unsigned long long *npairs;   // (1+K)*B
    double *dd, *sp;              // (1+K)*B (dd: weighted samples only)
    double *sx, *var;             // B
};

// Planner view of one sample (per-call parameter block).  Its (column, slab
// group) cells occupy [cell0, cell0 + ncells) of the global cell arrays.
struct PlanSample {
    Grid g;
    int mode, periodic;
    int ng, G;           // slab groups per column, slabs per group
    int ncp, cpi;        // position columns per side (g.nc * g.m), columns per item
    int pbits, pad;      // positions' fine key = (cell << pbits) + line-of-sight part of the slab
    double fw, hq_inv;   // position column width, line-of-sight parts per length
    double reach_r, reach_z;
    double x_lo, x_hi;   // line-of-sight domain, for cutting slab runs to a block's window
    const int32_t *sstart;
    const int32_t *pfine;  // starts of the positions' fine keys
    const int32_t *flags;  // bit 1: some position lies in a column's tail
    const double *srec;  // shape records (block bounding boxes)
    int64_t cell0, ncells;
};

// Finalisation view of one sample: accumulators to caller outputs.
struct FinSample {
    const unsigned long long *np;
    const double *sp, *dd, *sx, *var;
    const unsigned long long *rcnt;   // [2K] objects per region (positions, shapes)
    const double *rsum;               // [2K] sum w_s, sum w_s (1 - e^2/2) per region
    mia_counts out;
    int K, B, weighted, var_on;
};

// Largest s in [0, n) with tab[s] <= v (tab ascending, tab[0] <= v).
__device__ __forceinline__ int find_sample(const int64_t *tab, int n, int64_t v) {
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (tab[mid] <= v)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

__device__ __forceinline__ int region_of(const Grid &g, int ia, int ib, int il) {
    if (g.jk <= 0) return 0;
    int j[3];
    j[g.ax_a] = ia / g.ncj;
    j[g.ax_b] = ib / g.ncj;
    j[g.los] = il / g.nzj;
    return j[0] * g.jk * g.jk + j[1] * g.jk + j[2];
}

// Separation range [lo, hi] (unwrapped) -> minimum |minimum-image value| and
// the shift class: 0 none, 1 +L for all, 2 -L for all, 3 mixed.
__device__ __forceinline__ void axis_class(double lo, double hi, double L, double half,
                                           bool periodic, double &dmin, int &cls) {
    if (!periodic) {
        dmin = lo > 0 ? lo : (hi < 0 ? -hi : 0.0);
        cls = 0;
        return;
    }
    dmin = 1e300;
    // piece below -half: value + L
    if (lo < -half) {
        double a = lo + L, b = (hi < -half ? hi : -half) + L;
        double d = a > 0 ? a : (b < 0 ? -b : 0.0);
        dmin = d < dmin ? d : dmin;
    }
    if (hi >= -half && lo <= half) {
        double a = lo > -half ? lo : -half, b = hi < half ? hi : half;
        double d = a > 0 ? a : (b < 0 ? -b : 0.0);
        dmin = d < dmin ? d : dmin;
    }
    if (hi > half) {
        double a = (lo > half ? lo : half) - L, b = hi - L;
        double d = a > 0 ? a : (b < 0 ? -b : 0.0);
        dmin = d < dmin ? d : dmin;
    }
    if (lo > half)
        cls = 2;
    else if (hi < -half)
        cls = 1;
    else if (lo >= -half && hi <= half)
        cls = 0;
    else
        cls = 3;
}

__device__ __forceinline__ double shift_val(int cls, double L) {
    return cls == 1 ? L : (cls == 2 ? -L : 0.0);
}

// Whether slab k is within line-of-sight reach of a block's shapes (extent
// [zlo, zhi]), and its shift class cz.
__device__ __forceinline__ bool slab_in(const PlanSample &P, double zlo, double zhi, int k, int &cz) {
    const Grid &g = P.g;
    const double m = g.margin;
    double dzmin;
    axis_class(zlo - (k + 1) * g.hz - 2 * m, zhi - k * g.hz + 2 * m, g.L, g.half, P.periodic, dzmin, cz);
    return dzmin < P.reach_z + 4 * m;
}

// The positions [pb, pb + n) of one position column (ja, jb) within reach of a
// block (bounding box of its shapes bb): slabs [k0, k1) of shift class cz, cut
// to the block's line-of-sight window, or (k0 == nz) the column's tail.
struct ColumnView {
    const int32_t *pfine;
    double L, half, margin, fw, hq_inv, reach_r, x_lo, x_hi;
    int ncp, nz, pbits, mode, periodic;
};

template <class PS>
__device__ __forceinline__ ColumnView column_view(const PS *p) {
    ColumnView v;
    v.pfine = p->pfine;
    v.L = p->g.L;
    v.half = p->g.half;
    v.margin = p->g.margin;
    v.fw = p->fw;
    v.hq_inv = p->hq_inv;
    v.reach_r = p->reach_r;
    v.x_lo = p->x_lo;
    v.x_hi = p->x_hi;
    v.ncp = p->ncp;
    v.nz = p->g.nz;
    v.pbits = p->pbits;
    v.mode = p->mode;
    v.periodic = p->periodic;
    return v;
}

__device__ __forceinline__ void column_positions(const ColumnView &v, double b0, double b1, double b2, double b3,
                                                 double zlo, double zhi, int ja, int jb, int k0, int k1, int shifts,
                                                 int cz, int &pb, int &n) {
    const double m = v.margin;
    double da, db;
    const double alo = b0 - (ja + 1) * v.fw - 2 * m, ahi = b1 - ja * v.fw + 2 * m;
    const double blo = b2 - (jb + 1) * v.fw - 2 * m, bhi = b3 - jb * v.fw + 2 * m;
    if (shifts & 64) {
        int ca, cb;
        axis_class(alo, ahi, v.L, v.half, v.periodic, da, ca);
        axis_class(blo, bhi, v.L, v.half, v.periodic, db, cb);
    } else {
        // one shift for the whole rectangle: the distance of the shifted ranges from zero
        const double sa = shift_val(shifts & 3, v.L), sb = shift_val((shifts >> 2) & 3, v.L);
        da = fmax(fmax(alo + sa, -(ahi + sa)), 0.0);
        db = fmax(fmax(blo + sb, -(bhi + sb)), 0.0);
    }
    const double rr = v.reach_r + 4 * m;
    const double dxy2 = da * da + db * db;
    pb = 0;
    n = 0;
    if (dxy2 >= rr * rr) return;
    const int64_t base = ((int64_t)ja * v.ncp + jb) * (v.nz + 1);
    int64_t f0 = (base + k0) << v.pbits, f1 = (base + k1) << v.pbits;
    if (cz != 3) {
        // a shape of the block pairs with l in (zlo + sh - x_hi, zhi + sh - x_lo]
        // for the run's shift sh ((r, mu): within the sphere over the column)
        const double sh = shift_val(cz, v.L);
        double wlo, whi;
        if (v.mode == MIA_RPPI) {
            wlo = zlo + sh - v.x_hi - 4 * m;
            whi = zhi + sh - v.x_lo + 4 * m;
        } else {
            const double rz = sqrt(rr * rr - dxy2);
            wlo = zlo + sh - rz - 4 * m;
            whi = zhi + sh + rz + 4 * m;
        }
        const double q0 = (double)(k0 << v.pbits), q1 = (double)(k1 << v.pbits);
        const double lo = fmin(fmax(floor(wlo * v.hq_inv), q0), q1), hi = fmin(fmax(floor(whi * v.hq_inv) + 1.0, q0), q1);
        f0 = (base << v.pbits) + (int64_t)lo;
        f1 = (base << v.pbits) + (int64_t)hi;
        if (f1 <= f0) return;
    }
    pb = v.pfine[f0];
    n = v.pfine[f1] - pb;
}

constexpr int kPlanThreads = 256;
constexpr int kPlanWaves = kPlanThreads / kWave;
constexpr int kPlanGridPerCu = 8;        // workgroups per CU of the planner's persistent grids
constexpr int kItemPositions = 8192;    // positions of an item, about
// Segments a block's reach falls into along one axis: the sub-boxes it meets
// (at most one of them twice, where the periodic image closes on itself) plus
// the changes of shift class (-L, mixed, none, mixed, +L).
constexpr int kSegExtra = 6;
constexpr int kMaxSegs = 16 + kSegExtra;  // fast_path_fits: at most 16 sub-boxes per side

struct PlanLaunch {
    const PlanSample *ps;
    int64_t ncells;           // cells of all samples
    int K1;                   // regions + 1 of the largest sample's key space (keys per sample K1^2)
    int kseg;                 // segments stored per axis
    int one_key;              // one sample, no regions: a single key, counted per workgroup
    const int32_t *boff;      // block offset of every cell (exclusive scan of the block counts)
    const Block *blocks;
    double *bbox;             // bounding box {a_lo, a_hi, b_lo, b_hi, l_lo, l_hi} of every block's shapes
    uint32_t *geo;            // per block: 3 counts, then kseg segments per axis (a, b, l)
    unsigned long long *key_count;   // k_block_geom
    unsigned long long *key_cursor;  // k_emit_items
    const int64_t *key_off;
    Item *items;
    int64_t cap;              // item capacity
    unsigned long long *overflow;  // set when the items exceed their capacity
    // deterministic order: with it, every item's (key, block, rectangle) word;
    // a stable sort by it fixes the order the cursor atomics gave the items of one key
    unsigned long long *sort_key;
    int sort_shift;
};

// A segment: indices [j0, j1] of one shift class, 12 bits each and 2 bits of class.
__device__ __forceinline__ int seg_j0(uint32_t s) { return s & 0xfff; }
__device__ __forceinline__ int seg_j1(uint32_t s) { return (s >> 16) & 0xfff; }
__device__ __forceinline__ int seg_cls(uint32_t s) { return (s >> 12) & 3; }

// The rectangles of one block: every combination of an a segment, a b segment
// and a line-of-sight run (plus, where the sample has tail positions, the
// tails).  Calls f(index, key, items, seg a, seg b, run, R_p), the run ~0 for
// the tail, for this lane's combinations.
template <class F>
__device__ __forceinline__ void for_rects(const PlanSample &P, int rs, int K1, int nA, int nB, int nR,
                                          const uint32_t *segA, const uint32_t *segB, const uint32_t *segR, int lane,
                                          F &&f) {
    const Grid &g = P.g;
    const int nL = nR + ((*P.flags & 2) ? 1 : 0);
    const int T = nA * nB * nL;
    const int pj = g.ncj * g.m;
    for (int t = lane; t < T; t += kWave) {
        const int ir = t % nL, ib = (t / nL) % nB, ia = t / (nL * nB);
        const uint32_t a = segA[ia], b = segB[ib], r = ir < nR ? segR[ir] : ~0u;
        const int cols = (seg_j1(a) - seg_j0(a) + 1) * (seg_j1(b) - seg_j0(b) + 1);
        int rp = 0;
        if (g.jk > 0 && ir < nR) {
            int j[3];
            j[g.ax_a] = seg_j0(a) / pj;
            j[g.ax_b] = seg_j0(b) / pj;
            j[g.los] = seg_j0(r) / g.nzj;
            rp = j[0] * g.jk * g.jk + j[1] * g.jk + j[2];
        }
        f(t, rs * K1 + rp, (cols + P.cpi - 1) / P.cpi, a, b, r, rp);
    }
}

// One wave per shape block: the bounding box of its shapes, its reach along
// each axis as segments of one sub-box and one shift class, and the items per
// key.  Reach is tested from the bounding box, not from the block's cells.
__global__ __launch_bounds__(kPlanThreads) void k_block_geom(PlanLaunch A) {
    __shared__ uint32_t seg[kPlanWaves][3][kMaxSegs + 2];
    const int lane = threadIdx.x & (kWave - 1);
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    __shared__ int s_same;
    if (threadIdx.x == 0) s_same = 0;
    __syncthreads();
    const int nblk = A.boff[A.ncells];
    const int gstride = 3 + 3 * A.kseg;
    int same = 0;
    for (int blk = blockIdx.x * kPlanWaves + wv; blk < nblk; blk += gridDim.x * kPlanWaves) {
        const Block B = A.blocks[blk];
        const PlanSample &P = A.ps[B.sample];
        const Grid &g = P.g;
        double lo[3], hi[3];
        {
            const double *r = P.srec + 8 * (int64_t)(B.s0 + (lane < B.ns ? lane : 0));
#pragma unroll
            for (int k = 0; k < 3; ++k) lo[k] = hi[k] = r[k];
        }
        for (int d = kWave / 2; d > 0; d >>= 1)
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                lo[k] = fmin(lo[k], __shfl_xor(lo[k], d));
                hi[k] = fmax(hi[k], __shfl_xor(hi[k], d));
            }
        if (lane < 3) {
            A.bbox[6 * (int64_t)blk + 2 * lane] = lane == 0 ? lo[0] : (lane == 1 ? lo[1] : lo[2]);
            A.bbox[6 * (int64_t)blk + 2 * lane + 1] = lane == 0 ? hi[0] : (lane == 1 ? hi[1] : hi[2]);
        }
        const double m = g.margin, rr = P.reach_r + 4 * m;
        int cnt[3];
        // lane i of a pass holds the i-th column (slab) of the axis with its
        // state (index | class << 12 | sub-box << 16, -1: out of reach); a
        // segment starts where the state does not continue the one before
#pragma unroll
        for (int ax = 0; ax < 3; ++ax) {
            uint16_t *half = (uint16_t *)seg[wv][ax];
            int u0 = 0, W = g.nz;
            const int n = ax < 2 ? P.ncp : g.nz;
            if (ax < 2) {
                const int a0 = (int)floor((lo[ax] - rr) / P.fw) - 1, a1 = (int)floor((hi[ax] + rr) / P.fw) + 1;
                u0 = a0;
                W = a1 - a0 + 1;
                if (W >= n || !P.periodic) {
                    u0 = 0;
                    W = n;
                }
            }
            auto state = [&](int i) {
                if (i < 0 || i >= W) return -1;
                int j = u0 + i;
                int cls;
                if (ax < 2) {
                    j = j < 0 ? j + n : (j >= n ? j - n : j);
                    double dmin;
                    axis_class(lo[ax] - (j + 1) * P.fw - 2 * m, hi[ax] - j * P.fw + 2 * m, g.L, g.half, P.periodic,
                               dmin, cls);
                    if (!(dmin < rr)) return -1;
                    return j | (cls << 12) | (j / (g.ncj * g.m) << 16);
                }
                if (!slab_in(P, lo[2], hi[2], j, cls)) return -1;
                return j | (cls << 12) | (j / g.nzj << 16);
            };
            // b continues a: the next index of the same class and sub-box
            auto cont = [](int a, int b) { return a >= 0 && b >= 0 && b == a + 1; };
            int c = 0;
            for (int i0 = 0; i0 < W; i0 += kWave) {
                const int i = i0 + lane;
                const int s = state(i);
                const bool st = s >= 0 && !cont(state(i - 1), s), en = s >= 0 && !cont(s, state(i + 1));
                const uint64_t ms = __ballot(st);
                const int at = c + __popcll(ms & ((2ull << lane) - 1)) - 1;
                if (st && at < A.kseg) half[2 * at] = (uint16_t)(s & 0x3fff);
                if (en && at < A.kseg) half[2 * at + 1] = (uint16_t)(s & 0xfff);
                c += __popcll(ms);
            }
            // (kseg bounds the segments of any reach; see kSegExtra)
            cnt[ax] = c < A.kseg ? c : A.kseg;
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        uint32_t *G = A.geo + (int64_t)gstride * blk;
        if (lane < 3) G[lane] = lane == 0 ? cnt[0] : (lane == 1 ? cnt[1] : cnt[2]);
#pragma unroll
        for (int ax = 0; ax < 3; ++ax)
            if (lane < cnt[ax]) G[3 + ax * A.kseg + lane] = seg[wv][ax][lane];
        const int kb = B.sample * A.K1 * A.K1;
        for_rects(P, B.rs, A.K1, cnt[0], cnt[1], cnt[2], seg[wv][0], seg[wv][1], seg[wv][2], lane,
                  [&](int, int key, int items, uint32_t, uint32_t, uint32_t, int) {
                      if (A.K1 == 1)
                          same += items;
                      else
                          atomicAdd(&A.key_count[kb + key], (unsigned long long)items);
                  });
        if (A.K1 == 1 && !A.one_key) {
            for (int d = kWave / 2; d > 0; d >>= 1) same += __shfl_xor(same, d);
            if (lane == 0 && same) atomicAdd(&A.key_count[kb], (unsigned long long)same);
            same = 0;
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");  // seg is reused
    }
    if (!A.one_key) return;
    // (one atomic per workgroup: one per block and rectangle on a single counter
    // took 0.3 ms of a count of 400,000 positions without regions)
    if (same) atomicAdd(&s_same, same);
    __syncthreads();
    if (threadIdx.x == 0 && s_same) atomicAdd(&A.key_count[0], (unsigned long long)s_same);
}

// One wave per shape block: its items, counting-sorted by key (sample, R_s,
// R_p).  Items beyond the capacity are not written and raise the overflow flag
// (the host then grows the capacity and counts again).
__global__ __launch_bounds__(kPlanThreads) void k_emit_items(PlanLaunch A) {
    const int lane = threadIdx.x & (kWave - 1);
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int nblk = A.boff[A.ncells];
    const int gstride = 3 + 3 * A.kseg;
    // a single key: the workgroup's items are counted first and reserved with one atomic
    __shared__ unsigned long long s_next[kPlanWaves];
    __shared__ int s_count[kPlanWaves];
    if (A.one_key) {
        int c = 0;
        for (int blk = blockIdx.x * kPlanWaves + wv; blk < nblk; blk += gridDim.x * kPlanWaves) {
            const uint32_t *G = A.geo + (int64_t)gstride * blk;
            for_rects(A.ps[0], 0, A.K1, G[0], G[1], G[2], G + 3, G + 3 + A.kseg, G + 3 + 2 * A.kseg, lane,
                      [&](int, int, int n, uint32_t, uint32_t, uint32_t, int) { c += n; });
        }
        for (int d = kWave / 2; d > 0; d >>= 1) c += __shfl_xor(c, d);
        if (lane == 0) s_count[wv] = c;
        __syncthreads();
        if (threadIdx.x == 0) {
            int all = 0;
            for (int k = 0; k < kPlanWaves; ++k) all += s_count[k];
            unsigned long long at = all ? atomicAdd(&A.key_cursor[0], (unsigned long long)all) : 0;
            for (int k = 0; k < kPlanWaves; ++k) {
                s_next[k] = at;
                at += s_count[k];
            }
        }
        __syncthreads();
    }
    for (int blk = blockIdx.x * kPlanWaves + wv; blk < nblk; blk += gridDim.x * kPlanWaves) {
        const Block B = A.blocks[blk];
        const PlanSample &P = A.ps[B.sample];
        const uint32_t *G = A.geo + (int64_t)gstride * blk;
        const int kb = B.sample * A.K1 * A.K1;
        for_rects(P, B.rs, A.K1, G[0], G[1], G[2], G + 3, G + 3 + A.kseg, G + 3 + 2 * A.kseg, lane,
                  [&](int t, int key, int n, uint32_t a, uint32_t b, uint32_t r, int rp) {
                      unsigned long long *next = A.one_key ? &s_next[wv] : &A.key_cursor[kb + key];
                      const int64_t slot = A.key_off[kb + key] + (int64_t)atomicAdd(next, (unsigned long long)n);
                      if (slot + n > A.cap) {
                          atomicOr(A.overflow, 1ull);
                          return;
                      }
                      const int ca = seg_cls(a), cb = seg_cls(b), cz = r == ~0u ? 3 : seg_cls(r);
                      // mixed shift classes take the per-pair minimum-image wrap; a
                      // non-periodic box never wraps (classes are always 0 there, and
                      // the tail's "any line-of-sight value" class means no shift)
                      const bool wrap = P.periodic && ((ca == 3) || (cb == 3) || (cz == 3));
                      const int sh = (ca == 3 ? 0 : ca) | ((cb == 3 ? 0 : cb) << 2) | ((cz == 3 ? 0 : cz) << 4) |
                                     (wrap ? 64 : 0);
                      const int cols = (seg_j1(a) - seg_j0(a) + 1) * (seg_j1(b) - seg_j0(b) + 1);
                      Item it;
                      it.blk = blk;
                      it.w = (rp & 0xffff) | (sh << 16) | (cz << 24);
                      it.ja = (uint16_t)seg_j0(a);
                      it.jb = (uint16_t)seg_j0(b);
                      it.wb = (uint16_t)(seg_j1(b) - seg_j0(b) + 1);
                      it.k0 = (uint16_t)(r == ~0u ? P.g.nz : seg_j0(r));
                      it.k1 = (uint16_t)(r == ~0u ? P.g.nz + 1 : seg_j1(r) + 1);
                      it.np = 0;
                      it.key = kb + key;
                      for (int i = 0; i < n; ++i) {
                          it.c0 = i * P.cpi;
                          it.nc = (uint16_t)(cols - it.c0 < P.cpi ? cols - it.c0 : P.cpi);
                          A.items[slot + i] = it;
                          if (A.sort_key)
                              A.sort_key[slot + i] = (A.sort_shift < 64 ? (unsigned long long)(kb + key) << A.sort_shift : 0ull) |
                                                     ((unsigned long long)blk * (kMaxSegs * kMaxSegs * (kMaxSegs + 1)) + t);
                      }
                  });
    }
}

// The lane's column of an item, and its positions.
__device__ __forceinline__ void item_column(const ColumnView &v, const double *bb, int ja, int jb, int wb, int nc,
                                            int c0, int k0, int k1, int w, int lane, int &pb, int &n) {
    pb = 0;
    n = 0;
    if (lane < nc) {
        // the first column's row and place in it are the wave's; the lane's
        // quotient is of numbers below 2^13, exact in FP32 from half a unit up
        const int row0 = c0 / wb, x = c0 - row0 * wb + lane;
        const int row = (int)(((float)x + 0.5f) * __frcp_rn((float)wb));
        column_positions(v, bb[0], bb[1], bb[2], bb[3], bb[4], bb[5], ja + row0 + row, jb + (x - row * wb), k0, k1,
                         (w >> 16) & 0xff, (w >> 24) & 3, pb, n);
    }
}

// One wave per item: its positions and balancing cost.
__global__ __launch_bounds__(kPlanThreads) void k_item_cost(const PlanSample *ps, const Block *blocks,
                                                            const double *bbox, const int64_t *n_items, Item *items,
                                                            int64_t *cost, unsigned long long *candidates) {
    __shared__ unsigned long long cand_l;
    const int lane = threadIdx.x & (kWave - 1);
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    if (threadIdx.x == 0) cand_l = 0;
    __syncthreads();
    const int64_t n = *n_items;
    unsigned long long cand = 0;
    for (int64_t i = (int64_t)blockIdx.x * kPlanWaves + wv; i < n; i += (int64_t)gridDim.x * kPlanWaves) {
        // (wave-uniform: read through the scalar cache)
        const MIA_CONST int32_t *ip = (const MIA_CONST int32_t *)items + 8 * i;
        const int blk = ip[0], w = ip[1], jj = ip[2], wn = ip[3], c0 = ip[4], kk = ip[5];
        const MIA_CONST int32_t *bp = (const MIA_CONST int32_t *)blocks + 4 * (int64_t)blk;
        const MIA_CONST double *bc = (const MIA_CONST double *)bbox + 6 * (int64_t)blk;
        const double bb[6] = {bc[0], bc[1], bc[2], bc[3], bc[4], bc[5]};
        const int ns = bp[1];
        int pb, np;
        item_column(column_view((const MIA_CONST PlanSample *)ps + bp[2]), bb, jj & 0xffff, (jj >> 16) & 0xffff,
                    wn & 0xffff, (wn >> 16) & 0xffff, c0, kk & 0xffff, (kk >> 16) & 0xffff, w, lane, pb, np);
        for (int d = kWave / 2; d > 0; d >>= 1) np += __shfl_xor(np, d);
        if (lane == 0) {
            items[i].np = np;
            // a wave pays for whole 64-lane position batches plus a fixed
            // per-item overhead, whatever the item's true pair count
            cost[i] = (int64_t)ns * (((np + kWave - 1) / kWave) * kWave) + kItemOverhead;
            cand += (unsigned long long)ns * np;
        }
    }
    if (cand) atomicAdd(&cand_l, cand);
    __syncthreads();
    if (threadIdx.x == 0 && cand_l) atomicAdd(candidates, cand_l);
}

// Shape blocks: per (column, slab group) cell of every sample, the number of
// blocks of at most bsz shapes (count), then the blocks themselves at the
// scanned offsets (emit).  cell0[S + 1] locates each sample's cells.
__global__ void k_blocks(const PlanSample *ps, const int64_t *cell0, int S, int bsz,
                         int32_t *nb, const int32_t *boff, Block *blocks) {
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= cell0[S]) return;
    const int s = find_sample(cell0, S, c);
    const PlanSample &P = ps[s];
    const Grid &g = P.g;
    const int64_t local = c - P.cell0;
    const int col = (int)(local / (P.ng + 1)), grp = (int)(local % (P.ng + 1));
    const int64_t base = (int64_t)col * (g.nz + 1);
    int s0, n, rs;
    if (grp < P.ng) {
        s0 = P.sstart[base + grp * P.G];
        n = P.sstart[base + (grp + 1) * P.G] - s0;
        rs = region_of(g, col / g.nc, col % g.nc, grp * P.G);
    } else {
        s0 = P.sstart[base + g.nz];
        n = P.sstart[base + g.nz + 1] - s0;
        rs = 0;
    }
    if (!boff) {
        nb[c] = (n + bsz - 1) / bsz;
        return;
    }
    const int o = boff[c];
    for (int b = 0; b * bsz < n; ++b) {
        Block B;
        B.s0 = s0 + b * bsz;
        B.ns = n - b * bsz < bsz ? n - b * bsz : bsz;
        B.sample = s;
        B.rs = rs;
        blocks[o + b] = B;
    }
}

// n_items = total of the key counts (0 past the capacity); raw total kept for the host.
__global__ void k_items_total(const int64_t *key_off, int64_t nkeys, int64_t cap, int64_t *n_items,
                              unsigned long long *raw) {
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        const int64_t t = key_off[nkeys];
        // beyond the capacity the host counts again; nothing is scheduled
        *n_items = t <= cap ? t : 0;
        *raw = (unsigned long long)t;
    }
}

// Deterministic order of the items: the permutation of a stable sort by
// (key, block, rectangle) applied to the items and their costs.
__global__ void k_iota(int32_t *a, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = (int32_t)i;
}

// The planner keys of the items in a given order.
__global__ void k_item_keys(const int32_t *order, const int64_t *n_dev, int64_t cap, const Item *items,
                            unsigned long long *key) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < cap) key[i] = i < *n_dev ? (unsigned long long)items[order[i]].key : ~0ull;
}

__global__ void k_gather_items(const int32_t *order, const int64_t *n_dev, const Item *items, const int64_t *cost,
                               Item *items_out, int64_t *cost_out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= *n_dev) return;
    const int32_t o = order[i];
    items_out[i] = items[o];
    cost_out[i] = cost[o];
}

// The pair kernel's statistics, summed over their copies into the words the
// host reads back (one wave).
__device__ __forceinline__ void collect_stats(const unsigned long long *stat, unsigned long long *words) {
    const int lane = threadIdx.x;
    unsigned long long v[4] = {0, 0, 0, 0};
    if (lane < kStatCopies)
        for (int k = 0; k < 4; ++k) v[k] = stat[lane * kStatStride + k];
    for (int d = kWave / 2; d > 0; d >>= 1)
        for (int k = 0; k < 4; ++k) {
            const unsigned long long o = __shfl_down(v[k], d);
            v[k] = k < 2 ? v[k] + o : (o > v[k] ? o : v[k]);
        }
    if (lane == 0) {
        words[0] = v[0];
        words[6] = v[1];
        words[4] = v[2];
        words[5] = v[3];
    }
}

// Caller outputs from the accumulators: counts, DD (the pair count itself for
// unit weights), S+D, their tallies, SxD, the variance and the region stats.
__global__ void k_finalize(const FinSample *fs, const int64_t *fin0, int S, const unsigned long long *stat,
                           unsigned long long *words) {
    if (blockIdx.x == 0 && threadIdx.x < kWave) collect_stats(stat, words);
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= fin0[S]) return;
    const int s = find_sample(fin0, S, i);
    const FinSample &F = fs[s];
    const int64_t j = i - fin0[s];
    const int64_t nb = (int64_t)(1 + F.K) * F.B;
    if (j < nb) {
        const unsigned long long c = F.np[j];
        F.out.npairs[j] = c;
        if (F.out.dd) F.out.dd[j] = F.weighted ? F.dd[j] : (double)c;
        F.out.splus[j] = F.sp[j];
        if (j < F.B) {
            F.out.scross[j] = F.sx[j];
            if (F.out.variance) F.out.variance[j] = F.var_on ? F.var[j] : 0.0;
        }
        return;
    }
    const int64_t k = j - nb;  // region k < K
    if (F.out.region_stats) {
        double *r = F.out.region_stats + 4 * k;
        r[0] = (double)F.rcnt[k];
        r[1] = (double)F.rcnt[F.K + k];
        r[2] = F.rsum[k];
        r[3] = F.rsum[F.K + k];
    }
}

// Deterministic reduction, step 1: the histogram flushes of every wave of an
// all-static schedule (bounds from schedule_bounds(all_static)), which are the
// distinct planner keys among its items: the non-empty keys from the first to
// the last item that its range of batches touches (key_off: nkeys + 1 item
// offsets), 0 for an empty range.  Their exclusive scan numbers the slots.
__device__ __forceinline__ int64_t key_of_item(const int64_t *key_off, int64_t nkeys, int64_t i) {
    int64_t lo = 0, hi = nkeys - 1;  // largest k with key_off[k] <= i
    while (lo < hi) {
        const int64_t mid = (lo + hi + 1) >> 1;
        if (key_off[mid] <= i)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

// ne[k] = 1 when key k holds items; its exclusive scan counts the non-empty
// keys below k (empty keys between a wave's first and last key get no flush).
__global__ void k_key_nonempty(const int64_t *key_off, int64_t nkeys, int64_t *ne) {
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k < nkeys) ne[k] = key_off[k + 1] > key_off[k] ? 1 : 0;
}

// The item after the last one of which a range of batches that ends at b takes some.
__device__ __forceinline__ int64_t items_end(int64_t b) {
    return (b >> kBatchBits) + ((b & ((1ll << kBatchBits) - 1)) != 0 ? 1 : 0);
}

__global__ void k_slot_runs(const int64_t *bounds, int W, const int64_t *key_off, int64_t nkeys,
                            const int64_t *ne_pre, int64_t *runs) {
    const int w = blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= W) return;
    const int64_t b0 = bounds[(int64_t)w * kScheduleUnits], b1 = bounds[(int64_t)(w + 1) * kScheduleUnits];
    const int64_t i0 = b0 >> kBatchBits, i1 = items_end(b1);
    runs[w] = b1 > b0 ? ne_pre[key_of_item(key_off, nkeys, i1 - 1) + 1] - ne_pre[key_of_item(key_off, nkeys, i0)]
                      : 0;
}

// Neumaier's compensated addition: s + c carries the sum with the rounding
// error of every addition recovered in c.
__device__ __forceinline__ void neumaier(double &s, double &c, double v) {
    const double t = s + v;
    c += fabs(s) >= fabs(v) ? (s - t) + v : (v - t) + s;
    s = t;
}

// Deterministic reduction, step 2: the slots of one key are consecutive and are
// cut into pieces of kPieceSlots from the key's first; the first slot of a piece
// (its head) takes the piece's sum, and the second, where there is one, the sum's
// compensation, bin by bin.  One workgroup per piece and 256 bins: a count
// without regions has all its waves' slots in one key (200,000 positions, 6,144
// slots of 200 bins: 4.3 ms of finalisation in one workgroup, now 0.15).
constexpr int kPieceSlots = 32;

// The key's first slot.
__device__ __forceinline__ int64_t first_slot(const int64_t *slot_key, int64_t n, int64_t key) {
    int64_t lo = 0, hi = n;
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (slot_key[mid] < key)
            lo = mid + 1;
        else
            hi = mid;
    }
    return lo;
}

// Whether slot q is a head.
__device__ __forceinline__ bool head_slot(const int64_t *slot_key, int64_t n, int64_t q) {
    return (q - first_slot(slot_key, n, slot_key[q])) % kPieceSlots == 0;
}

__device__ __forceinline__ void sum_run(double *slot, int64_t o, int64_t step, int n) {
    double s = slot[o], c = 0.0;
    for (int k = 1; k < n; ++k) neumaier(s, c, slot[o + k * step]);
    slot[o] = s;
    slot[o + step] = c;
}

__global__ __launch_bounds__(256) void k_sum_slots(const int64_t *slot_total, const int64_t *slot_key,
                                                   unsigned long long *slot_np, double *slot_sp, double *slot_sx,
                                                   double *slot_dd, double *slot_var, int BO) {
    const int64_t n = *slot_total;
    for (int64_t q = blockIdx.x; q < n; q += gridDim.x) {
        if (!head_slot(slot_key, n, q)) continue;
        const int64_t key = slot_key[q];
        int run = 1;
        while (run < kPieceSlots && q + run < n && slot_key[q + run] == key) ++run;
        if (run == 1) continue;
        for (int b = blockIdx.y * blockDim.x + threadIdx.x; b < BO; b += gridDim.y * blockDim.x) {
            const int64_t o = q * BO + b;
            unsigned long long c = slot_np[o];
            for (int k = 1; k < run; ++k) c += slot_np[o + (int64_t)k * BO];
            slot_np[o] = c;
            sum_run(slot_sp, o, BO, run);
            sum_run(slot_sx, o, BO, run);
            if (slot_dd) sum_run(slot_dd, o, BO, run);
            if (slot_var) sum_run(slot_var, o, BO, run);
        }
    }
}

// The heads in slot order: heads[i] = slot << 1 | whether a second slot follows,
// *n_heads of them (one workgroup).
__global__ __launch_bounds__(1024) void k_slot_heads(const int64_t *slot_total, const int64_t *slot_key,
                                                     int64_t *heads, int64_t *n_heads) {
    __shared__ int s_cnt[1024 / kWave];
    const int64_t n = *slot_total;
    const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
    int64_t base = 0;
    for (int64_t q0 = 0; q0 < n; q0 += blockDim.x) {
        const int64_t q = q0 + threadIdx.x;
        const bool head = q < n && head_slot(slot_key, n, q);
        const uint64_t m = __ballot(head);
        if (lane == 0) s_cnt[wv] = __popcll(m);
        __syncthreads();
        int before = 0, all = 0;
        for (int k = 0; k < 1024 / kWave; ++k) {
            before += k < wv ? s_cnt[k] : 0;
            all += s_cnt[k];
        }
        if (head) {
            const bool two = q + 1 < n && slot_key[q + 1] == slot_key[q];
            heads[base + before + __popcll(m & ((1ull << lane) - 1))] = (q << 1) | (two ? 1 : 0);
        }
        base += all;
        __syncthreads();
    }
    if (threadIdx.x == 0) *n_heads = base;
}

// Step 3: caller outputs from the pieces' sums, one wave per output.  Output
// element (tally t, bin b) of a sample sums the heads of that sample whose key
// (R_s, R_p) includes region t - 1 (every head for t = 0): lane l every 64th
// from the l-th, then the lanes pairwise, all with compensated FP64 sums, in an
// order fixed by the heads.  Region stats as k_finalize.  (One thread per
// output over all slots took 8.5 ms for 8,000 slots of 200 bins and 28 tallies,
// waiting on one slot after the other.)
struct DetSum {
    double s, c;
    __device__ __forceinline__ void add(const double *slot, int64_t at, int64_t second) {
        neumaier(s, c, slot[at]);
        if (second >= 0) c += slot[second];
    }
    __device__ __forceinline__ void reduce() {
        for (int d = kWave / 2; d > 0; d >>= 1) {
            const double os = __shfl_down(s, d), oc = __shfl_down(c, d);
            neumaier(s, c, os);
            c += oc;
        }
    }
};

__global__ __launch_bounds__(256) void k_finalize_det(const FinSample *fs, const int64_t *fin0, int S,
                                                      const int64_t *heads, const int64_t *n_heads,
                                                      const int64_t *slot_key, const unsigned long long *slot_np,
                                                      const double *slot_sp, const double *slot_sx,
                                                      const double *slot_dd, const double *slot_var, int BO,
                                                      const unsigned long long *stat, unsigned long long *words) {
    if (blockIdx.x == 0 && threadIdx.x < kWave) collect_stats(stat, words);
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t i = (int64_t)blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave;
    if (i >= fin0[S]) return;
    const int s = find_sample(fin0, S, i);
    const FinSample &F = fs[s];
    const int64_t j = i - fin0[s];
    const int64_t nb = (int64_t)(1 + F.K) * F.B;
    if (j >= nb) {
        const int64_t k = j - nb;  // region k < K
        if (F.out.region_stats && lane == 0) {
            double *r = F.out.region_stats + 4 * k;
            r[0] = (double)F.rcnt[k];
            r[1] = (double)F.rcnt[F.K + k];
            r[2] = F.rsum[k];
            r[3] = F.rsum[F.K + k];
        }
        return;
    }
    const int t = (int)(j / F.B), b = (int)(j % F.B);
    // the sample's heads: keys [s << 32, (s + 1) << 32) of the ascending key list
    const int64_t n = *n_heads;
    auto first_of = [&](int64_t key) {
        int64_t lo = 0, hi = n;
        while (lo < hi) {
            const int64_t mid = (lo + hi) >> 1;
            if (slot_key[heads[mid] >> 1] < key)
                lo = mid + 1;
            else
                hi = mid;
        }
        return lo;
    };
    const int64_t h0 = first_of((int64_t)s << 32), h1 = first_of((int64_t)(s + 1) << 32);
    unsigned long long c = 0;
    DetSum sp{0.0, 0.0}, dd{0.0, 0.0}, sx{0.0, 0.0}, vr{0.0, 0.0};
    for (int64_t h = h0 + lane; h < h1; h += kWave) {
        const int64_t e = heads[h], key = slot_key[e >> 1];
        const int rs = (int)((key >> 16) & 0xffff), rp = (int)(key & 0xffff);
        if (t > 0 && rs != t - 1 && rp != t - 1) continue;
        const int64_t at = (e >> 1) * BO + b, second = (e & 1) ? at + BO : -1;
        c += slot_np[at];
        sp.add(slot_sp, at, second);
        if (F.weighted) dd.add(slot_dd, at, second);
        if (t == 0) {
            sx.add(slot_sx, at, second);
            if (F.var_on) vr.add(slot_var, at, second);
        }
    }
    for (int d = kWave / 2; d > 0; d >>= 1) c += __shfl_down(c, d);
    sp.reduce();
    dd.reduce();
    sx.reduce();
    vr.reduce();
    if (lane) return;
    c += F.np[j];  // spilled counts
    F.out.npairs[j] = c;
    if (F.out.dd) F.out.dd[j] = F.weighted ? dd.s + dd.c : (double)c;
    F.out.splus[j] = sp.s + sp.c;
    if (t == 0) {
        F.out.scross[b] = sx.s + sx.c;
        if (F.out.variance) F.out.variance[b] = F.var_on ? vr.s + vr.c : 0.0;
    }
}

// ---------------------------------------------------------------------------
// pair kernel

struct PairArgs {
    const Item *items;
    const PlanSample *ps;        // position columns of every sample
    const double *bbox;          // bounding boxes of the blocks' shapes
    const unsigned long long *overflow;  // planner's capacity flag
    const Block *blocks;
    const int64_t *n_items;      // device: work items in the list
    int n_waves;
    const int64_t *key_off;      // first item of every key
    const int64_t *bounds;       // schedule unit -> first item, groups * kScheduleUnits + 3
    int *queue;                  // tail-chunk counter, zero at launch
    int mode, n_r, n_2, weighted, var, nbins;
    const double *T, *X;         // exact thresholds (global copy)
    double T0, Tn, X0, Xn;       // domain bounds (rppi: s and pi; rmu: r^2)
    float lgs, lgc;              // r bin guess: log2(v) * lgs + lgc
    float xs, xc;                // mu: (mu + 1) * xs + xc
    double xs64, xc64;           // pi: pi * xs64 + xc64
    float dr, d2f;               // guard bands: exact path when the fraction of a guess is below
    double d2;
    int scan;                    // 1: the exact path scans every threshold (guard band of a whole bin)
    const SampleDev *samples;
    int hist_stride;             // bytes of a histogram
    int apart;                   // the counts lie in front of the sums
    int shared, copies;          // the waves of a workgroup share `copies` histograms (else one per wave)
    int bin_off, nbins_out;      // this pass's first output bin (r0 * n_2) and the output's B
    // kStatCopies copies of: pairs binned exactly, wave-iterations (a 64-lane
    // position batch against one shape), and the wall-clock span of the busy
    // workgroups: max of ~start, max of end
    unsigned long long *stat;
    // deterministic reduction: the j-th histogram flush of wave w goes to
    // slot slot0[w] + j (all output bins of the pass, plain stores) with its
    // planner key; k_finalize_det sums the slots in slot order
    int det, K1;
    int64_t slot_cap;            // slots allocated (waves + planner keys bound every wave's flushes)
    const int64_t *slot0;
    int64_t *slot_key;
    unsigned long long *slot_np;
    double *slot_sp, *slot_sx, *slot_dd, *slot_var;
};

// One bin of a histogram: S+D and SxD, then DD (weighted samples) and the sum of
// e+^2 (variance requested), and the pair count.  Bins lie an odd number of 8-byte
// words apart, so that those of a wave's lanes spread over all LDS banks (32 bytes
// apart, three sums with their count, only every fourth pair of banks starts a
// bin: 300,001 weighted positions, 100,003 shapes, 200 bins 14.6 ms of pair kernel,
// now 12.0).  Two or four sums are padded to three or five words by the count; of
// three, the counts lie in front of the sums (APART), bin b's b + 1 words before
// them, which also leaves LDS for more waves (360 weighted bins: 16 per CU instead
// of 12, 21.9 -> 17.0 ms in 300,001 positions).  Two and four sums have the counts
// apart in the deterministic mode's larger binnings (pair_config).
template <bool WEIGHTED, bool VAR, bool APART>
struct Slot {
    static constexpr int kSums = 2 + WEIGHTED + VAR;
    static constexpr bool kApart = APART;
    static constexpr uint32_t kBytes = kApart ? 8 * kSums : 8 * kSums + 8;
    static_assert(APART || kSums != 3, "three sums have their counts apart");
    uint32_t c;
    double v[kSums];  // S+D, SxD, [DD], [sum of e+^2]
};
// bytes of a histogram of nbins bins
constexpr size_t hist_bytes(int nbins, bool weighted, bool var, bool apart) {
    const size_t n = (size_t)nbins, sums = 8 * (2 + weighted + var) * n;
    return (sums + (apart ? (4 * n + 7) & ~(size_t)7 : 8 * n) + 15) & ~(size_t)15;
}
// bytes of the counts in front of the sums
template <bool WEIGHTED, bool VAR, bool APART>
__device__ __forceinline__ int front_bytes(int nbins) {
    return Slot<WEIGHTED, VAR, APART>::kApart ? (4 * nbins + 7) & ~7 : 0;
}

// Shape record {a, b, l, ax, ay, e*w, w, 2*e*w} read through the scalar cache:
// the inner loop is uniform over shapes, so every field lands in SGPRs.
typedef const __attribute__((address_space(4))) double *ShapePtr;

// The place of bin b's count in a histogram.
template <bool WEIGHTED, bool VAR, bool APART>
__device__ __forceinline__ uint32_t *bin_count(char *sums, int b) {
    typedef Slot<WEIGHTED, VAR, APART> BinSlot;
    return BinSlot::kApart ? (uint32_t *)sums - 1 - b
                           : (uint32_t *)(sums + (uint32_t)b * BinSlot::kBytes + 8 * BinSlot::kSums);
}

// One bin of a histogram, summed over its copies and cleared.
template <bool WEIGHTED, bool VAR, bool APART>
__device__ __forceinline__ Slot<WEIGHTED, VAR, APART> take_bin(const PairArgs &P, char *hist, int copies, int b) {
    typedef Slot<WEIGHTED, VAR, APART> BinSlot;
    BinSlot t{};
    hist += front_bytes<WEIGHTED, VAR, APART>(P.nbins);
    for (int k = 0; k < copies; ++k, hist += P.hist_stride) {
        double *v = (double *)(hist + (uint32_t)b * BinSlot::kBytes);
        uint32_t *c = bin_count<WEIGHTED, VAR, APART>(hist, b);
        if (*c == 0) continue;
        t.c += *c;
        *c = 0;
#pragma unroll
        for (int i = 0; i < BinSlot::kSums; ++i) {
            t.v[i] += v[i];
            v[i] = 0.0;
        }
    }
    return t;
}

// c pairs of the pass's bin b for the total and the tallies of both regions.
__device__ __forceinline__ void add_pairs(const PairArgs &P, const SampleDev &S, int rs, int rp, int b,
                                          unsigned long long c) {
    const int gb = b + P.bin_off;  // the pass's local bin in the output grid
    atomicAdd(&S.npairs[gb], c);
    if (S.K > 0) {
        atomicAdd(&S.npairs[(int64_t)(1 + rs) * P.nbins_out + gb], c);
        if (rp != rs) atomicAdd(&S.npairs[(int64_t)(1 + rp) * P.nbins_out + gb], c);
    }
}

// A wave takes all but one pair of every count to the 64-bit sums, with adds of
// other waves in flight: the histogram's 32-bit counts then stay below 2^32 whatever
// its waves test before the next flush (a bin without a pair would not be flushed).
template <bool WEIGHTED, bool VAR, bool APART>
__device__ void spill_counts(const PairArgs &P, char *hist, int copies, const SampleDev &S, int rs, int rp, int lane) {
    for (int b = lane; b < P.nbins; b += kWave) {
        char *sums = hist + front_bytes<WEIGHTED, VAR, APART>(P.nbins);
        unsigned long long c = 0;
        for (int k = 0; k < copies; ++k, sums += P.hist_stride) {
            uint32_t *at = bin_count<WEIGHTED, VAR, APART>(sums, b);
            // (a count of one or more never falls below one before the flush)
            if (__hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) > 1)
                c += __hip_atomic_exchange(at, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) - 1;
        }
        if (c) add_pairs(P, S, rs, rp, b, c);
    }
}

template <bool WEIGHTED, bool VAR, bool APART>
__device__ void flush_hist(const PairArgs &P, char *hist, int copies, const SampleDev &S, int rs, int rp, int tid,
                           int nthr) {
    const bool dd = WEIGHTED, vr = VAR;
    const int B = P.nbins;
    const int BO = P.nbins_out;
    for (int b = tid; b < B; b += nthr) {
        const Slot<WEIGHTED, VAR, APART> t = take_bin<WEIGHTED, VAR, APART>(P, hist, copies, b);
        const uint32_t c = t.c;
        const double vsp = t.v[0], vsx = t.v[1];
        double vdd = 0.0, vvr = 0.0;
        if constexpr (WEIGHTED) vdd = t.v[2];
        if constexpr (VAR) vvr = t.v[WEIGHTED ? 3 : 2];
        if (c == 0) continue;
        const int gb = b + P.bin_off;
        add_pairs(P, S, rs, rp, b, c);
        atomicAdd(&S.sp[gb], vsp);
        atomicAdd(&S.sx[gb], vsx);
        if (dd && S.dd) atomicAdd(&S.dd[gb], vdd);
        if (vr && S.var) atomicAdd(&S.var[gb], vvr);
        if (S.K > 0) {
            int64_t o = (int64_t)(1 + rs) * BO + gb;
            atomicAdd(&S.sp[o], vsp);
            if (dd && S.dd) atomicAdd(&S.dd[o], vdd);
            if (rp != rs) {
                o = (int64_t)(1 + rp) * BO + gb;
                atomicAdd(&S.sp[o], vsp);
                if (dd && S.dd) atomicAdd(&S.dd[o], vdd);
            }
        }
    }
}

// A slot's key: sample << 32 | R_s << 16 | R_p (regions < 2^16), ascending in
// the planner's key order.
__device__ __forceinline__ int64_t slot_key_of(int sample, int rs, int rp) {
    return ((int64_t)sample << 32) | ((int64_t)rs << 16) | (int64_t)rp;
}

// The deterministic flush: the wave's histogram (every bin of the pass, the
// empty ones too) is stored into its slot instead of added by atomics.
template <bool WEIGHTED, bool VAR, bool APART>
__device__ void flush_slot(const PairArgs &P, char *hist, int copies, int64_t slot, int64_t key, int tid, int nthr) {
    if (slot >= P.slot_cap) return;  // cannot happen: the slot plan counts every flush
    for (int b = tid; b < P.nbins; b += nthr) {
        const Slot<WEIGHTED, VAR, APART> t = take_bin<WEIGHTED, VAR, APART>(P, hist, copies, b);
        const int64_t o = slot * P.nbins_out + P.bin_off + b;
        P.slot_np[o] = t.c;
        P.slot_sp[o] = t.v[0];
        P.slot_sx[o] = t.v[1];
        if constexpr (WEIGHTED) P.slot_dd[o] = t.v[2];
        if constexpr (VAR) P.slot_var[o] = t.v[WEIGHTED ? 3 : 2];
    }
    if (tid == 0) P.slot_key[slot] = key;
}


// r^2 summed in the reference's column order x, y, z: (a^2 + b^2) + l^2 with
// the line of sight along z (LZ), else (a^2 + l^2) + b^2 (line of sight x:
// (l^2 + a^2) + b^2, the same value since FP64 addition commutes).
template <bool LZ>
__device__ __forceinline__ double r2_column_order(double s, double a2, double b2, double l2) {
    return LZ ? s + l2 : (a2 + l2) + b2;
}

// #{k in 1..n-1 : E[k] <= v}, the exact bin of v in [E[0], E[n]).
__device__ __forceinline__ int count_edges(const double *E, int n, double v) {
    int k = 0;
    for (int i = 1; i < n; ++i) k += (E[i] <= v);
    return k;
}

// The same count from a guess g of v's position in bin units that is off by
// less than half a bin: with e the integer nearest g, every edge below E[e]
// lies below v and every edge above it above v, so one comparison decides.
// v lies in [E[0], E[n]) (the domain test), so e = 0 and e = n need none.
__device__ __forceinline__ int edge_near(const double *E, int n, double v, float g) {
    const int e = (int)rintf(g);
    if (e <= 0) return 0;
    if (e >= n) return n - 1;
    return e - 1 + (E[e] <= v ? 1 : 0);
}
__device__ __forceinline__ int edge_near(const double *E, int n, double v, double g) {
    const int e = (int)rint(g);
    if (e <= 0) return 0;
    if (e >= n) return n - 1;
    return e - 1 + (E[e] <= v ? 1 : 0);
}


// Per-sample values the pair loop needs, read once per item through the
// scalar cache (they are wave-uniform and end up in SGPRs).
struct SampleView {
    const double *prec;
    const double *srec;
    double L, half;
    int los;
};

__device__ __forceinline__ SampleView load_view(const SampleDev *sd) {
    const MIA_CONST SampleDev *c = (const MIA_CONST SampleDev *)sd;
    SampleView v;
    v.prec = c->prec;
    v.srec = c->srec;
    v.L = c->L;
    v.half = c->half;
    v.los = c->los;
    return v;
}

// Periodic handling of an item: no shift on any axis, a constant shift per
// axis, or the reference's per-pair minimum-image wrap.
enum { SH_NONE = 0, SH_CONST = 1, SH_WRAP = 2 };

// A lane's pending histogram slot: consecutive pairs of one lane (one
// position against the shapes of a block) that land in the same slot are
// summed in registers and reach the LDS histogram as one atomic per run,
// which cuts the same-address collisions of the hot (outer r) bins.
struct Pend {
    uint32_t at;  // LDS address of the bin; counts in front of the sums: the bin's number
    uint32_t c;
    double sp, sx, dd, vr;
};

#define MIA_LDS __attribute__((address_space(3)))

template <class T>
__device__ __forceinline__ void lds_add(uint32_t at, T v) {
    __hip_atomic_fetch_add((MIA_LDS T *)at, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// hist: LDS address of the histogram's sums; with counts in front of them 4 bytes
// less, so that no offset is negative.  The other kind of pending run holds its
// bin's address, and a flush computes none.
template <bool WEIGHTED, bool VAR, bool APART>
__device__ __forceinline__ uint32_t pend_at(uint32_t hist, int b) {
    typedef Slot<WEIGHTED, VAR, APART> BinSlot;
    return BinSlot::kApart ? (uint32_t)b : __umul24(b, BinSlot::kBytes) + hist;
}

template <bool WEIGHTED, bool VAR, bool APART>
__device__ __forceinline__ void hist_add(uint32_t hist, const Pend &p) {
    typedef Slot<WEIGHTED, VAR, APART> BinSlot;
    uint32_t at = p.at;
    if constexpr (BinSlot::kApart) {
        lds_add<uint32_t>((uint32_t)(__mul24((int)p.at, -4) + (int)hist), p.c);
        at = __umul24(p.at, BinSlot::kBytes) + hist + 4;
    } else {
        lds_add<uint32_t>(at + 8 * BinSlot::kSums, p.c);
    }
    lds_add<double>(at, p.sp);
    lds_add<double>(at + 8, p.sx);
    if constexpr (WEIGHTED) lds_add<double>(at + 16, p.dd);
    if constexpr (VAR) lds_add<double>(at + (WEIGHTED ? 24 : 16), p.vr);
}

template <int MODE, int SH, bool WEIGHTED, bool VAR, bool APART, bool LZ>
__device__ __forceinline__ void one_pair(const PairArgs &P, const SampleView &S, bool valid,
                                         double pa, double pb, double pl, double pw, double qa,
                                         double qb, double ql, double qax, double qay, double qew,
                                         double qw, double q2ew, double sha, double shb, double shl,
                                         uint32_t hist, uint32_t row, const double *T, const double *X,
                                         uint32_t &nre, Pend &pd, float vlgc, float vlg2, double vxs, double vxc) {
    const int n_r = P.n_r, n_2 = P.n_2;
    // the reference's own FP64 separation (measure_w_box_jk.py:159-162)
    double da = qa - pa, db = qb - pb, dl = ql - pl;
    if (SH == SH_WRAP) {
        da = wrap_sep(da, S.L, S.half);
        db = wrap_sep(db, S.L, S.half);
        dl = wrap_sep(dl, S.L, S.half);
    } else if (SH == SH_CONST) {
        da = da + sha;
        db = db + shb;
        dl = dl + shl;
    }
    double a2 = da * da, b2 = db * db;
    double s = a2 + b2;
    double rv;
    bool in;
    if (MODE == MIA_RPPI) {
        rv = s;
        in = valid & (s >= P.T0) & (s < P.Tn) & (dl >= P.X0) & (dl < P.Xn);
    } else {
        rv = r2_column_order<LZ>(s, a2, b2, dl * dl);
        in = valid & (s > 0.0) & (rv >= P.T0) & (rv < P.Tn);
    }
    if (in) {
        // bins: FP32 guess; exact FP64 threshold count when the guess lies
        // within the guard band of a bin edge (every edge, the domain edges
        // included, so no clamping is needed)
        float rv32 = (float)rv;
        const float gr = __fmaf_rn(__log2f(rv32), P.lgs, vlgc);
        const bool near_r = __builtin_amdgcn_fractf(gr) < P.dr;
        // pi: an FP64 guess (one FMA; its error is ~1e-14 bins, so a 1e-9 guard
        // band); mu = pi / r: an FP32 guess from rsqrt.  The constants of the
        // guesses hold half the guard band, so a guess close to an edge on
        // either side has a fraction below the whole band
        int i2;
        double g2;
        bool near2;
        if (MODE == MIA_RPPI) {
            g2 = fma(dl, vxs, vxc);
            near2 = __builtin_amdgcn_fract(g2) < P.d2;
            i2 = (int)g2;
        } else {
            const float g2f = __fmaf_rn(__fmaf_rn((float)dl, __builtin_amdgcn_rsqf(rv32), 1.0f), P.xs, vlg2);
            near2 = __builtin_amdgcn_fractf(g2f) < P.d2f;
            i2 = (int)g2f;
            g2 = g2f;
        }
        // truncation is floor for the non-negative guesses; a guess within
        // the guard band of an integer (an edge, or a slightly negative
        // guess at the lower domain edge) takes the exact path
        int ir = (int)gr;
        const bool near = near_r | near2;
        if (near) {
            if (P.scan) {
                ir = count_edges(T, n_r, rv);
                if (MODE == MIA_RPPI) {
                    i2 = count_edges(X, n_2, dl);
                } else {
                    double mu64 = dl / sqrt(rv);
                    i2 = mu64 < X[0] ? n_2 - 1 : count_edges(X, n_2, mu64);
                }
            } else {
                ir = edge_near(T, n_r, rv, gr);
                if (MODE == MIA_RPPI) {
                    i2 = edge_near(X, n_2, dl, g2);
                } else {
                    double mu64 = dl / sqrt(rv);
                    i2 = mu64 < X[0] ? n_2 - 1 : edge_near(X, n_2, mu64, g2);
                }
            }
            ++nre;
        }
        // e+ = e cos 2phi = e (2 cos^2 phi - 1), ex = e sin 2phi = 2 e cos phi |sin phi|
        // (|.| because phi = arccos(d) lies in [0, pi]); cos phi = t/r_p,
        // |sin phi| = |c|/r_p with t, c the dot and cross products.
        double t = fma(da, qax, db * qay);
        double c = fma(da, qay, -(db * qax));
        double r0 = __builtin_amdgcn_rcp(s);
        double inv = fma(r0, fma(-s, r0, 1.0), r0);
        // 2 e w t / r_p^2: e+ = that * t - e w, ex = that * |c|
        double tw = (q2ew * t) * inv;
        double ep = fma(tw, t, -qew);
        double ex = tw * fabs(c);
        if (fabs(c) < fabs(t) * kSinExact) {
            // nearly parallel: the reference's d may round outside [-1, 1],
            // where arccos gives NaN and the pair adds no e+ (measure_w_box_jk.py:170-175)
            double rp = sqrt(s);
            double d = 0.0 + (da / rp) * qax;
            d = d + (db / rp) * qay;
            if (!(fabs(d) <= 1.0)) {
                ep = 0.0;
                ex = 0.0;
            }
        }
        if (WEIGHTED) {
            ep = pw * ep;
            ex = pw * ex;
        }
        const uint32_t at = Slot<WEIGHTED, VAR, APART>::kApart
                                ? (uint32_t)(__mul24(ir, n_2) + i2)
                                : __umul24(ir, row) + (__umul24(i2, Slot<WEIGHTED, VAR, APART>::kBytes) + hist);
        double dd = WEIGHTED ? pw * qw : 0.0;
        double vr = VAR ? ep * ep : 0.0;
        // a new slot flushes the pending run; the run then restarts from this
        // pair: keep = 0 drops the old sums (fma(0, sum, x) = x, fma(1, sum, x)
        // = sum + x, both exactly as the plain assignment and addition)
        const bool nw = at != pd.at;
        if (nw) hist_add<WEIGHTED, VAR, APART>(hist, pd);
        const double keep = nw ? 0.0 : 1.0;
        pd.at = at;
        pd.c = (nw ? 0u : pd.c) + 1u;
        pd.sp = fma_into(keep, pd.sp, ep);
        pd.sx = fma_into(keep, pd.sx, ex);
        if (WEIGHTED) pd.dd = fma_into(keep, pd.dd, dd);
        if (VAR) pd.vr = fma_into(keep, pd.vr, vr);
    }
}

// An item's np positions lie in the columns of its lanes (lane c: positions
// [pb, pb + n)); item coordinate k runs over them column by column.  Lane l
// takes coordinates l * nb .. l * nb + nb - 1, one per batch: a batch then
// spans all columns and the whole line-of-sight range of the item, and its
// pairs spread over many (r, pi) bins (64 consecutive positions mostly share a
// few: with them same-address LDS atomics bound the kernel, 9.9 against 8.6 ms on
// a million clustered positions, 200,000 shapes).
struct ColumnWalk {
    int pb, end;        // own column: first position minus its first coordinate; end coordinate
    int c, base, ce;    // the column the lane reads from
    int np, nb;

    // batches are read from bt0 on, in ascending order
    __device__ __forceinline__ void begin(int lane, int pb_, int n, int bt0) {
        end = n;
#pragma unroll
        for (int d = 1; d < kWave; d <<= 1) {
            const int o = __shfl_up(end, d);
            end += lane >= d ? o : 0;
        }
        pb = pb_ - (end - n);
        np = __builtin_amdgcn_readlane(end, kWave - 1);
        nb = (np + kWave - 1) / kWave;
        // the first column that ends past the lane's first coordinate
        const int k = lane * nb + bt0 < np ? lane * nb + bt0 : np - 1;
        c = 0;
#pragma unroll
        for (int d = kWave / 2; d > 0; d >>= 1) c += __shfl(end, c + d - 1) <= k ? d : 0;
        base = __shfl(pb, c);
        ce = __shfl(end, c);
    }
    // the lane's position of batch bt (a lane past the end gets a valid one)
    __device__ __forceinline__ int position(int bt, int lane, bool &v) {
        int k = bt + lane * nb;
        v = k < np;
        k = v ? k : np - 1;
        while (__any(k >= ce)) {  // every lane takes part: a shuffle reads active lanes only
            c += k >= ce ? 1 : 0;
            base = __shfl(pb, c);
            ce = __shfl(end, c);
        }
        return base + k;
    }
};

template <int MODE, int SH, bool WEIGHTED, bool VAR, bool APART, bool LZ>
__device__ __forceinline__ void run_item(const PairArgs &P, const SampleView &S, int cpb, int cn, int bt0, int bt1,
                                         int shifts, ShapePtr shp, int ns, uint32_t hist,
                                         const double *T, const double *X, int lane,
                                         uint32_t &nre, uint64_t &iterations) {
    const double L = S.L;
    const double sha = SH == SH_CONST ? shift_val(shifts & 3, L) : 0.0;
    const double shb = SH == SH_CONST ? shift_val((shifts >> 2) & 3, L) : 0.0;
    const double shl = SH == SH_CONST ? shift_val((shifts >> 4) & 3, L) : 0.0;
    // the additive constants of the FP32 bin guesses, held in VGPRs for the
    // whole item (a VOP3 FMA reads one scalar operand; the other would be
    // copied into a VGPR on every pair)
    float vlgc, vlg2 = 0.0f;
    double vxs = 0.0, vxc = 0.0;
    asm volatile("v_mov_b32 %0, %1" : "=v"(vlgc) : "s"(P.lgc));
    if (MODE == MIA_RPPI) {
        asm volatile("v_mov_b64 %0, %1" : "=v"(vxs) : "s"(P.xs64));
        asm volatile("v_mov_b64 %0, %1" : "=v"(vxc) : "s"(P.xc64));
    } else {
        asm volatile("v_mov_b32 %0, %1" : "=v"(vlg2) : "s"(P.xc));
    }
    ColumnWalk walk;
    walk.begin(lane, cpb, cn, bt0);
    iterations += (uint64_t)(bt1 - bt0) * ns;
    // an empty run adds its zeros to some bin, another one for every lane
    const uint32_t row = (uint32_t)P.n_2 * Slot<WEIGHTED, VAR, APART>::kBytes;
    Pend pd{pend_at<WEIGHTED, VAR, APART>(hist, lane < P.nbins ? lane : 0), 0, 0, 0, 0, 0};
    // positions are loaded one batch ahead
    bool vn;
    const double2 *prn = (const double2 *)(S.prec + 4 * (int64_t)walk.position(bt0, lane, vn));
    double2 abn = prn[0], lwn = prn[1];
    for (int bt = bt0; bt < bt1; ++bt) {
        const bool v0 = vn;
        const double2 ab = abn, lw = lwn;
        if (bt + 1 < bt1) {
            prn = (const double2 *)(S.prec + 4 * (int64_t)walk.position(bt + 1, lane, vn));
            abn = prn[0];
            lwn = prn[1];
        }
        double pa0 = ab.x, pb0 = ab.y, pl0 = lw.x;
        double pw0 = WEIGHTED ? lw.y : 1.0;
        // two shapes per iteration, the record after them loaded ahead (scalar
        // loads while the current pairs are evaluated)
        double qa = shp[0], qb = shp[1], ql = shp[2], qax = shp[3], qay = shp[4], qew = shp[5],
               qw = shp[6], q2ew = shp[7];
        int j = 0;
        // byte offsets of the records: 32-bit scalars added to the block's
        // base address by the scalar loads themselves
        const uint32_t olast = (uint32_t)(ns - 1) * 64u;
        uint32_t o = 0;
        for (; j + 1 < ns; j += 2, o += 128u) {
            ShapePtr r1 = (ShapePtr)((const MIA_CONST char *)shp + (o + 64u));
            const double b0 = r1[0], b1 = r1[1], b2 = r1[2], b3 = r1[3], b4 = r1[4], b5 = r1[5],
                         b6 = r1[6], b7 = r1[7];
            one_pair<MODE, SH, WEIGHTED, VAR, APART, LZ>(P, S, v0, pa0, pb0, pl0, pw0, qa, qb, ql, qax, qay, qew, qw,
                                         q2ew, sha, shb, shl, hist, row, T, X, nre, pd, vlgc, vlg2, vxs, vxc);
            ShapePtr r2 = (ShapePtr)((const MIA_CONST char *)shp + (o + 128u < olast ? o + 128u : olast));
            const double c0 = r2[0], c1 = r2[1], c2 = r2[2], c3 = r2[3], c4 = r2[4], c5 = r2[5],
                         c6 = r2[6], c7 = r2[7];
            one_pair<MODE, SH, WEIGHTED, VAR, APART, LZ>(P, S, v0, pa0, pb0, pl0, pw0, b0, b1, b2, b3, b4, b5, b6,
                                         b7, sha, shb, shl, hist, row, T, X, nre, pd, vlgc, vlg2, vxs, vxc);
            qa = c0;
            qb = c1;
            ql = c2;
            qax = c3;
            qay = c4;
            qew = c5;
            qw = c6;
            q2ew = c7;
        }
        if (j < ns)
            one_pair<MODE, SH, WEIGHTED, VAR, APART, LZ>(P, S, v0, pa0, pb0, pl0, pw0, qa, qb, ql, qax, qay, qew, qw,
                                         q2ew, sha, shb, shl, hist, row, T, X, nre, pd, vlgc, vlg2, vxs, vxc);
    }
    hist_add<WEIGHTED, VAR, APART>(hist, pd);
}

// The batches [bt0, bt1) of an item, in the pair loop for its periodic-shift variant.
template <int MODE, bool WEIGHTED, bool VAR, bool APART, bool LZ>
__device__ __forceinline__ void run_shifted(const PairArgs &P, const SampleView &S, int cpb, int cn, int bt0, int bt1,
                                            int shifts, ShapePtr shp, int ns, uint32_t hist, const double *T,
                                            const double *X, int lane, uint32_t &nre, uint64_t &iterations) {
    if (shifts & 64)
        run_item<MODE, SH_WRAP, WEIGHTED, VAR, APART, LZ>(P, S, cpb, cn, bt0, bt1, shifts, shp, ns, hist, T, X, lane, nre,
                                                   iterations);
    else if (shifts & 63)
        run_item<MODE, SH_CONST, WEIGHTED, VAR, APART, LZ>(P, S, cpb, cn, bt0, bt1, shifts, shp, ns, hist, T, X, lane, nre,
                                                    iterations);
    else
        run_item<MODE, SH_NONE, WEIGHTED, VAR, APART, LZ>(P, S, cpb, cn, bt0, bt1, shifts, shp, ns, hist, T, X, lane, nre,
                                                   iterations);
}

// Persistent groups of waves over the cost-balanced batches of the key-sorted
// items (a share may begin and end inside an item, so its length does not hang on
// the largest item: 20,000 weighted clustered galaxies and 5,000 shapes in a box
// of 75, 1,500 items for 6,144 waves, 0.83 ms of pair kernel with whole items, now
// 0.13).  A group works on the items of one key at a time and adds into its
// histogram, which goes to the key's sums when the key changes.  A group is one
// wave; or, where private histograms would leave too few waves per CU (P.shared),
// the four waves of a workgroup, which claim the items of a key from a counter in
// LDS and share P.copies copies of one histogram, a lane adding into the copy of
// its place (so neighbouring lanes, which often hit one bin, hit different
// addresses).  With few items per group a claim is a quarter of an item's batches;
// with many whole items even the waves out, and the empty claims of small items
// cost more (a batch of samples with 91 items per group, 1.5 against 2.1 ms;
// 2,000,000 multipoles 196 against 204).
template <int MODE, bool WEIGHTED, bool VAR, bool APART>
__global__ __launch_bounds__(kThreads, kPairWavesPerSimd) void k_pairs(PairArgs P) {
    extern __shared__ __align__(16) char lds[];
    __shared__ unsigned s_next[2];
    __shared__ int s_chunk, s_left;
    __shared__ unsigned long long s_stat[3];
    const int lane = threadIdx.x & (kWave - 1);
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const bool shared = P.shared != 0;
    // exact thresholds for the rare FP64 bin path
    double *T = (double *)lds;
    double *X = T + (P.n_r + 1);
    int nx = P.n_2 + 1;
    for (int i = threadIdx.x; i < P.n_r + 1; i += blockDim.x) T[i] = P.T[i];
    for (int i = threadIdx.x; i < nx; i += blockDim.x) X[i] = P.X[i];
    size_t thr_bytes = ((size_t)(P.n_r + 1 + nx) * 8 + 15) & ~(size_t)15;
    char *hist0 = lds + thr_bytes;
    const int nhist = shared ? P.copies : (int)(blockDim.x / kWave);
    for (int i = threadIdx.x * 4; i < nhist * P.hist_stride; i += blockDim.x * 4) *(uint32_t *)(hist0 + i) = 0u;
    if (threadIdx.x < 2) {
        s_next[threadIdx.x] = 0;
        s_stat[threadIdx.x] = 0;
    }
    if (threadIdx.x == 0) {
        s_left = blockDim.x / kWave;
        s_stat[2] = wall_clock64();
    }
    __syncthreads();

    // runs of neighbouring items of the key-sorted list (which read the same
    // position cells) stay on one XCD
    const int wpb = blockDim.x / kWave, wg = xcd_run_block();
    const int64_t n_items = *(const MIA_CONST int64_t *)P.n_items;
    const int wave = wg * wpb + wv;
    // a plan that overflowed its capacities is counted again by the host
    if (n_items == 0 || *(const MIA_CONST unsigned long long *)P.overflow) return;
    const int tid = shared ? threadIdx.x : lane, nthr = shared ? blockDim.x : kWave;
    char *hist = hist0 + (shared ? 0 : wv * P.hist_stride);
    const int place = ((lane & 7) << 3) | (lane >> 3);
    const uint32_t hist_at = (uint32_t)(uintptr_t)(MIA_LDS char *)(hist + (shared ? place % P.copies : 0) * P.hist_stride) +
                             front_bytes<WEIGHTED, VAR, APART>(P.nbins) - (Slot<WEIGHTED, VAR, APART>::kApart ? 4 : 0);
    // a contiguous share of the cost, then tail chunks from the counter
    const WaveSchedule sch = make_schedule(P.bounds, shared ? (int)gridDim.x : P.n_waves);
    int64_t it0, it1;  // item << kBatchBits | batch
    sch.first(shared ? wg : (wave < P.n_waves ? wave : 0), it0, it1);
    const bool idle = wave >= P.n_waves;
    const bool split = n_items < (int64_t)kSplitItems * gridDim.x;  // (shared)
    if (!shared && idle) it1 = it0;
    it0 = uniform64(it0);
    it1 = uniform64(it1);
    int cur_key = -1, flushes = 0, par = 0;
    uint32_t nre = 0;
    uint64_t iterations = 0;  // wave-uniform
    uint32_t spills = 0;

    auto sync = [&]() {
        if (shared)
            __syncthreads();
        else
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    };
    // The arguments that only the code around the pair loop needs, read again
    // where they are needed: held in scalar registers across the pair loop they
    // push its own out into vector lanes
    auto args = [] {
        const MIA_CONST PairArgs *q = (const MIA_CONST PairArgs *)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(q));
        return q;
    };
    // the histogram goes to its key's sums, the next adds are for `key` (every
    // thread of the group, with no adds in flight)
    auto turn_to = [&](int key) {
        if (cur_key >= 0) {
            sync();
            const PairArgs &P = *(const PairArgs *)args();
            const int kk = P.K1 * P.K1;
            const int sample = cur_key / kk, in = cur_key - sample * kk;
            const int rs = in / P.K1, rp = in - rs * P.K1;
            const int n = shared ? P.copies : 1;
            if (P.det)
                flush_slot<WEIGHTED, VAR, APART>(P, hist, n, P.slot0[wave] + flushes++, slot_key_of(sample, rs, rp), tid, nthr);
            else
                flush_hist<WEIGHTED, VAR, APART>(P, hist, n, P.samples[sample], rs, rp, tid, nthr);
            sync();
        }
        cur_key = key;
    };

    while (true) {
        it0 = uniform64(it0);
        it1 = uniform64(it1);
        const int i0 = (int)(it0 >> kBatchBits), i1 = (int)(it1 >> kBatchBits);
        const int b0 = (int)(it0 & ((1 << kBatchBits) - 1)), b1 = (int)(it1 & ((1 << kBatchBits) - 1));
        const int end = it1 > it0 ? i1 + (b1 > 0 ? 1 : 0) : i0;
        for (int it = i0; it < end;) {
            // the items [it, se) of one key
            const MIA_CONST PairArgs *Q = args();
            const int key = __builtin_amdgcn_readfirstlane(((const MIA_CONST int32_t *)Q->items)[8 * (int64_t)it + 7]);
            const int ke = (int)((const MIA_CONST int64_t *)Q->key_off)[key + 1];
            const int se = __builtin_amdgcn_readfirstlane(ke < end ? ke : end);
            if (key != cur_key) turn_to(key);
            for (int j = it;; ++j) {
                // shared: an item is one claim, or four, its quarters (all of it and
                // three empty ones where it is a single batch)
                int quarter = 0;
                if (shared) {
                    if (idle) break;
                    unsigned t = 0;
                    if (lane == 0) t = atomicAdd(&s_next[par], 1u);
                    t = __builtin_amdgcn_readfirstlane(t);
                    j = it + (int)(split ? t >> 2 : t);
                    quarter = split ? t & 3 : 0;
                }
                // (the compiler does not see that the item is wave-uniform; vector
                // loads of the shape records would cost 70 registers)
                const int i = __builtin_amdgcn_readfirstlane(j);
                if (i >= se) break;
                const MIA_CONST PairArgs *Q = args();
                const MIA_CONST int32_t *ip = (const MIA_CONST int32_t *)Q->items + 8 * (int64_t)i;
                int bt0 = i == i0 ? b0 : 0;
                int bt1 = i == i1 ? b1 : (ip[6] + kWave - 1) / kWave;
                if (shared) {
                    const int n = bt1 - bt0;
                    if (split && n > 1) {
                        bt1 = bt0 + (n * (quarter + 1) >> 2);
                        bt0 += n * quarter >> 2;
                    } else if (quarter) {
                        continue;
                    }
                }
                bt0 = __builtin_amdgcn_readfirstlane(bt0);
                bt1 = __builtin_amdgcn_readfirstlane(bt1);
                if (bt0 >= bt1) continue;  // (no batch: no column of the item is in reach)
                const int blk = ip[0], w = ip[1], jj = ip[2], wn = ip[3], c0 = ip[4], kk = ip[5];
                const int shifts = (w >> 16) & 0xff;
                const MIA_CONST int32_t *bp = (const MIA_CONST int32_t *)Q->blocks + 4 * (int64_t)blk;
                const int s0 = bp[0], ns = bp[1], sample = bp[2];
                const SampleView S = load_view(Q->samples + sample);
                ShapePtr shp = (ShapePtr)(S.srec + 8 * (int64_t)s0);
                int cpb, cn;
                {
                    const MIA_CONST double *bc = (const MIA_CONST double *)Q->bbox + 6 * (int64_t)blk;
                    const double bb[6] = {bc[0], bc[1], bc[2], bc[3], bc[4], bc[5]};
                    item_column(column_view((const MIA_CONST PlanSample *)Q->ps + sample), bb, jj & 0xffff,
                                (jj >> 16) & 0xffff, wn & 0xffff, (wn >> 16) & 0xffff, c0, kk & 0xffff,
                                (kk >> 16) & 0xffff, w, lane, cpb, cn);
                }
                for (int b = bt0; b < bt1; b += kRunBatches) {
                    const int e = bt1 - b < kRunBatches ? bt1 : b + kRunBatches;
                    // (r, mu) sums r^2 in an order fixed by the line of sight: one
                    // loop per order, so the pair loop holds no branch on it
                    if (MODE == MIA_RMU && S.los != 2)
                        run_shifted<MODE, WEIGHTED, VAR, APART, false>(P, S, cpb, cn, b, e, shifts, shp, ns, hist_at, T, X,
                                                                lane, nre, iterations);
                    else
                        run_shifted<MODE, WEIGHTED, VAR, APART, true>(P, S, cpb, cn, b, e, shifts, shp, ns, hist_at, T, X,
                                                               lane, nre, iterations);
                    if ((uint32_t)(iterations >> kSpillBits) == spills) continue;
                    spills = (uint32_t)(iterations >> kSpillBits);
                    const PairArgs &A = *(const PairArgs *)args();
                    const int kk = A.K1 * A.K1, in = cur_key % kk;
                    spill_counts<WEIGHTED, VAR, APART>(A, hist, shared ? A.copies : 1, A.samples[cur_key / kk], in / A.K1,
                                                in % A.K1, lane);
                }
            }
            if (shared) {
                __syncthreads();
                // (the other counter serves the next key, and a barrier lies
                // between this reset and this counter's next use)
                if (threadIdx.x == 0) s_next[par] = 0;
                par ^= 1;
            }
            it = se;
        }
        if (!shared) {
            if (idle || !sch.next(args()->queue, lane, it0, it1)) break;
        } else {
            if (sch.tail == 0) break;
            if (threadIdx.x == 0) s_chunk = atomicAdd(args()->queue, 1);
            __syncthreads();
            const int k = __builtin_amdgcn_readfirstlane(s_chunk);
            __syncthreads();
            if (!sch.chunk(k, it0, it1)) break;
        }
    }
    turn_to(-1);
    // Statistics: the last wave of the workgroup adds them, to one of
    // kStatCopies copies a cache line apart (four atomics of every wave on one
    // line took 0.1 ms of a count of 2,000 galaxies).
    if (nre) atomicAdd(&s_stat[0], (unsigned long long)nre);
    if (lane == 0) {
        if (iterations) atomicAdd(&s_stat[1], (unsigned long long)iterations);
        if (__hip_atomic_fetch_add(&s_left, -1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP) == 1 && s_stat[1]) {
            unsigned long long *st = args()->stat + (wg % kStatCopies) * kStatStride;
            atomicAdd(&st[0], s_stat[0]);
            atomicAdd(&st[1], s_stat[1]);
            atomicMax(&st[2], ~s_stat[2]);
            atomicMax(&st[3], (unsigned long long)wall_clock64());
        }
    }
}

template <int MODE, bool WEIGHTED, bool VAR, bool APART>
void launch_pairs(const PairArgs &A, unsigned grid, int wpb, size_t lds, hipStream_t st) {
    hipLaunchKernelGGL((k_pairs<MODE, WEIGHTED, VAR, APART>), dim3(grid), dim3(kWave * wpb), lds, st, A);
    MIA_HIP(hipGetLastError());
}

template <int MODE>
void launch_pairs_mode(const PairArgs &A, unsigned grid, int wpb, size_t lds, hipStream_t st) {
    if (A.weighted && A.var)
        A.apart ? launch_pairs<MODE, true, true, true>(A, grid, wpb, lds, st)
                : launch_pairs<MODE, true, true, false>(A, grid, wpb, lds, st);
    else if (A.weighted)
        launch_pairs<MODE, true, false, true>(A, grid, wpb, lds, st);
    else if (A.var)
        launch_pairs<MODE, false, true, true>(A, grid, wpb, lds, st);
    else
        A.apart ? launch_pairs<MODE, false, false, true>(A, grid, wpb, lds, st)
                : launch_pairs<MODE, false, false, false>(A, grid, wpb, lds, st);
}

// LDS bytes of the thresholds of a workgroup.
size_t threshold_bytes(const mia_bins &bins) {
    return ((size_t)(bins.n_r + 1 + bins.n_2 + 1) * 8 + 15) & ~(size_t)15;
}

inline unsigned nblk(int64_t n, int t) { return (unsigned)((n + t - 1) / t < 1 ? 1 : (n + t - 1) / t); }

// Pair-kernel configuration of a binning: FP32 guess constants and guard
// bands, passes over r-bin ranges, histogram copies and offsets, waves.
struct PairConfig {
    PairArgs A{};        // pointers unset
    int nrp = 0, npass = 0, wpb = 0, waves = 0, groups = 0;
    unsigned grid = 0;
    size_t lds = 0;
    double l0 = 0, lgs = 0, shift_r = 0;
};

// The pair kernel of a count.
template <int M>
const void *pair_kernel(bool weighted, bool var, bool apart) {
    if (weighted != var)
        return weighted ? (const void *)k_pairs<M, true, false, true> : (const void *)k_pairs<M, false, true, true>;
    if (apart)
        return weighted ? (const void *)k_pairs<M, true, true, true> : (const void *)k_pairs<M, false, false, true>;
    return weighted ? (const void *)k_pairs<M, true, true, false> : (const void *)k_pairs<M, false, false, false>;
}
const void *pair_kernel(int mode, bool weighted, bool var, bool apart) {
    return mode == MIA_RPPI ? pair_kernel<MIA_RPPI>(weighted, var, apart) : pair_kernel<MIA_RMU>(weighted, var, apart);
}

// Workgroups of that kernel a CU holds at once (registers and LDS).
int resident_workgroups(const PairArgs &A, int wpb, size_t lds) {
    int n = 0;
    MIA_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, pair_kernel(A.mode, A.weighted, A.var, A.apart),
                                                         kWave * wpb, lds));
    return std::max(1, std::min(n, workgroups_by_lds(lds + kPairStaticLds)));
}

// Waves per CU whose histograms (hs bytes) and thresholds LDS holds, with a
// histogram per wave (workgroups of 4, 2 or 1 waves) or per workgroup of 4.
int private_waves(size_t thr_bytes, size_t hs) {
    int w = kMaxWavesPerBlock;
    while (w > 1 && thr_bytes + hs * w + kPairStaticLds > kLdsBytes) w /= 2;
    return std::min(32 / w, workgroups_by_lds(thr_bytes + hs * w + kPairStaticLds)) * w;
}
int shared_waves(size_t thr_bytes, size_t hs) {
    return std::min(32 / kMaxWavesPerBlock, workgroups_by_lds(thr_bytes + hs + kPairStaticLds)) * kMaxWavesPerBlock;
}

// candidates: expected (shape, position) pairs of the count.
PairConfig pair_config(const mia_bins &bins, bool any_w, bool any_var, const mia_tuning *tuning, int cu_count,
                       double candidates) {
    PairConfig C;
    PairArgs &A = C.A;
    const bool det = tuning && tuning->deterministic != 0;
    const int n_r = bins.n_r, n_2 = bins.n_2, B = n_r * n_2;
    A.mode = bins.mode;
    A.n_r = n_r;
    A.n_2 = n_2;
    A.weighted = any_w ? 1 : 0;
    A.var = any_var ? 1 : 0;
    A.nbins = B;
    // FP32 bin guesses and their guard bands (bin units).  The guess error
    // is bounded by a few FP32 ulps of the log2 / linear transform (the
    // bounds below, with a 20x margin); the exact FP64 count runs only for
    // guesses within the band of an edge.
    A.T0 = bins.r2_edges[0];
    A.Tn = bins.r2_edges[n_r];
    double l0 = std::log2(bins.r2_edges[0]), ln = std::log2(bins.r2_edges[n_r]);
    double lgs = n_r / (ln - l0);
    C.l0 = l0;
    C.lgs = lgs;
    A.lgs = (float)lgs;
    const double u = std::ldexp(1.0, -23);  // FP32 ulp of 1
    // (+ 2u n_r for a pass's shifted constant -l0 lgs - r0)
    double err_r = (4 * u * std::fmax(std::fabs(l0), std::fabs(ln)) + 4 * u) * lgs + 4 * u * n_r;
    double err_2;
    double d2;
    if (bins.mode == MIA_RPPI) {
        A.X0 = bins.x2_edges[0];
        A.Xn = bins.x2_edges[n_2];
        // FP64 guess fma(pi, xs, xc): a few FP64 ulps of |pi| xs + n_2 bins,
        // far inside the 1e-9-bin guard band
        const double xs = n_2 / (bins.x2_edges[n_2] - bins.x2_edges[0]);
        A.xs64 = xs;
        A.xc64 = -bins.x2_edges[0] * xs;
        const double mx = std::fmax(std::fabs(bins.x2_edges[0]), std::fabs(bins.x2_edges[n_2]));
        const double e64 = std::ldexp(1.0, -52);
        err_2 = 8 * e64 * (mx * xs + n_2);
        d2 = std::fmax(1e-9, 20 * err_2);
    } else {
        A.X0 = 0;
        A.Xn = 0;
        A.xs = (float)(n_2 / 2.0);
        err_2 = 6 * u * n_2;
        d2 = std::fmax(1e-4, 20 * err_2);
    }
    double dr = std::fmax(1e-4, 20 * err_r);
    // pathological binnings (guard band > 5% of a bin): every pair takes the exact path
    bool exact_only = dr > 0.05 || d2 > 0.05;
    // the guesses are raised by the half width d, and an edge within d of one
    // then leaves it a fraction below 2 d
    A.dr = exact_only ? 2.0f : (float)(2.0 * dr);
    A.d2 = exact_only ? 2.0 : 2.0 * d2;
    A.d2f = (float)A.d2;
    C.shift_r = exact_only ? 0.0 : dr;
    const double shift_2 = exact_only ? 0.0 : d2;
    A.xc64 += shift_2;
    A.xc = (float)shift_2;
    A.scan = exact_only ? 1 : 0;
    // Passes over r-bin ranges.  Pass [r0, r0 + nrp) takes the pairs with
    // T[r0] <= r^2 < T[r0 + nrp] (exact FP64 comparisons, so every pair lands
    // in one pass), bins them locally and flushes to output bins
    // r0 * n_2 + local.  A pass's time goes about as 1 / min(1, w / W), w the
    // waves per CU its histogram leaves room for, so nrp minimises
    // passes / min(1, w / W) (ties: fewer passes), with at least 4 waves per
    // CU where any split allows it (at 2 a pass runs slower than that model
    // says).  W is 7 with histograms per wave (deterministic) and 10 with
    // histograms per workgroup, whose waves wait for each other.  Pair kernels
    // with W = 16 and now, 1,000,000 positions and 200,000 shapes: deterministic
    // 100 x 100 bins 25 passes of 16 waves 181 ms, 7 of 4 121; 60 x 60 8 of 12 70 ms,
    // 5 of 8 54 (counts inside the bins); shared, 200,000 and 50,000: 100 x 100 5 of 12 6.1 ms, 2 of 4
    // 4.1.  Ordinary binnings run in one pass.
    const size_t thr_bytes = threshold_bytes(bins);
    int nrp = n_r;
    {
        auto waves_per_cu = [&](int c, bool apart) {
            const size_t hs = hist_bytes(c * n_2, any_w, any_var, apart);
            const int w = private_waves(thr_bytes, hs);
            return det ? w : std::max(w, shared_waves(thr_bytes, hs));
        };
        // rows of the cheapest pass and its price
        auto best_pass = [&](bool apart, double &best) {
            int best_c = 1, best_p = 0;
            best = 1e300;
            for (int pass_min_waves : {4, 1}) {
                for (int c = n_r; c >= 1; --c) {
                    const int w = waves_per_cu(c, apart);
                    if (w < pass_min_waves) continue;
                    const int passes = (n_r + c - 1) / c;
                    const double cost = (double)passes / std::min(1.0, w / (det ? 7.0 : 10.0));
                    if (cost < best * (1 - 1e-9) || (cost <= best * (1 + 1e-9) && passes < best_p)) {
                        best = cost;
                        best_p = passes;
                        best_c = c;
                    }
                }
                if (best_p) break;
            }
            return best_c;
        };
        // Two or four sums have their counts apart only in the deterministic mode,
        // where narrower bins save passes or leave more private waves; elsewhere
        // the lanes' bins collide more on the banks (200 bins, 1,000,000 positions
        // 7.7 -> 8.3 ms of pair kernel).  Deterministic, 1,000,000 positions and
        // 200,000 shapes, inside / apart: 60 x 60 bins 56.5 / 44.0 ms, 100 x 100
        // 127 / 92; 300,000 and 60,000: 100 x 20 4.4 / 3.2, with weights and variances
        // 33 x 101 10.0 / 8.0, 80 x 80 16.3 / 15.2, but 120 x 120, 0.93 of the price,
        // 32.0 / 32.4.
        double cost = 1e300, cost_apart;
        const int c_apart = best_pass(true, cost_apart);
        if (any_w == any_var) nrp = best_pass(false, cost);
        A.apart = any_w != any_var || (det && cost_apart < 0.92 * cost);
        if (A.apart) nrp = c_apart;
        if (tuning && tuning->r_bins_per_pass > 0) {
            // as asked, but no more than one wave's histogram can hold
            nrp = std::min(n_r, tuning->r_bins_per_pass);
            while (nrp > 1 && waves_per_cu(nrp, A.apart) == 0) --nrp;
        }
    }
    C.nrp = nrp;
    C.npass = (n_r + nrp - 1) / nrp;
    const int Bp = nrp * n_2;     // bins of the largest pass
    A.nbins_out = B;
    A.bin_off = 0;
    A.hist_stride = (int)hist_bytes(Bp, any_w, any_var, A.apart);
    // A private histogram per wave (one copy: the pending-slot registers already
    // absorb most same-address collisions), or one per workgroup, shared by its
    // four waves, in as many copies (at most 4) as leave room for
    // kPairWavesPerSimd waves per SIMD.  Sharing keeps the SIMDs full where
    // private histograms leave LDS for few waves, and a key's histogram is flushed
    // once for four waves; but a group of four waits for its slowest wave wherever
    // the key or the chunk changes.  Shared / private, pair kernel in ms:
    //   - below kSharedBelow private waves per CU shared: 600 bins, 3,000,000
    //     positions to 100 Mpc/h 188 / 306 (8 waves); 1600 bins, 43,140 weightless
    //     positions 1.3 / 2.3 (4 waves);
    //   - the smallest launches shared, where the flushes weigh most: 20,000 with 27
    //     regions 0.096 / 0.175, 20,000 in 100,000 0.21 / 0.26, 30,000 in 150,000 0.41
    //     / 0.45 (2,000 galaxies equal); from 24,000 in 120,000 (0.285 / 0.26) on
    //     private: 40,000 in 200,000 0.61 / 0.57, 60,000 in 300,000 1.43 /
    //     1.14, 200,000 in 1,000,000 10.4 / 7.6, a batch of eight uneven samples
    //     3.7 / 2.7;
    //   - with weights and variances, whose bins leave 16 private waves for 200 bins,
    //     shared up to eight times as many: 40,000 in 200,000 0.71 / 0.87, 75,025 in
    //     317,811 1.89 / 2.08, but 80,000 in 400,000 2.44 / 2.21;
    //   - where registers allow more waves than LDS and the launch is so large
    //     that its chunks hold many items shared: 2,000,000 multipoles, 300 bins
    //     195 / 202.
    // Never where the reduction is deterministic, since a shared histogram's sums
    // depend on timing.  mia_tuning.hist_copies is ignored.
    int wpb = kMaxWavesPerBlock;
    const size_t hs = A.hist_stride;
    const int pw = private_waves(thr_bytes, hs), most = std::min(4 * kPairWavesPerSimd, shared_waves(thr_bytes, hs));
    const bool small = candidates < (any_w && any_var ? 0.65 : 0.08) * kTailMinCost * pw * cu_count;
    const bool large = candidates > 16 * kTailMinCost * pw * cu_count;
    A.shared = !det && most > 0 && (small || (pw < most && (pw < kSharedBelow || large)));
    if (A.shared) {
        const size_t share = kLdsBytes / kPairWavesPerSimd / kLdsGranule * kLdsGranule - kPairStaticLds;
        A.copies = share > thr_bytes + hs ? (int)std::min<size_t>(4, (share - thr_bytes) / hs) : 1;
        C.lds = thr_bytes + hs * A.copies;
    } else {
        while (wpb > 1 && thr_bytes + hs * wpb + kPairStaticLds > kLdsBytes) wpb /= 2;
        A.copies = 1;
        C.lds = thr_bytes + hs * wpb;
    }
    if (C.lds + kPairStaticLds > kLdsBytes)
        throw Error{MIA_E_UNSUPPORTED, "histogram too large for LDS (n_r*n_2 too big for MIA_FAST)"};
    C.wpb = wpb;
    // as many workgroups as are resident at once
    const int blocks_per_cu = resident_workgroups(A, wpb, C.lds);
    int waves = tuning && tuning->waves > 0 ? std::min(tuning->waves, kMaxWaves) : cu_count * blocks_per_cu * wpb;
    C.waves = std::max(1, waves);
    A.n_waves = C.waves;
    C.grid = (unsigned)((C.waves + wpb - 1) / wpb);
    C.groups = A.shared ? (int)C.grid : C.waves;
    return C;
}

}  // namespace

bool fast_path_fits(const mia_bins &bins, bool weighted, int jk) {
    const int64_t K1 = jk > 0 ? (int64_t)jk * jk * jk : 1;
    if (K1 * K1 > kMaxKeysPerSample) return false;
    // larger binnings run in passes over r-bin ranges: one r row must fit
    return threshold_bytes(bins) + hist_bytes(bins.n_2, weighted, bins.accumulate_variance, true) + kPairStaticLds <=
           kLdsBytes;
}

// Sets the dynamic-LDS limit of every pair-kernel variant (once per process).
void pair_kernels_init() {
    static std::mutex mu;
    static uint64_t done = 0;  // one bit per device
    int dev = 0;
    MIA_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(mu);
    if (dev < 64 && (done >> dev & 1)) return;
    for (int i = 0; i < 16; ++i)
        MIA_HIP(hipFuncSetAttribute(pair_kernel(i & 4 ? MIA_RMU : MIA_RPPI, i & 2, i & 1, i & 8),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)(kLdsBytes - kPairStaticLds)));
    if (dev < 64) done |= 1ull << dev;
}

// ---------------------------------------------------------------------------
// staged count: host plan, workspace binding, launch sequence

struct CountPlan {
    int S = 0;
    int K1 = 1, kseg = 0, bsz = kMaxBlockShapes;
    int64_t ncells = 0, nblk_cap = 0, nkeys = 0, fin_total = 0, item_cap = 0;
    int64_t acc_total = 0;           // accumulator words (u64 / f64) of all samples
    double margin = 0;               // largest geometric slack of the samples' grids
    PairConfig pc;
    bool any_w = false, any_var = false;
    bool det = false;                // deterministic reduction (slots instead of atomics)
    int64_t slot_cap = 0;            // slots: at most waves + planner keys
    std::vector<double> T, X;        // thresholds (X padded to n_2 + 1)
    std::vector<PlanSample> ps;
    std::vector<SampleDev> sd;
    std::vector<FinSample> fs;
    std::vector<int64_t> cell0, fin0;
    std::vector<int64_t> acc0;       // first accumulator word of each sample
    std::vector<int> Bs;             // per sample: K
    // bound workspace
    char *param_dev = nullptr;
    std::vector<char> param;         // host image of the parameter block
    size_t off_T = 0, off_X = 0, off_cell0 = 0, off_fin0 = 0, off_ps = 0, off_sd = 0, off_fs = 0;
    size_t param_bytes = 0;
    unsigned long long *zero_begin = nullptr;
    size_t zero_words = 0;
    int32_t *nb = nullptr, *boff = nullptr;
    Block *blocks = nullptr;
    unsigned long long *kc = nullptr, *kcur = nullptr;
    int64_t *ko = nullptr;
    Item *items = nullptr;
    int64_t *cost = nullptr, *cpre = nullptr, *n_items = nullptr, *bounds = nullptr;
    double *bbox = nullptr;
    uint32_t *geo = nullptr;
    unsigned long long *words = nullptr;   // [kCountReadback] read back after the count
    unsigned long long *stat = nullptr;    // the pair kernel's statistics, kStatCopies copies
    int *queue = nullptr;
    unsigned long long *acc = nullptr;
    int64_t *heads = nullptr, *n_heads = nullptr;
    int64_t *runs = nullptr, *slot0 = nullptr, *slot_key = nullptr, *ne = nullptr, *ne_pre = nullptr;
    unsigned long long *skey = nullptr, *skey2 = nullptr;   // deterministic item order
    int32_t *sidx = nullptr, *sidx2 = nullptr;
    Item *items2 = nullptr;
    int64_t *cost2 = nullptr;
    void *stmp = nullptr;
    size_t stmp_bytes = 0;
    unsigned long long *slot_np = nullptr;
    double *slot_sp = nullptr, *slot_sx = nullptr, *slot_dd = nullptr, *slot_var = nullptr;
    ScanBufs<int32_t> scan_nb;
    ScanBufs<int64_t> scan_keys, scan_cost, scan_runs, scan_ne;
    std::vector<int> G;
    std::string key;
};

int count_waves(const CountPlan &p) { return p.pc.waves; }
int count_bsz(const CountPlan &p) { return p.bsz; }
bool count_det(const CountPlan &p) { return p.det; }
int count_G(const CountPlan &p, int s) { return p.G[s]; }
int64_t count_item_cap(const CountPlan &p) { return p.item_cap; }
std::string count_key(const CountPlan &p) { return p.key; }
size_t count_param_bytes(const CountPlan &p) { return p.param_bytes; }
const void *count_param_image(const CountPlan &p) { return p.param.data(); }
void *count_param_dev(const CountPlan &p) { return p.param_dev; }
const unsigned long long *count_readback(const CountPlan &p) { return p.words; }
void free_plan(CountPlan *p) { delete p; }

// Expected work items of a sample (mia_grid.hip's uniform-density model).
double estimate_items(const Grid &g, int G, int cpi, double reach_r, double reach_z, bool rmu, int64_t ns, int64_t np,
                      int64_t blk_cap);

// Deterministic item sort key: planner key, then block and rectangle (the low
// det_low_bits bits).
int det_low_bits(const CountPlan &p) {
    const int64_t n = p.nblk_cap * (kMaxSegs * kMaxSegs * (kMaxSegs + 1));
    int b = 1;
    while (b < 62 && ((int64_t)1 << b) < n) ++b;
    return b;
}
int det_index_bits(const CountPlan &p) {
    int b = 1;
    while (b < 31 && ((int64_t)1 << b) < p.nkeys + 1) ++b;
    return b;
}
// A key and a block's rectangle that do not fit one word take two stable sorts,
// by rectangle and then by key (50,000,000 shape blocks with 4,096 regions).
bool det_two_sorts(const CountPlan &p) { return det_low_bits(p) + det_index_bits(p) > 64; }
int det_key_bits(const CountPlan &p) {
    return det_two_sorts(p) ? std::max(det_low_bits(p), det_index_bits(p)) : det_low_bits(p) + det_index_bits(p);
}

CountPlan *plan_count(Ctx &ctx, const std::vector<SortedSample> &ss, const mia_bins &bins,
                      const mia_tuning *tuning, int64_t item_cap, bool cap_exact) {
    pair_kernels_init();
    std::unique_ptr<CountPlan> P(new CountPlan());
    CountPlan &p = *P;
    const int S = (int)ss.size();
    MIA_REQUIRE(S >= 1, "no samples");
    p.S = S;
    const int n_r = bins.n_r, n_2 = bins.n_2, B = n_r * n_2;
    MIA_REQUIRE(n_r >= 1 && n_r <= kMaxBinsR && n_2 >= 1 && n_2 <= kMaxBins2, "bin counts out of range");
    const double reach_r = std::sqrt(bins.r2_edges[n_r]);
    const double reach_z = bins.mode == MIA_RPPI
                               ? std::fmax(std::fabs(bins.x2_edges[0]), std::fabs(bins.x2_edges[n_2]))
                               : reach_r;
    const int nx2 = bins.mode == MIA_RPPI ? n_2 + 1 : n_2;
    p.T.assign(bins.r2_edges, bins.r2_edges + n_r + 1);
    p.X.assign(n_2 + 1, 3.0);
    for (int i = 0; i < nx2; ++i) p.X[i] = bins.x2_edges[i];
    p.bsz = tuning && tuning->block_shapes > 0 ? std::min(tuning->block_shapes, kMaxBlockShapes) : kMaxBlockShapes;
    p.any_var = bins.accumulate_variance != 0;
    for (const auto &x : ss) p.any_w = p.any_w || x.weighted;
    // (shape, position) pairs within reach at the mean densities, half as many
    // again for the blocks' extents
    double candidates = 0;
    for (const auto &x : ss) {
        const double L = x.g.L, pi = 3.14159265358979;
        const double v = bins.mode == MIA_RPPI ? pi * reach_r * reach_r * std::min(L, 2 * reach_z)
                                               : 4.0 / 3.0 * pi * reach_r * reach_r * reach_r;
        candidates += 1.5 * (double)x.n_shape * (double)x.n_pos * std::min(1.0, v / (L * L * L));
    }
    p.pc = pair_config(bins, p.any_w, p.any_var, tuning, ctx.cu_count, candidates);
    p.det = tuning && tuning->deterministic != 0;

    p.ps.resize(S);
    p.sd.resize(S);
    p.fs.resize(S);
    p.G.resize(S);
    p.cell0.assign(S + 1, 0);
    p.fin0.assign(S + 1, 0);
    p.acc0.assign(S + 1, 0);
    double est_items = 0;
    int jk_max = 1;
    for (int si = 0; si < S; ++si) {
        const SortedSample &x = ss[si];
        const Grid &g = x.g;
        p.K1 = std::max(p.K1, x.K > 0 ? x.K : 1);
        // slabs per block: explicit, else the grid's choice, else ~16 shapes
        // per block; always a divisor of the per-jk slab count
        int G = 1;
        if (tuning && tuning->slabs_per_block > 0) {
            G = tuning->slabs_per_block;
        } else if (g.G > 0) {
            G = g.G;
        } else {
            double per_slab = (double)x.n_shape / ((double)g.nc * g.nc * g.nz);
            double want = per_slab > 0 ? 16.0 / per_slab : g.nzj;
            G = (int)std::floor(want);
        }
        G = std::max(1, std::min(G, g.nzj));
        while (g.nzj % G) --G;
        p.G[si] = G;
        PlanSample &Q = p.ps[si];
        std::memset(&Q, 0, sizeof(Q));
        p.margin = std::max(p.margin, g.margin);
        Q.g = g;
        Q.mode = bins.mode;
        Q.periodic = x.periodic;
        Q.ng = g.nz / G;
        Q.G = G;
        Q.ncp = g.nc * g.m;
        Q.pbits = x.pbits;
        Q.fw = g.cw / g.m;
        Q.hq_inv = (double)(1 << x.pbits) / g.hz;
        // columns per item: about kItemPositions positions at the mean density
        // (mia_tuning.item_positions), at most one column per lane
        const double per_col = (double)x.n_pos / ((double)Q.ncp * Q.ncp) *
                               std::min(1.0, 2.0 * reach_z / std::max(g.L, 1e-300));
        const double want_pos = tuning && tuning->item_positions > 0 ? tuning->item_positions : kItemPositions;
        Q.cpi = (int)std::max(1.0, std::min((double)kWave, std::floor(want_pos / std::max(per_col, 1e-9) + 0.5)));
        jk_max = std::max(jk_max, g.jk);
        Q.reach_r = reach_r;
        Q.reach_z = reach_z;
        Q.x_lo = bins.mode == MIA_RPPI ? bins.x2_edges[0] : -reach_r;
        Q.x_hi = bins.mode == MIA_RPPI ? bins.x2_edges[n_2] : reach_r;
        Q.sstart = x.sstart;
        Q.ncells = (int64_t)g.nc * g.nc * (Q.ng + 1);
        Q.cell0 = p.cell0[si];
        p.cell0[si + 1] = Q.cell0 + Q.ncells;
        const int64_t blk_cap = (x.n_shape + p.bsz - 1) / p.bsz + std::min<int64_t>(Q.ncells, x.n_shape);
        p.nblk_cap += blk_cap;
        const int K = x.K;
        p.fin0[si + 1] = p.fin0[si] + (int64_t)(1 + K) * B + K;
        // accumulators: npairs, sp, dd ((1+K) B each), sx, var (B each)
        p.acc0[si + 1] = p.acc0[si] + 3 * (int64_t)(1 + K) * B + 2 * (int64_t)B;
        est_items += estimate_items(g, G, Q.cpi, reach_r, reach_z, bins.mode == MIA_RMU, x.n_shape, x.n_pos, blk_cap);
    }
    p.kseg = std::min(jk_max + kSegExtra, kMaxSegs);
    p.ncells = p.cell0[S];
    p.fin_total = p.fin0[S];
    p.acc_total = p.acc0[S];
    MIA_REQUIRE((double)S * p.K1 * p.K1 < 2e9, "too many planner keys (samples x regions^2)");
    p.nkeys = (int64_t)S * p.K1 * p.K1;
    p.slot_cap = p.det ? (int64_t)p.pc.waves + p.nkeys : 0;
    MIA_REQUIRE(p.nblk_cap < ((int64_t)1 << 31), "too many shape blocks");
    // item capacity: the caller's (grown after an overflow), at least twice
    // the uniform-density estimate plus a margin
    p.item_cap = cap_exact ? item_cap : std::max<int64_t>(item_cap, (int64_t)(2.0 * est_items) + 65536);
    p.item_cap = std::min<int64_t>(p.item_cap, (int64_t)1 << 31);

    // the launch-sequence key: everything the launches depend on except the
    // caller's pointers (which live in the parameter block)
    std::string &k = p.key;
    auto put = [&](const void *v, size_t n) { k.append((const char *)v, n); };
    put(&S, sizeof(S));
    put(&bins.mode, sizeof(int) * 4);
    put(p.T.data(), sizeof(double) * p.T.size());
    put(p.X.data(), sizeof(double) * p.X.size());
    if (tuning) put(tuning, sizeof(*tuning));
    put(&p.item_cap, sizeof(p.item_cap));
    for (int si = 0; si < S; ++si) {
        PlanSample q = p.ps[si];
        q.sstart = q.pfine = q.flags = nullptr;
        q.srec = nullptr;
        put(&q, sizeof(q));
        put(&ss[si].n_pos, sizeof(int64_t));
        put(&ss[si].n_shape, sizeof(int64_t));
        put(&ss[si].K, sizeof(int));
        put(&ss[si].weighted, sizeof(int));
    }
    return P.release();
}

size_t count_bytes(const CountPlan &p) {
    Carve c;
    CountPlan q = p;
    count_bind(q, c, {}, nullptr);
    return c.off;
}

void count_bind(CountPlan &p, Carve &c, const std::vector<SortedSample> &ss, const mia_counts *outs) {
    const int S = p.S;
    const int n_r = p.pc.A.n_r, n_2 = p.pc.A.n_2, B = n_r * n_2;
    const bool dry = c.dry;
    // parameter block
    Carve pc;
    pc.dry = true;
    p.off_T = pc.off; pc.take<double>(n_r + 1);
    p.off_X = pc.off; pc.take<double>(n_2 + 1);
    p.off_cell0 = pc.off; pc.take<int64_t>(S + 1);
    p.off_fin0 = pc.off; pc.take<int64_t>(S + 1);
    p.off_ps = pc.off; pc.take<PlanSample>(S);
    p.off_sd = pc.off; pc.take<SampleDev>(S);
    p.off_fs = pc.off; pc.take<FinSample>(S);
    p.param_bytes = pc.off;
    p.param_dev = c.take<char>(p.param_bytes);
    // zeroed at the start of every count: accumulators, key counters,
    // read-back words, tail-chunk counters (one contiguous range)
    char *z0 = c.dry ? nullptr : c.base + c.off;
    p.acc = c.take<unsigned long long>(p.acc_total);
    p.kc = c.take<unsigned long long>(p.nkeys + 1);
    p.kcur = c.take<unsigned long long>(p.nkeys + 1);
    p.words = c.take<unsigned long long>(kCountReadback);
    p.stat = c.take<unsigned long long>(kStatCopies * kStatStride);
    p.queue = c.take<int>(kMaxBinsR);
    p.zero_begin = (unsigned long long *)z0;
    p.zero_words = dry ? 0 : (size_t)((c.base + c.off) - z0) / 8;
    // plan
    p.nb = c.take<int32_t>(p.ncells + 1);
    p.boff = c.take<int32_t>(p.ncells + 1);
    scan_carve<int32_t>(c, p.ncells, p.scan_nb);
    const int64_t blk_total = std::max<int64_t>(p.nblk_cap, 1);
    p.blocks = c.take<Block>(blk_total);
    p.bbox = c.take<double>(6 * blk_total);
    p.geo = c.take<uint32_t>((3 + 3 * (int64_t)p.kseg) * blk_total);
    p.ko = c.take<int64_t>(p.nkeys + 1);
    scan_carve<int64_t>(c, p.nkeys, p.scan_keys);
    p.items = c.take<Item>(p.item_cap);
    p.cost = c.take<int64_t>(p.item_cap + 1);
    p.cpre = c.take<int64_t>(p.item_cap + 1);
    scan_carve<int64_t>(c, p.item_cap, p.scan_cost);
    p.n_items = c.take<int64_t>(1);
    p.bounds = c.take<int64_t>((size_t)p.pc.groups * kScheduleUnits + 3);
    if (p.det) {
        const int64_t W = p.pc.waves, sw = p.slot_cap * B;
        p.runs = c.take<int64_t>(W + 1);
        p.slot0 = c.take<int64_t>(W + 1);
        scan_carve<int64_t>(c, W, p.scan_runs);
        p.ne = c.take<int64_t>(p.nkeys + 1);
        p.ne_pre = c.take<int64_t>(p.nkeys + 1);
        scan_carve<int64_t>(c, p.nkeys, p.scan_ne);
        p.slot_key = c.take<int64_t>(p.slot_cap);
        p.heads = c.take<int64_t>(p.slot_cap);
        p.n_heads = c.take<int64_t>(1);
        p.slot_np = c.take<unsigned long long>(sw);
        p.slot_sp = c.take<double>(sw);
        p.slot_sx = c.take<double>(sw);
        p.slot_dd = p.any_w ? c.take<double>(sw) : nullptr;
        p.slot_var = p.any_var ? c.take<double>(sw) : nullptr;
        p.skey = c.take<unsigned long long>(p.item_cap);
        p.skey2 = c.take<unsigned long long>(p.item_cap);
        p.sidx = c.take<int32_t>(p.item_cap);
        p.sidx2 = c.take<int32_t>(p.item_cap);
        p.items2 = c.take<Item>(p.item_cap);
        p.cost2 = c.take<int64_t>(p.item_cap + 1);
        size_t bytes = 0;
        MIA_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, (const unsigned long long *)nullptr,
                                                   (unsigned long long *)nullptr, (const int32_t *)nullptr,
                                                   (int32_t *)nullptr, (int)p.item_cap, 0, det_key_bits(p),
                                                   (hipStream_t)0));
        p.stmp_bytes = std::max<size_t>(bytes, 256);
        p.stmp = c.take<char>(p.stmp_bytes);
    }
    if (dry) return;

    // parameter block image
    p.param.assign(p.param_bytes, 0);
    char *img = p.param.data();
    std::memcpy(img + p.off_T, p.T.data(), sizeof(double) * (n_r + 1));
    std::memcpy(img + p.off_X, p.X.data(), sizeof(double) * (n_2 + 1));
    std::memcpy(img + p.off_cell0, p.cell0.data(), sizeof(int64_t) * (S + 1));
    std::memcpy(img + p.off_fin0, p.fin0.data(), sizeof(int64_t) * (S + 1));
    unsigned long long *acc = p.acc;
    double *accd = (double *)p.acc;
    for (int si = 0; si < S; ++si) {
        const SortedSample &x = ss[si];
        const int K = x.K;
        const int64_t nb = (int64_t)(1 + K) * B;
        const int64_t a0 = p.acc0[si];
        PlanSample &Q = p.ps[si];
        Q.sstart = x.sstart;
        Q.pfine = x.pfine;
        Q.flags = x.flags;
        Q.srec = x.srec;
        SampleDev &D = p.sd[si];
        std::memset(&D, 0, sizeof(D));
        D.prec = x.prec;
        D.srec = x.srec;
        D.L = x.g.L;
        D.half = x.g.half;
        D.los = x.g.los;
        D.K = K;
        D.nbins = B;
        D.npairs = acc + a0;
        D.sp = accd + a0 + nb;
        D.dd = x.weighted ? accd + a0 + 2 * nb : nullptr;
        D.sx = accd + a0 + 3 * nb;
        D.var = p.any_var ? accd + a0 + 3 * nb + B : nullptr;
        FinSample &F = p.fs[si];
        std::memset(&F, 0, sizeof(F));
        F.np = acc + a0;
        F.sp = accd + a0 + nb;
        F.dd = accd + a0 + 2 * nb;
        F.sx = accd + a0 + 3 * nb;
        F.var = accd + a0 + 3 * nb + B;
        F.rcnt = x.rcnt;
        F.rsum = x.rsum;
        F.out = outs[si];
        F.K = K;
        F.B = B;
        F.weighted = x.weighted;
        F.var_on = p.any_var ? 1 : 0;
    }
    std::memcpy(img + p.off_ps, p.ps.data(), sizeof(PlanSample) * S);
    std::memcpy(img + p.off_sd, p.sd.data(), sizeof(SampleDev) * S);
    std::memcpy(img + p.off_fs, p.fs.data(), sizeof(FinSample) * S);
}

void count_enqueue(const CountPlan &p, hipStream_t st, const hipEvent_t *ev) {
    const int S = p.S;
    const char *pd = p.param_dev;
    const PlanSample *ps = (const PlanSample *)(pd + p.off_ps);
    const int64_t *cell0 = (const int64_t *)(pd + p.off_cell0);
    const int64_t *fin0 = (const int64_t *)(pd + p.off_fin0);
    if (ev) MIA_HIP(hipEventRecord(ev[0], st));
    fill<unsigned long long>(p.zero_begin, 0ull, (int64_t)p.zero_words, st);
    // shape blocks of every (column, slab group) cell
    hipLaunchKernelGGL(k_blocks, dim3(nblk(p.ncells, 256)), dim3(256), 0, st, ps, cell0, S, p.bsz, p.nb,
                       (const int32_t *)nullptr, (Block *)nullptr);
    MIA_HIP(hipGetLastError());
    scan_ws<int32_t>(p.nb, p.boff, p.ncells, nullptr, p.scan_nb, st);
    hipLaunchKernelGGL(k_blocks, dim3(nblk(p.ncells, 256)), dim3(256), 0, st, ps, cell0, S, p.bsz, p.nb,
                       (const int32_t *)p.boff, p.blocks);
    MIA_HIP(hipGetLastError());
    // their reach, and the items per key
    PlanLaunch L{};
    L.ps = ps;
    L.ncells = p.ncells;
    L.K1 = p.K1;
    L.kseg = p.kseg;
    L.one_key = p.nkeys == 1;
    L.boff = p.boff;
    L.blocks = p.blocks;
    L.bbox = p.bbox;
    L.geo = p.geo;
    L.key_count = p.kc;
    L.key_cursor = p.kcur;
    L.key_off = p.ko;
    L.items = p.items;
    L.cap = p.item_cap;
    L.overflow = p.words + 2;
    const unsigned bgrid = (unsigned)std::max<int64_t>(
        1, std::min<int64_t>((p.nblk_cap + kPlanWaves - 1) / kPlanWaves, 256 * kPlanGridPerCu));
    hipLaunchKernelGGL(k_block_geom, dim3(bgrid), dim3(kPlanThreads), 0, st, L);
    MIA_HIP(hipGetLastError());
    scan_ws<int64_t>((const int64_t *)p.kc, p.ko, p.nkeys, nullptr, p.scan_keys, st);
    hipLaunchKernelGGL(k_items_total, dim3(1), dim3(64), 0, st, (const int64_t *)p.ko, p.nkeys, p.item_cap,
                       p.n_items, p.words + 3);
    MIA_HIP(hipGetLastError());
    const Item *items = p.items;
    const int64_t *cost = p.cost;
    if (p.det) {
        fill<unsigned long long>(p.skey, ~0ull, p.item_cap, st);
        hipLaunchKernelGGL(k_iota, dim3(nblk(p.item_cap, 256)), dim3(256), 0, st, p.sidx, p.item_cap);
        MIA_HIP(hipGetLastError());
        L.sort_key = p.skey;
        L.sort_shift = det_two_sorts(p) ? 64 : det_low_bits(p);
    }
    hipLaunchKernelGGL(k_emit_items, dim3(bgrid), dim3(kPlanThreads), 0, st, L);
    MIA_HIP(hipGetLastError());
    const unsigned igrid = (unsigned)std::max<int64_t>(
        1, std::min<int64_t>((p.item_cap + kPlanWaves - 1) / kPlanWaves, 256 * kPlanGridPerCu));
    hipLaunchKernelGGL(k_item_cost, dim3(igrid), dim3(kPlanThreads), 0, st, ps, (const Block *)p.blocks,
                       (const double *)p.bbox, (const int64_t *)p.n_items, p.items, p.cost, p.words + 1);
    MIA_HIP(hipGetLastError());
    if (p.det) {
        // items of one key in (block, rectangle) order: a stable sort of the whole
        // capacity (unused slots keep the largest key and sort last)
        const bool two = det_two_sorts(p);
        const int32_t *order = p.sidx2;
        size_t bytes = p.stmp_bytes;
        MIA_HIP(hipcub::DeviceRadixSort::SortPairs(p.stmp, bytes, (const unsigned long long *)p.skey, p.skey2,
                                                   (const int32_t *)p.sidx, p.sidx2, (int)p.item_cap, 0,
                                                   two ? det_low_bits(p) : det_key_bits(p), st));
        if (two) {
            hipLaunchKernelGGL(k_item_keys, dim3(nblk(p.item_cap, 256)), dim3(256), 0, st, (const int32_t *)p.sidx2,
                               (const int64_t *)p.n_items, p.item_cap, (const Item *)p.items, p.skey);
            MIA_HIP(hipGetLastError());
            MIA_HIP(hipcub::DeviceRadixSort::SortPairs(p.stmp, bytes, (const unsigned long long *)p.skey, p.skey2,
                                                       (const int32_t *)p.sidx2, p.sidx, (int)p.item_cap, 0,
                                                       det_index_bits(p), st));
            order = p.sidx;
        }
        hipLaunchKernelGGL(k_gather_items, dim3(nblk(p.item_cap, 256)), dim3(256), 0, st, order,
                           (const int64_t *)p.n_items, (const Item *)p.items, (const int64_t *)p.cost, p.items2,
                           p.cost2);
        MIA_HIP(hipGetLastError());
        items = p.items2;
        cost = p.cost2;
    }
    scan_ws<int64_t>(cost, p.cpre, p.item_cap, p.n_items, p.scan_cost, st);
    schedule_batches(p.cpre, p.n_items, &items->np, sizeof(Item) / sizeof(int32_t), p.pc.groups, p.bounds, st, p.det,
                     p.pc.A.shared ? p.pc.wpb : 1);
    if (p.det) {
        // slot numbers of every wave's flushes (slot0[W] = slots in all)
        hipLaunchKernelGGL(k_key_nonempty, dim3(nblk(p.nkeys, 256)), dim3(256), 0, st, (const int64_t *)p.ko,
                           p.nkeys, p.ne);
        MIA_HIP(hipGetLastError());
        scan_ws<int64_t>(p.ne, p.ne_pre, p.nkeys, nullptr, p.scan_ne, st);
        hipLaunchKernelGGL(k_slot_runs, dim3(nblk(p.pc.waves, 256)), dim3(256), 0, st, (const int64_t *)p.bounds,
                           p.pc.waves, (const int64_t *)p.ko, p.nkeys, (const int64_t *)p.ne_pre, p.runs);
        MIA_HIP(hipGetLastError());
        scan_ws<int64_t>(p.runs, p.slot0, p.pc.waves, nullptr, p.scan_runs, st);
    }
    if (ev) MIA_HIP(hipEventRecord(ev[1], st));
    // pair kernel, one launch per r-bin pass
    PairArgs A = p.pc.A;
    A.items = items;
    A.ps = ps;
    A.bbox = p.bbox;
    A.overflow = p.words + 2;
    A.blocks = p.blocks;
    A.n_items = p.n_items;
    A.bounds = p.bounds;
    A.key_off = p.ko;
    A.T = (const double *)(pd + p.off_T);
    A.X = (const double *)(pd + p.off_X);
    A.samples = (const SampleDev *)(pd + p.off_sd);
    A.stat = p.stat;
    A.det = p.det ? 1 : 0;
    A.K1 = p.K1;
    A.slot_cap = p.slot_cap;
    A.slot0 = p.slot0;
    A.slot_key = p.slot_key;
    A.slot_np = p.slot_np;
    A.slot_sp = p.slot_sp;
    A.slot_sx = p.slot_sx;
    A.slot_dd = p.slot_dd;
    A.slot_var = p.slot_var;
    const int n_r = p.pc.A.n_r, n_2 = p.pc.A.n_2;
    for (int pass = 0; pass < p.pc.npass; ++pass) {
        const int r0 = pass * p.pc.nrp, r1 = std::min(n_r, r0 + p.pc.nrp);
        A.n_r = r1 - r0;
        A.nbins = (r1 - r0) * n_2;
        A.bin_off = r0 * n_2;
        A.T = (const double *)(pd + p.off_T) + r0;
        A.T0 = p.T[r0];
        A.Tn = p.T[r1];
        A.lgc = (float)(-p.pc.l0 * p.pc.lgs - r0 + p.pc.shift_r);
        A.queue = p.queue + pass;
        if (A.mode == MIA_RPPI)
            launch_pairs_mode<MIA_RPPI>(A, p.pc.grid, p.pc.wpb, p.pc.lds, st);
        else
            launch_pairs_mode<MIA_RMU>(A, p.pc.grid, p.pc.wpb, p.pc.lds, st);
    }
    if (ev) MIA_HIP(hipEventRecord(ev[2], st));
    if (p.det) {
        const int64_t *slots = p.slot0 + p.pc.waves;  // their number
        const unsigned sgrid = (unsigned)std::max<int64_t>(1, std::min<int64_t>(p.slot_cap, 8192));
        hipLaunchKernelGGL(k_sum_slots, dim3(sgrid, nblk(n_r * n_2, 256)), dim3(256), 0, st, slots, (const int64_t *)p.slot_key, p.slot_np,
                           p.slot_sp, p.slot_sx, p.slot_dd, p.slot_var, n_r * n_2);
        MIA_HIP(hipGetLastError());
        hipLaunchKernelGGL(k_slot_heads, dim3(1), dim3(1024), 0, st, slots, (const int64_t *)p.slot_key, p.heads,
                           p.n_heads);
        MIA_HIP(hipGetLastError());
        hipLaunchKernelGGL(k_finalize_det, dim3(nblk(p.fin_total, 256 / kWave)), dim3(256), 0, st,
                           (const FinSample *)(pd + p.off_fs), fin0, S, (const int64_t *)p.heads,
                           (const int64_t *)p.n_heads, (const int64_t *)p.slot_key,
                           (const unsigned long long *)p.slot_np, (const double *)p.slot_sp, (const double *)p.slot_sx,
                           (const double *)p.slot_dd, (const double *)p.slot_var, n_r * n_2,
                           (const unsigned long long *)p.stat, p.words);
    } else {
        hipLaunchKernelGGL(k_finalize, dim3(nblk(p.fin_total, 256)), dim3(256), 0, st,
                           (const FinSample *)(pd + p.off_fs), fin0, S, (const unsigned long long *)p.stat, p.words);
    }
    MIA_HIP(hipGetLastError());
    if (ev) MIA_HIP(hipEventRecord(ev[3], st));
}

}  // namespace mia
