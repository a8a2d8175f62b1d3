// Batched form: thousands of independent tensor-product integrals of mixed
// rule, family, dimension and size in one launch per kernel class.
//
// The host plan splits every integral into tiles and orders the tile list by
// decreasing integral size (longest first), the tiles of an integral
// contiguous; the dispatcher hands out the large tiles first as workgroups
// finish.  Multi-axis integrals whose factor tables fit in LDS (tq_product.hpp)
// take one workgroup per tile, whose waves share the tables; one-axis
// integrals, and multi-axis ones with longer axes, one wave per tile
// (grid_tile).  Every tile writes one FP64 partial; a last kernel reduces each
// integral's partials in tile order, so results are deterministic for a given
// tiling.  No memset is issued and no counter is kept, so the launches can be
// captured in a graph and replayed.
#include <algorithm>
#include <mutex>
#include <new>
#include <vector>

#include "tq_product.hpp"

namespace tq {

template <typename T>
struct BatchDev {
    int rule, fam, d, n, m, L, nl, lane_count, lane_waves;
    int product;      // 1: `split` and the product kernel, 0: the fields above and grid_tile
    ProductSplit split;
    long long items;
    long long gl_offset;
    double scale;
    Axis ax[TQ_MAX_DIM];
    Params<T> p;
};

template <typename T>
struct BatchTab {
    static constexpr int N = (sizeof(T) == 4) ? 1024 : 512;  // general kernel: per-wave loop table entries
};

// Kernel classes: 0: one-axis integrals; 1, 2: the product kernel with tables
// of up to 26 KB (six workgroups per CU) and up to 60 KB; 3: the general
// kernel.
constexpr int kBatchClasses = 4;
constexpr size_t kProductLdsSmall = 26 * 1024;
constexpr size_t kProductLdsBig = 60 * 1024;
// Lane states of the product kernel: 4 share an entry's LDS read without
// leaving the lanes of small integrals empty.
constexpr int kBatchStates = 4;
// Outer lane tables (ProductSplit) of two axes up to this many entries: from
// n = 17 on, four parts of a single axis lose little.
constexpr int kBatchOuter = 256;

// General kernel: loop-axis table when it fits, row axes recomputed per row.
template <typename T, int FAM, int PATHS>
__device__ __forceinline__ double batch_tile_general(const BatchDev<T>& D, const Axis* ax, T* tab, bool table,
                                                     const double* glx, const double* glw, int lw0, int lw1,
                                                     long long t0, long long t1) {
    if (table) {
        const int lane = threadIdx.x & (kWave - 1);
        for (int j = lane; j < D.nl; j += kWave)
            loop_table_entry<T, FAM>(tab, j, ax, D.L, D.n, D.rule, glx, glw, D.p);
    }
    // make this wave's LDS writes visible to all of its lanes
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    double acc = 0.0;
    for (int lw = lw0; lw < lw1; ++lw)
        acc += table ? grid_tile<T, FAM, true, false, true, PATHS>(D.d, D.n, D.nl, D.m, D.L, D.rule, D.lane_count,
                                                                   D.p, ax, tab, glx, glw, lw, t0, t1)
                     : grid_tile<T, FAM, false, false, true, PATHS>(D.d, D.n, D.nl, D.m, D.L, D.rule, D.lane_count,
                                                                    D.p, ax, tab, glx, glw, lw, t0, t1);
    return acc;
}

template <typename T, int PATHS>
__device__ __forceinline__ double batch_tile(const BatchDev<T>& D, const Axis* ax, T* tab, bool table,
                                             const double* glx, const double* glw, int lw0, int lw1, long long t0,
                                             long long t1) {
    switch (D.fam) {
#define TQ_BT(F) \
    case F: return batch_tile_general<T, F, PATHS>(D, ax, tab, table, glx, glw, lw0, lw1, t0, t1);
        TQ_BT(TQ_FAM_GAUSSIAN_PEAK)
        TQ_BT(TQ_FAM_OSCILLATORY)
        TQ_BT(TQ_FAM_PRODUCT_PEAK)
        TQ_BT(TQ_FAM_EXP_LINEAR)
        TQ_BT(TQ_FAM_SIN_SUM)
        TQ_BT(TQ_FAM_DOUBLE_GAUSSIAN)
        TQ_BT(TQ_FAM_CONSTANT)
#undef TQ_BT
        default: return 0.0;
    }
}

// A Gauss-Legendre integral whose n nodes at gl_offset are not all inside
// the gl_len-entry tables reads nothing and yields NaN (tq_batch_plan checks
// items without the tables; this is where their length is known).
template <typename T>
__device__ inline bool gl_in_range(const BatchDev<T>& D, const double* glx, const double* glw, long long gl_len) {
    return D.rule != TQ_RULE_GAUSS_LEGENDRE || (glx && glw && D.gl_offset >= 0 && D.gl_offset + D.n <= gl_len);
}

// One-axis Gauss-Legendre tiles of FP32 batches whose tables are given as
// FP32 pairs: gl_pair_rows instead of grid_tile.
template <typename T>
__device__ inline bool gl_pair_tile(const BatchDev<T>& D, const float* glp32) {
    return sizeof(T) == 4 && glp32 && D.m == 0 && D.rule == TQ_RULE_GAUSS_LEGENDRE;
}

__device__ __forceinline__ double gl_pair_tile_sum(const BatchDev<float>& D, const float* pairs, long long t0,
                                                   long long t1) {
    switch (D.fam) {
#define TQ_GP(F) \
    case F: return gl_pair_rows<F>(D.n, D.p, D.ax[0], pairs, t0, t1);
        TQ_GP(TQ_FAM_GAUSSIAN_PEAK)
        TQ_GP(TQ_FAM_OSCILLATORY)
        TQ_GP(TQ_FAM_PRODUCT_PEAK)
        TQ_GP(TQ_FAM_EXP_LINEAR)
        TQ_GP(TQ_FAM_SIN_SUM)
        TQ_GP(TQ_FAM_DOUBLE_GAUSSIAN)
        TQ_GP(TQ_FAM_CONSTANT)
#undef TQ_GP
        default: return 0.0;
    }
}

// One wave's tile of a grid_tile integral; `ax` and `region` are the wave's
// LDS (region unused by one-axis tiles).  PATHS (grid_tile) keeps the code of
// other kinds of tiles out.  PAIRS: the FP32 pair tables are there, so a
// one-axis Gauss-Legendre tile reads those.
template <typename T, int PATHS, bool PAIRS>
__device__ __forceinline__ void wave_tile(const BatchDev<T>& D, const tq_batch_tile& tile, Axis* ax, double* region,
                                          const double* glx, const double* glw, const float* glp32, long long gl_len,
                                          double* part) {
    const int lane = threadIdx.x & (kWave - 1);
    double acc = __longlong_as_double(0x7ff8000000000000ll);
    if (gl_in_range(D, glx, glw, gl_len)) {
        bool done = false;
        if constexpr (PAIRS && sizeof(T) == 4) {
            if (gl_pair_tile(D, glp32)) {
                acc = gl_pair_tile_sum(D, glp32 + 2 * D.gl_offset, tile.t0, tile.t1);
                done = true;
            }
        }
        if (!done) {
            constexpr int NT = BatchTab<T>::N;
            const double* gx = glx ? glx + D.gl_offset : nullptr;
            const double* gw = glw ? glw + D.gl_offset : nullptr;
            for (int k = lane; k < D.d; k += kWave) ax[k] = D.ax[k];
            wave_lds_fence();
            const bool table = (PATHS & kPathsMultiAxis) != 0 && D.m > 0 && D.L >= 0 && D.nl * tab_stride(D.fam) <= 2 * NT;
            acc = batch_tile<T, PATHS>(D, ax, reinterpret_cast<T*>(region), table, gx, gw, tile.lane_wave,
                                       tile.lane_wave_end, tile.t0, tile.t1);
        }
        acc = wave_sum(acc);
    }
    if (lane == 0) *part = acc;
}

// One wave per tile, tiles [0, n_tiles) in the planner's order (longest
// integrals first), so the hardware dispatcher hands them out largest first
// as waves finish.  A persistent form (each wave claiming tiles from 16
// atomic queues) held its claim loop's state and the hoisted per-tile
// invariants for the whole kernel: 164 VGPRs against 112, and the
// 8192-integral Genz batch took 0.441 ms against 0.344.  PATHS ==
// kPathsAll serves runs without classes: product tiles are left to that kernel.
template <typename T, int PATHS>
__global__ __launch_bounds__(kBlock) void k_batch(const BatchDev<T>* descs, const tq_batch_tile* tiles,
                                                  long long n_tiles, const double* glx, const double* glw,
                                                  const float* glp32, long long gl_len, double* tile_part) {
    __shared__ Axis s_ax[kWavesPerBlock][TQ_MAX_DIM];
    __shared__ double s_region[kWavesPerBlock][(int)(2 * BatchTab<T>::N * sizeof(T)) / 8];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long long t = (long long)blockIdx.x * kWavesPerBlock + wave;
    if (t >= n_tiles) return;
    const tq_batch_tile tile = tiles[t];
    const BatchDev<T>& D = descs[tile.item];
    if (PATHS == kPathsAll && D.product) return;
    wave_tile<T, PATHS, (PATHS & kPathsGauss) != 0>(D, tile, s_ax[wave], s_region[wave], glx, glw, glp32, gl_len,
                                                    tile_part + t);
}

// Product tiles: one workgroup per tile.  Its waves build the integral's
// tables together and then share the tile's work: (lane group, quarter of
// the items) pairs, or whole lane groups when their number is a multiple of
// the waves.
template <typename T, int FAM>
__device__ __forceinline__ double batch_product_tile(const BatchDev<T>& D, const Axis* ax, const double* glx,
                                                     const double* glw, const tq_batch_tile& tile,
                                                     unsigned char* lds, int* s_exp) {
    const ProductSplit& S = D.split;
    const ProductTables<T> tab = build_product_tables<FAM, T>(S, D.rule, ax, glx, glw, D.p, lds, s_exp);
    const int lane_groups = tile.lane_wave_end - tile.lane_wave;
    const long long items = tile.t1 - tile.t0;
    const int parts = lane_groups % kWavesPerBlock == 0 ? 1 : kWavesPerBlock;
    const long long per = (items + parts - 1) / parts;
    double acc = 0.0;
    Factor<FAM, T> own[kBatchStates];
    double wl[kBatchStates];
    for (int u = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); u < lane_groups * parts; u += kWavesPerBlock) {
        const int lg = u / parts, part = u - lg * parts;
        const long long t0 = tile.t0 + part * per, t1 = t0 + per < tile.t1 ? t0 + per : tile.t1;
        if (t0 >= t1) continue;
        lane_states<FAM, T, kBatchStates>(S, tab, (tile.lane_wave + lg) * kWave + (int)(threadIdx.x & (kWave - 1)), own,
                                          wl);
        acc += sum_items<FAM, T, kBatchStates>(S, tab, own, wl, t0, t1);
    }
    return acc;
}

template <typename T>
__device__ __forceinline__ void product_block(const BatchDev<T>& D, const tq_batch_tile& tile, Axis* s_ax,
                                              unsigned char* s_lds, const double* glx, const double* glw,
                                              long long gl_len, double* part) {
    __shared__ int s_exp[kExpSlots];
    __shared__ double s_red[kWavesPerBlock];
    const int tid = threadIdx.x;
    if (!gl_in_range(D, glx, glw, gl_len)) {
        if (tid == 0) *part = __longlong_as_double(0x7ff8000000000000ll);
        return;
    }
    const double* gx = glx ? glx + D.gl_offset : nullptr;
    const double* gw = glw ? glw + D.gl_offset : nullptr;
    if (tid < D.d) s_ax[tid] = D.ax[tid];
    __syncthreads();
    double acc = 0.0;
    switch (D.fam) {
#define TQ_BP(F) \
    case F: acc = batch_product_tile<T, F>(D, s_ax, gx, gw, tile, s_lds, s_exp); break;
        TQ_BP(TQ_FAM_GAUSSIAN_PEAK)
        TQ_BP(TQ_FAM_OSCILLATORY)
        TQ_BP(TQ_FAM_PRODUCT_PEAK)
        TQ_BP(TQ_FAM_EXP_LINEAR)
        TQ_BP(TQ_FAM_SIN_SUM)
        TQ_BP(TQ_FAM_DOUBLE_GAUSSIAN)
        TQ_BP(TQ_FAM_CONSTANT)
#undef TQ_BP
    }
    acc = block_sum(acc, s_red);
    if (tid == 0) *part = scale_back(D.fam, acc, D.d, s_exp);
}

// Product tiles alone (big tables; runs without classes).
template <typename T>
__global__ __launch_bounds__(kBlock) void k_batch_product(const BatchDev<T>* descs, const tq_batch_tile* tiles,
                                                          const double* glx, const double* glw, long long gl_len,
                                                          double* tile_part) {
    extern __shared__ __align__(16) unsigned char s_lds[];
    __shared__ Axis s_ax[TQ_MAX_DIM];
    const tq_batch_tile tile = tiles[blockIdx.x];
    const BatchDev<T>& D = descs[tile.item];
    if (!D.product) return;  // a run without classes: the other kernel's tile
    product_block<T>(D, tile, s_ax, s_lds, glx, glw, gl_len, tile_part + blockIdx.x);
}

// The two main classes in one launch: one-axis tiles, a wave each (their
// Gauss-Legendre rows are bound by table reads, the others by arithmetic),
// and product tiles, a workgroup each, interleaved over the grid in
// proportion, each class in its own order.  Both kinds then share every CU
// from start to end; on two streams the second kernel waited for the first
// one's workgroups to leave, and forking and joining the streams alone took
// about 30 us.  8192 Genz integrals (1.05e9 points, default tiles): 370 us
// with a transcendental per point, 175 us with product tiles on their own
// stream, 150 us so (one-axis tiles alone 76 us, product tiles alone 71 us:
// the multiply-adds and the one-axis transcendentals bound it).
template <typename T, bool PAIRS>
__global__ __launch_bounds__(kBlock) void k_batch_mixed(const BatchDev<T>* descs, const tq_batch_tile* tiles,
                                                        unsigned n_one, unsigned n_product, const double* glx,
                                                        const double* glw, const float* glp32, long long gl_len,
                                                        double* tile_part) {
    extern __shared__ __align__(16) unsigned char s_lds[];
    __shared__ Axis s_ax[TQ_MAX_DIM];
    const unsigned one_blocks = (n_one + kWavesPerBlock - 1) / kWavesPerBlock;
    const unsigned long long total = (unsigned long long)one_blocks + n_product;
    // one-axis blocks among the first b blocks: floor(b one_blocks / total)
    const unsigned before = (unsigned)((unsigned long long)blockIdx.x * one_blocks / total);
    const unsigned upto = (unsigned)(((unsigned long long)blockIdx.x + 1) * one_blocks / total);
    if (upto == before) {
        const unsigned t = n_one + blockIdx.x - before;
        const tq_batch_tile tile = tiles[t];
        product_block<T>(descs[tile.item], tile, s_ax, s_lds, glx, glw, gl_len, tile_part + t);
        return;
    }
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const unsigned t = before * kWavesPerBlock + wave;
    if (t >= n_one) return;
    const tq_batch_tile tile = tiles[t];
    wave_tile<T, PAIRS && sizeof(T) == 4 ? kPathsNewtonCotes : kPathsOneAxis, PAIRS>(
        descs[tile.item], tile, s_ax + wave, nullptr, glx, glw, glp32, gl_len, tile_part + t);
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_batch_finalize(const BatchDev<T>* descs, long long count,
                                                           const int64_t* tile_begin, const int64_t* tile_count,
                                                           const double* tile_part, T* out, double* out64) {
    const long long i = (long long)blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6);
    const int lane = threadIdx.x & (kWave - 1);
    if (i >= count) return;
    const long long b = tile_begin[i], c = tile_count[i];
    double v = 0.0;
    for (long long j = lane; j < c; j += kWave) v += tile_part[b + j];
    v = wave_sum(v);
    if (lane == 0) {
        const double r = v * descs[i].scale;
        if (out) out[i] = (T)r;
        if (out64) out64[i] = r;
    }
}

static int check_item(const tq_batch_item& it) {
    if (it.family < 0 || it.family >= TQ_NUM_FAMILIES) return fail(TQ_E_ARG, "batch item: unknown family");
    if (it.dim < 1 || it.dim > TQ_MAX_DIM) return fail(TQ_E_ARG, "batch item: dim out of range (1..16)");
    switch (it.rule) {
        case TQ_RULE_TRAPEZOID:
            if (it.n < 2) return fail(TQ_E_ARG, "batch item: Trapezoid needs n >= 2");
            break;
        case TQ_RULE_SIMPSON:
            if (it.n < 3 || it.n % 2 != 1) return fail(TQ_E_ARG, "batch item: Simpson needs odd n >= 3");
            break;
        case TQ_RULE_BOOLE:
            if (it.n < 5 || (it.n - 1) % 4 != 0) return fail(TQ_E_ARG, "batch item: Boole needs n = 1 + 4k");
            break;
        case TQ_RULE_GAUSS_LEGENDRE:
            if (it.n < 1 || it.gl_offset < 0) return fail(TQ_E_ARG, "batch item: bad Gauss-Legendre n/offset");
            break;
        default: return fail(TQ_E_ARG, "batch item: unknown rule");
    }
    long long P;
    if (ipow_checked(it.n, it.dim, 1LL << 62, &P) != 0) return fail(TQ_E_ARG, "batch item: n^dim too large");
    return TQ_OK;
}

// Split-mode integrals (one axis, m == 0) walk one 64-node row per item
// (Gauss-Legendre: 64 nodes and their 64 mirrors).  Gauss-Legendre rows
// wait on global loads of the node tables, so shorter tiles spread them
// over more waves; Newton-Cotes rows compute their nodes and take longer
// tiles, which spread the per-tile cost over more points.
constexpr long long kSplitMaxItemsGL = 128;
constexpr long long kSplitMaxItemsNC = 512;

static long long tile_ipw(const GridGeom& G, long long tile_points) {
    long long ipw = tile_points / kWave;
    const long long cap = G.rule == TQ_RULE_GAUSS_LEGENDRE ? kSplitMaxItemsGL : kSplitMaxItemsNC;
    if (G.m == 0 && ipw > cap) ipw = cap;
    if (ipw < 1) ipw = 1;
    if (ipw > G.items) ipw = G.items;
    return ipw;
}

// Workgroups share a tile's tables, so product tiles are this many times the
// wave tiles' points: the tables' cost (d n FP64 evaluations) stays a
// fraction of the tile's (6920 integrals, default tiles: 106 us with 16, 80
// with 64).
constexpr long long kProductTileFactor = 64;

struct BatchGeom {
    GridGeom g;
    ProductSplit s;
    bool product;
    int cls;
    long long lane_step;  // 64-lane groups per tile
};

// Geometry of an integral in the product kernel; false: its tables do not fit.
static bool plan_product_item(const tq_batch_item& it, int tsize, long long tile_points, BatchGeom& B) {
    const int d = it.dim, n = it.n, C = family_comps(it.family);
    const long long entries = 8192 / ((long long)C * tsize);  // two loop axes while their table stays at 8 KB
    if (!split_product_axes(d, n, kBatchStates, C, tsize, entries < n + kGroup ? n + kGroup : entries, kBatchOuter, 0,
                            kProductLdsBig, B.s))
        return false;
    const ProductSplit& S = B.s;
    B.cls = product_lds_bytes(S, C, tsize) <= kProductLdsSmall ? 1 : 2;
    GridGeom& G = B.g;
    G.d = d;
    G.n = n;
    G.rule = it.rule;
    G.m = S.outer + S.inner;
    G.L = S.L;
    G.nl = S.nl;
    G.lane_count = S.slots;
    G.lane_waves = S.lane_groups;
    G.items = S.items;
    // tiles: ranges of whole lane groups (a multiple of the waves, so that
    // each takes whole ones), and ranges of at least 16 items where that does
    // not make enough of them
    long long P;
    ipow_checked(n, d, 1LL << 62, &P);
    const long long target = tile_points * kProductTileFactor;
    const long long tiles = (P + target - 1) / target;
    long long lane_parts = S.lane_groups / kWavesPerBlock;
    if (lane_parts > tiles) lane_parts = tiles;
    if (lane_parts < 1) lane_parts = 1;
    B.lane_step = (S.lane_groups + lane_parts - 1) / lane_parts;
    if (lane_parts > 1) B.lane_step = (B.lane_step + kWavesPerBlock - 1) / kWavesPerBlock * kWavesPerBlock;
    const long long item_parts = (tiles + lane_parts - 1) / lane_parts;
    G.ipw = (S.items + item_parts - 1) / item_parts;
    if (G.ipw < 16) G.ipw = S.items < 16 ? S.items : 16;
    G.chunks = (G.items + G.ipw - 1) / G.ipw;
    return true;
}

template <typename T>
static int plan_batch(const tq_batch_item* items, long long count, long long tile_points, BatchDev<T>* desc,
                      tq_batch_tile* tiles, int64_t* tile_begin, int64_t* tile_count, long long* n_tiles_out,
                      int64_t* class_offsets = nullptr) {
    struct Entry {
        int cls;
        long long cost;
        long long idx;
    };
    std::vector<Entry> order(count > 0 ? count : 1);
    std::vector<BatchGeom> geo(count > 0 ? count : 1);
    long long total = 0;
    for (long long i = 0; i < count; ++i) {
        const tq_batch_item& it = items[i];
        BatchGeom& B = geo[i];
        int rc = check_item(it);
        if (rc) return rc;
        B.product = plan_product_item(it, (int)sizeof(T), tile_points, B);
        if (!B.product) {
            rc = plan_geom(it.dim, it.n, it.rule, 0, 1, 1, B.g);
            if (rc) return rc;
            GridGeom& G = B.g;
            G.ipw = tile_ipw(G, tile_points);
            G.chunks = (G.items + G.ipw - 1) / G.ipw;
            // a lane group's whole loop is shorter than a tile: several groups per tile
            long long step = 1;
            if (G.chunks == 1) {
                step = tile_points / ((long long)kWave * G.items);
                if (step < 1) step = 1;
                if (step > G.lane_waves) step = G.lane_waves;
            }
            B.lane_step = step;
            B.cls = G.m == 0 ? 0 : 3;
        }
        const GridGeom& G = B.g;
        long long P;
        ipow_checked(it.n, it.dim, 1LL << 62, &P);
        order[i] = {B.cls, P, i};
        total += G.chunks * ((G.lane_waves + B.lane_step - 1) / B.lane_step);
        if (desc) {
            BatchDev<T>& D = desc[i];
            D.rule = it.rule;
            D.fam = it.family;
            D.d = it.dim;
            D.n = it.n;
            D.m = G.m;
            D.L = G.L;
            D.nl = G.nl;
            D.lane_count = G.lane_count;
            D.lane_waves = G.lane_waves;
            D.product = B.product ? 1 : 0;
            if (B.product) D.split = B.s;
            D.items = G.items;
            D.gl_offset = it.rule == TQ_RULE_GAUSS_LEGENDRE ? it.gl_offset : 0;
            double scale = it.c0;
            for (int k = 0; k < TQ_MAX_DIM; ++k) {
                if (k < it.dim) {
                    D.ax[k] = make_axis_host(it.domain[2 * k], it.domain[2 * k + 1], it.n, it.rule);
                    scale *= axis_scale(it.domain[2 * k], it.domain[2 * k + 1], it.n, it.rule);
                } else {
                    D.ax[k] = Axis{0.0, 0.0, 0.0};
                }
            }
            D.scale = scale;
            tq_integrand f{};
            f.family = it.family;
            f.dim = it.dim;
            f.c0 = it.c0;
            f.c1 = it.c1;
            f.c2 = it.c2;
            f.c3 = it.c3;
            for (int k = 0; k < TQ_MAX_DIM; ++k) {
                f.a[k] = it.a[k];
                f.u[k] = it.u[k];
            }
            D.p = make_params<T>(f);
        }
    }
    if (tiles) {
        // by kernel class, then longest integrals first; stable on the index
        std::sort(order.begin(), order.begin() + count, [](const Entry& x, const Entry& y) {
            if (x.cls != y.cls) return x.cls < y.cls;
            return x.cost != y.cost ? x.cost > y.cost : x.idx < y.idx;
        });
        long long t = 0;
        int next_cls = 0;
        for (long long o = 0; o < count; ++o) {
            const long long i = order[o].idx;
            while (class_offsets && next_cls <= order[o].cls) class_offsets[next_cls++] = t;
            const GridGeom& G = geo[i].g;
            tile_begin[i] = t;
            const long long step = geo[i].lane_step;
            for (long long lw = 0; lw < G.lane_waves; lw += step) {
                for (long long c = 0; c < G.chunks; ++c) {
                    tq_batch_tile& tl = tiles[t++];
                    tl.item = (int32_t)i;
                    tl.lane_wave = (int32_t)lw;
                    tl.lane_wave_end = (int32_t)(lw + step < G.lane_waves ? lw + step : G.lane_waves);
                    tl.reserved = 0;
                    tl.t0 = c * G.ipw;
                    tl.t1 = (c + 1) * G.ipw < G.items ? (c + 1) * G.ipw : G.items;
                }
            }
            tile_count[i] = t - tile_begin[i];
        }
        while (class_offsets && next_cls <= kBatchClasses) class_offsets[next_cls++] = t;
    }
    *n_tiles_out = total;
    return TQ_OK;
}

static int plan_any(const tq_batch_item* items, long long count, int dtype, long long tile_points, void* desc,
                    tq_batch_tile* tiles, int64_t* tile_begin, int64_t* tile_count, long long* n_tiles,
                    int64_t* class_offsets) {
    try {
        return dtype == TQ_F32 ? plan_batch<float>(items, count, tile_points, (BatchDev<float>*)desc, tiles,
                                                   tile_begin, tile_count, n_tiles, class_offsets)
                               : plan_batch<double>(items, count, tile_points, (BatchDev<double>*)desc, tiles,
                                                    tile_begin, tile_count, n_tiles, class_offsets);
    } catch (const std::bad_alloc&) {
        return fail(TQ_E_WORKSPACE, "out of host memory for the batch plan");
    }
}

template <typename T, int PATHS>
static int launch_class(const void* desc, const tq_batch_tile* tiles, long long n, const double* glx,
                        const double* glw, const float* glp32, long long gl_len, double* tile_part, hipStream_t s) {
    if (n <= 0) return TQ_OK;
    const long long blocks = (n + kWavesPerBlock - 1) / kWavesPerBlock;
    hipLaunchKernelGGL((k_batch<T, PATHS>), dim3((unsigned)blocks), dim3(kBlock), 0, s, (const BatchDev<T>*)desc,
                       tiles, n, glx, glw, glp32, gl_len, tile_part);
    return check_launch("k_batch");
}

// Classes 0 and 1: tiles [0, n_one) and [n_one, n_one + n_product).
template <typename T>
static int launch_mixed(const void* desc, const tq_batch_tile* tiles, long long n_one, long long n_product,
                        const double* glx, const double* glw, const float* glp32, long long gl_len, double* tile_part,
                        hipStream_t s) {
    if (n_one + n_product <= 0) return TQ_OK;
    const long long blocks = (n_one + kWavesPerBlock - 1) / kWavesPerBlock + n_product;
    const size_t lds = n_product > 0 ? kProductLdsSmall : 0;
    if constexpr (sizeof(T) == 4) {
        if (glp32) {
            hipLaunchKernelGGL((k_batch_mixed<T, true>), dim3((unsigned)blocks), dim3(kBlock), lds, s,
                               (const BatchDev<T>*)desc, tiles, (unsigned)n_one, (unsigned)n_product, glx, glw, glp32,
                               gl_len, tile_part);
            return check_launch("k_batch_mixed");
        }
    }
    hipLaunchKernelGGL((k_batch_mixed<T, false>), dim3((unsigned)blocks), dim3(kBlock), lds, s,
                       (const BatchDev<T>*)desc, tiles, (unsigned)n_one, (unsigned)n_product, glx, glw, glp32, gl_len,
                       tile_part);
    return check_launch("k_batch_mixed");
}

template <typename T>
static int launch_product(const void* desc, const tq_batch_tile* tiles, long long n, const double* glx,
                          const double* glw, long long gl_len, double* tile_part, size_t lds, hipStream_t s) {
    if (n <= 0) return TQ_OK;
    hipLaunchKernelGGL((k_batch_product<T>), dim3((unsigned)n), dim3(kBlock), lds, s, (const BatchDev<T>*)desc, tiles,
                       glx, glw, gl_len, tile_part);
    return check_launch("k_batch_product");
}

// Library-owned stream on which the rare classes (big tables, general
// kernel) run beside the mixed launch when both have tiles.  Created once per
// device (default priority) and kept; fork and join go through events, so a
// captured run is one forked subgraph.  Runs on one device enqueue their
// fork, launches and join under that device's lock, since the events are
// shared.
constexpr int kMaxBatchDevices = 64;
struct BatchAux {
    hipStream_t st = nullptr;
    hipEvent_t fork = nullptr;
    hipEvent_t join = nullptr;
    std::mutex mu;
    bool ready = false;
};
static BatchAux g_aux[kMaxBatchDevices];
static std::mutex g_aux_mu;

static int hip_check(hipError_t e, const char* what) {
    if (e == hipSuccess) return TQ_OK;
    set_error("%s: %s", what, hipGetErrorString(e));
    return (int)e;
}

static int batch_aux(BatchAux** out) {
    int dev = -1;
    int rc = hip_check(hipGetDevice(&dev), "hipGetDevice");
    if (rc) return rc;
    if (dev < 0 || dev >= kMaxBatchDevices) return fail(TQ_E_UNSUPPORTED, "device index beyond the batch stream table");
    std::lock_guard<std::mutex> lock(g_aux_mu);
    BatchAux& a = g_aux[dev];
    if (!a.ready) {
        rc = hip_check(hipStreamCreateWithFlags(&a.st, hipStreamNonBlocking), "hipStreamCreateWithFlags");
        if (!rc) rc = hip_check(hipEventCreateWithFlags(&a.fork, hipEventDisableTiming), "hipEventCreateWithFlags");
        if (!rc) rc = hip_check(hipEventCreateWithFlags(&a.join, hipEventDisableTiming), "hipEventCreateWithFlags");
        if (rc) return rc;
        a.ready = true;
    }
    *out = &a;
    return TQ_OK;
}

// Classes 0 and 1 on s0, the rare ones on s1.
template <typename T>
static int run_classes(const void* desc, const tq_batch_tile* tiles, const int64_t* off, const double* glx,
                       const double* glw, const float* glp32, long long gl_len, double* tile_part, hipStream_t s0,
                       hipStream_t s1) {
    int rc = launch_mixed<T>(desc, tiles, off[1], off[2] - off[1], glx, glw, glp32, gl_len, tile_part, s0);
    if (!rc)
        rc = launch_product<T>(desc, tiles + off[2], off[3] - off[2], glx, glw, gl_len, tile_part + off[2],
                               kProductLdsBig, s1);
    if (!rc)
        rc = launch_class<T, kPathsMultiAxis>(desc, tiles + off[3], off[4] - off[3], glx, glw, glp32, gl_len,
                                              tile_part + off[3], s1);
    return rc;
}

template <typename T>
static int run_batch(const void* desc, long long count, const tq_batch_tile* tiles, long long n_tiles,
                     const int64_t* tile_begin, const int64_t* tile_count, const double* glx, const double* glw,
                     const float* glp32, long long gl_len, double* tile_part, void* out, double* out64,
                     const int64_t* class_offsets, hipStream_t s) {
    int rc = TQ_OK;
    if (!class_offsets) {
        // no classes: each tile is taken by one of the general kernel with
        // all paths and the product kernel
        rc = launch_class<T, kPathsAll>(desc, tiles, n_tiles, glx, glw, glp32, gl_len, tile_part, s);
        if (!rc) rc = launch_product<T>(desc, tiles, n_tiles, glx, glw, gl_len, tile_part, kProductLdsBig, s);
    } else {
        const int64_t* off = class_offsets;
        for (int c = 0; c < kBatchClasses; ++c)
            if (off[0] != 0 || off[c] < 0 || off[c] > off[c + 1] || off[kBatchClasses] != n_tiles)
                return fail(TQ_E_ARG, "class_offsets do not partition the tiles");
        if (off[2] == 0 || off[4] == off[2]) {
            rc = run_classes<T>(desc, tiles, off, glx, glw, glp32, gl_len, tile_part, s, s);
        } else {
            BatchAux* aux = nullptr;
            rc = batch_aux(&aux);
            if (rc) return rc;
            std::lock_guard<std::mutex> lock(aux->mu);
            rc = hip_check(hipEventRecord(aux->fork, s), "hipEventRecord");
            if (!rc) rc = hip_check(hipStreamWaitEvent(aux->st, aux->fork, 0), "hipStreamWaitEvent");
            if (!rc) rc = run_classes<T>(desc, tiles, off, glx, glw, glp32, gl_len, tile_part, s, aux->st);
            if (!rc) rc = hip_check(hipEventRecord(aux->join, aux->st), "hipEventRecord");
            if (!rc) rc = hip_check(hipStreamWaitEvent(s, aux->join, 0), "hipStreamWaitEvent");
        }
    }
    if (rc) return rc;
    const long long fb = (count + kWavesPerBlock - 1) / kWavesPerBlock;
    hipLaunchKernelGGL((k_batch_finalize<T>), dim3((unsigned)(fb > 0 ? fb : 1)), dim3(kBlock), 0, s,
                       (const BatchDev<T>*)desc, count, tile_begin, tile_count, tile_part, (T*)out, out64);
    return check_launch("k_batch_finalize");
}

}  // namespace tq

using namespace tq;

extern "C" {

int tq_batch_plan_sizes(const tq_batch_item* items, int64_t count, int32_t dtype, int64_t tile_points,
                        int64_t* desc_bytes, int64_t* n_tiles) {
    if (!items || !desc_bytes || !n_tiles) return fail(TQ_E_NULL, "NULL argument");
    if (count < 0 || tile_points < 1) return fail(TQ_E_ARG, "count/tile_points out of range");
    if (dtype != TQ_F32 && dtype != TQ_F64) return fail(TQ_E_ARG, "dtype must be TQ_F32 or TQ_F64");
    long long nt = 0;
    const int rc = plan_any(items, count, dtype, tile_points, nullptr, nullptr, nullptr, nullptr, &nt, nullptr);
    if (rc) return rc;
    *n_tiles = nt;
    *desc_bytes = (int64_t)count * (dtype == TQ_F32 ? (int64_t)sizeof(BatchDev<float>) : (int64_t)sizeof(BatchDev<double>));
    return TQ_OK;
}

int tq_batch_plan(const tq_batch_item* items, int64_t count, int32_t dtype, int64_t tile_points, void* desc_out,
                  tq_batch_tile* tiles_out, int64_t* tile_begin, int64_t* tile_count, int64_t* class_offsets) {
    if (!items || !desc_out || !tiles_out || !tile_begin || !tile_count) return fail(TQ_E_NULL, "NULL argument");
    if (count < 0 || tile_points < 1) return fail(TQ_E_ARG, "count/tile_points out of range");
    if (dtype != TQ_F32 && dtype != TQ_F64) return fail(TQ_E_ARG, "dtype must be TQ_F32 or TQ_F64");
    long long nt = 0;
    return plan_any(items, count, dtype, tile_points, desc_out, tiles_out, tile_begin, tile_count, &nt, class_offsets);
}

int tq_batch_run(int32_t dtype, const void* desc, int64_t count, const tq_batch_tile* tiles, int64_t n_tiles,
                 const int64_t* tile_begin, const int64_t* tile_count, const double* gl_nodes,
                 const double* gl_weights, const float* gl_pairs32, int64_t gl_len, double* tile_partials,
                 void* out, double* out64, const int64_t* class_offsets, void* stream) {
    if (!desc || !tiles || !tile_begin || !tile_count || !tile_partials) return fail(TQ_E_NULL, "NULL argument");
    if (gl_len < 0) return fail(TQ_E_ARG, "gl_len must be >= 0");
    if (gl_len > 0 && (!gl_nodes || !gl_weights)) return fail(TQ_E_NULL, "gl_len > 0 with NULL node/weight tables");
    if (count < 0 || n_tiles < 0 || n_tiles > 0xffffffffLL) return fail(TQ_E_ARG, "count/n_tiles out of range");
    if (!out && !out64) return fail(TQ_E_NULL, "no output pointer");
    if (dtype == TQ_F32)
        return run_batch<float>(desc, count, tiles, n_tiles, tile_begin, tile_count, gl_nodes, gl_weights,
                                gl_pairs32, gl_len, tile_partials, out, out64, class_offsets, as_stream(stream));
    if (dtype == TQ_F64)
        return run_batch<double>(desc, count, tiles, n_tiles, tile_begin, tile_count, gl_nodes, gl_weights,
                                 nullptr, gl_len, tile_partials, out, out64, class_offsets, as_stream(stream));
    return fail(TQ_E_ARG, "dtype must be TQ_F32 or TQ_F64");
}

}  // extern "C"
