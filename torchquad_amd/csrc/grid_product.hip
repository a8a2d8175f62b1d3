// The fused grid kernel of integrals with at least two axes whose factor
// tables fit in LDS (tq_product.hpp says how values become products).
//
// Index space (ProductSplit): lanes hold K combinations of the last axes, the
// loop runs over one or two axes whose combined factors form an LDS table,
// and the leading axes are rows, their factors merged into the states once
// per row.  A wave owns one group of 64 lane slots and a contiguous range of
// (row, group of four loop points).
#include "tq_grid_launch.hpp"
#include "tq_product.hpp"

namespace tq {

struct ProductGeom {
    ProductSplit s;
    int rule, K;
    long long ipw;  // items per wave
    long long num_waves, blocks;
};

template <typename T>
struct ProductArgs {
    ProductGeom g;
    const T* domain;
    const double* glx;
    const double* glw;
    BlockSums sums;
    T* out;
    double* out64;
    double c0;
    Params<T> p;
};

constexpr int kProductWaves = 8;  // waves per block

// Waves per SIMD that the registers must allow (80 VGPRs, 96 where the FP64
// sine of the table build needs them): more waves did not help (d=5 n=65:
// 34.5 us with 6, 34.6 with 8, 35.8 with 4, 45 with 2).
constexpr int product_waves_per_simd(int fam, int tsize) {
    return (family_comps(fam) == 2 && tsize == 8) || fam == TQ_FAM_SIN_SUM ? 5 : 6;
}

template <typename T, int FAM, int K>
__global__ __launch_bounds__(kProductWaves * kWave, product_waves_per_simd(FAM, sizeof(T))) void k_grid_product(ProductArgs<T> A) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ Axis s_axis[TQ_MAX_DIM];
    __shared__ int s_exp[kExpSlots];
    __shared__ double s_red[kProductWaves], s_scale[TQ_MAX_DIM];
    const ProductGeom& g = A.g;
    const int tid = threadIdx.x, d = g.s.d;
    if (tid < d) {
        const Axis a = make_axis(A.domain, tid, g.s.n, g.rule);
        s_axis[tid] = a;
        s_scale[tid] = axis_scale_of(a, g.rule);
    }
    __syncthreads();
    const ProductTables<T> tab = build_product_tables<FAM, T>(g.s, g.rule, s_axis, A.glx, A.glw, A.p, smem_raw, s_exp);

    double acc = 0.0;
    const long long wave = (long long)blockIdx.x * kProductWaves + __builtin_amdgcn_readfirstlane(tid >> 6);
    if (wave < g.num_waves) {
        const unsigned uw = (unsigned)wave, ulg = (unsigned)g.s.lane_groups;
        const unsigned chunk = uw / ulg;
        const int lg = (int)(uw - chunk * ulg);
        const long long t0 = (long long)chunk * g.ipw;
        const long long t1 = t0 + g.ipw < g.s.items ? t0 + g.ipw : g.s.items;
        Factor<FAM, T> own[K];
        double wl[K];
        lane_states<FAM, T, K>(g.s, tab, lg * kWave + (tid & (kWave - 1)), own, wl);
        acc = sum_items<FAM, T, K>(g.s, tab, own, wl, t0, t1);
    }
    double v;
    if (!sum_over_blocks(acc, A.sums, s_red, &v)) return;
    if (tid == 0) {
        double scale = A.c0;
        for (int k = 0; k < d; ++k) scale *= s_scale[k];
        const double r = scale_back(FAM, v, d, s_exp) * scale;
        if (A.out) *A.out = (T)r;
        if (A.out64) *A.out64 = r;
    }
}

// LDS of a two-axis loop table, of a two-axis outer table, and of all tables.
constexpr size_t kProductLoopLds = 40 * 1024;
constexpr size_t kProductOuterLds = 20 * 1024;
constexpr size_t kProductLdsMax = 60 * 1024;

// Plan; false: the grid does not take this kernel.
static bool plan_product(const tq_grid_desc* gd, int C, int tsize, ProductGeom& G) {
    const int d = gd->dim, n = gd->n;
    if (d < 3) return false;
    G.rule = gd->rule;
    double P = 1.0;
    for (int k = 0; k < d; ++k) P *= n;
    // States per lane (they share the LDS reads of the loop entries) where
    // the grid still fills the chip: 2 from 8.4e6 points, 4 from 3.4e7, 8 (FP32
    // only) from 1.3e8.  d=5 n=65: 34.5 us with 8, 36 with 4; d=4 n=65 (1.8e7
    // points): 12 us with 2, 14 with 4 and 8.
    const int kmax = tsize == 4 ? 8 : 4;
    G.K = 1;
    while (G.K < kmax && P >= (double)(4 * G.K * G.K) * (1 << 21)) G.K *= 2;
    const long long entry = (long long)C * tsize;
    const int lane_axes = gd->lane_axes > 0 ? (gd->lane_axes < d ? gd->lane_axes : d - 1) : 0;
    return split_product_axes(d, n, G.K, C, tsize, (long long)kProductLoopLds / entry,
                              G.K > 1 ? (long long)kProductOuterLds / entry : 0, lane_axes, kProductLdsMax, G.s);
}

// Splits the items over waves and the waves over blocks: one fill of the
// resident waves, but at least kLeastItems items (64 loop points) per wave, so
// that small grids do not pay for blocks whose waves have next to nothing to
// do (each block builds the tables and is counted at the end).
constexpr long long kLeastItems = 16;
// Table entries per block above which one block per CU is enough: each block
// evaluates them again, in FP64 (Simpson d=3 n=901: 34 us with two waves per
// SIMD, 39 with six).
constexpr int kManyFactors = 1024;

static void split_product(ProductGeom& G, long long items_per_wave, int waves_per_simd, int cus,
                          long long max_blocks) {
    long long ipw = items_per_wave > 0 ? (items_per_wave + kGroup - 1) / kGroup : 0;
    if (ipw <= 0) {
        const long long waves = 4LL * cus * waves_per_simd;
        long long per = waves / G.s.lane_groups;
        if (per < 1) per = 1;
        ipw = (G.s.items + per - 1) / per;
        if (ipw < kLeastItems) ipw = kLeastItems;
    }
    if (ipw > G.s.items) ipw = G.s.items;
    for (;; ipw *= 2) {
        G.ipw = ipw;
        G.num_waves = ((G.s.items + ipw - 1) / ipw) * (long long)G.s.lane_groups;
        G.blocks = (G.num_waves + kProductWaves - 1) / kProductWaves;
        if (G.blocks <= max_blocks || ipw >= G.s.items) return;
    }
}

template <typename T, int FAM>
static int launch_family(ProductGeom& G, ProductArgs<T>& A, hipStream_t st) {
    const size_t lds = product_lds_bytes(G.s, family_comps(FAM), (int)sizeof(T));
    A.g = G;
    const dim3 grid((unsigned)G.blocks), block(kProductWaves * kWave);
    switch (G.K) {
        case 1: hipLaunchKernelGGL((k_grid_product<T, FAM, 1>), grid, block, lds, st, A); break;
        case 2: hipLaunchKernelGGL((k_grid_product<T, FAM, 2>), grid, block, lds, st, A); break;
        case 4: hipLaunchKernelGGL((k_grid_product<T, FAM, 4>), grid, block, lds, st, A); break;
        default:
            if constexpr (sizeof(T) == 4) hipLaunchKernelGGL((k_grid_product<T, FAM, 8>), grid, block, lds, st, A);
            else return fail(TQ_E_ARG, "product plan with 8 FP64 states");
    }
    return check_launch("k_grid_product");
}

template <typename T>
int launch_grid_product(const tq_grid_desc* gd, const tq_integrand* f, const void* domain, void* ws,
                        size_t ws_bytes, void* out, double* out64, hipStream_t st, bool* taken) {
    *taken = false;
    ProductGeom G;
    const int cus = device_cus();
    if (cus <= 0 || !plan_product(gd, family_comps(f->family), (int)sizeof(T), G)) return TQ_OK;
    const bool many = family_comps(f->family) * G.s.d * G.s.n > kManyFactors;
    split_product(G, gd->items_per_wave, many ? 2 : product_waves_per_simd(f->family, (int)sizeof(T)), cus,
                  (long long)((ws_bytes - kWsHeader) / sizeof(double)));
    if (kWsHeader + (size_t)G.blocks * sizeof(double) > ws_bytes || G.num_waves > 0x7fffffffLL) return TQ_OK;
    *taken = true;
    ProductArgs<T> A;
    A.domain = (const T*)domain;
    A.glx = gd->gl_nodes;
    A.glw = gd->gl_weights;
    A.sums = block_sums(ws);
    A.out = (T*)out;
    A.out64 = out64;
    A.c0 = f->c0;
    A.p = make_params<T>(*f);
    TQ_DISPATCH_FAMILY(f->family, { return (launch_family<T, FAM>(G, A, st)); });
    return TQ_OK;
}

template int launch_grid_product<float>(const tq_grid_desc*, const tq_integrand*, const void*, void*, size_t, void*,
                                        double*, hipStream_t, bool*);
template int launch_grid_product<double>(const tq_grid_desc*, const tq_integrand*, const void*, void*, size_t, void*,
                                         double*, hipStream_t, bool*);

}  // namespace tq
