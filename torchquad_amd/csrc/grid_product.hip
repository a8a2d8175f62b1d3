// The fused grid kernel of integrals with at least two axes whose factor
// tables fit in LDS (tq_product.hpp says how values become products).
//
// Index space: the last m axes are spread over lanes, K combinations per
// lane (64 K per wave); the loop runs over one or two axes whose combined
// factors form an LDS table; the leading axes are rows, their factors merged
// into the lane's states once per row.  A wave owns one group of 64 K lane
// combinations and a contiguous range of (row, group of four loop points).
#include "tq_grid_launch.hpp"
#include "tq_product.hpp"

namespace tq {

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
    using F = Factor<FAM, T>;
    constexpr int C = F::C, nt = kProductWaves * kWave;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ Axis s_axis[TQ_MAX_DIM];
    __shared__ int s_top[TQ_MAX_DIM], s_exp[TQ_MAX_DIM];
    __shared__ double s_red[kProductWaves], s_scale[TQ_MAX_DIM];
    const ProductGeom& g = A.g;
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int d = g.d, n = g.n, L = g.L, total = d * n, entries = g.groups * kGroup;
    if (tid < d) {
        const Axis a = make_axis(A.domain, tid, n, g.rule);
        s_axis[tid] = a;
        s_scale[tid] = axis_scale_of(a, g.rule);
    }
    __syncthreads();
    T* axis = reinterpret_cast<T*>(smem_raw);
    unsigned char* second = smem_raw + (((size_t)C * total * sizeof(T) + 15) & ~(size_t)15);
    T* tab = reinterpret_cast<T*>(second);
    build_axis_factors<FAM, T>(d, n, g.rule, s_axis, A.glx, A.glw, A.p, g.by_n, axis,
                               reinterpret_cast<double*>(second), s_top, s_exp);
    // Loop table, over the FP64 copies (they are done with).  Four entries
    // per thread and trip: their reads go out together.
    for (int e0 = tid; e0 < entries; e0 += 4 * nt) {
        F f[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int e = e0 + i * nt;
            f[i] = F::one(false);
            if (e < g.nl) {
                if (g.q == 2) {
                    const int j1 = (int)g.by_n.div((uint32_t)e);
                    f[i] = F::merge(axis_factor<FAM, T>(axis, total, L * n + j1),
                                    axis_factor<FAM, T>(axis, total, (L + 1) * n + e - j1 * n));
                } else {
                    f[i] = axis_factor<FAM, T>(axis, total, L * n + e);
                }
                f[i] = f[i].dual();
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int c = 0; c < C; ++c)
                if (e0 + i * nt < entries) tab[c * entries + e0 + i * nt] = f[i].v[c];
    }
    __syncthreads();

    double acc = 0.0;
    const long long wave = (long long)blockIdx.x * kProductWaves + __builtin_amdgcn_readfirstlane(tid >> 6);
    if (wave < g.num_waves) {
        const unsigned uw = (unsigned)wave, ulg = (unsigned)g.lane_groups;
        const unsigned chunk = uw / ulg;
        const int lg = (int)(uw - chunk * ulg);
        const long long t0 = (long long)chunk * g.ipw;
        const long long t1 = t0 + g.ipw < g.items ? t0 + g.ipw : g.items;
        // the lane's K states over the lane axes; lanes past the last combination carry zeros
        F own[K];
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int slot = (lg * K + k) * kWave + lane;
            const bool on = slot < g.lane_count;
            uint32_t r = on ? (uint32_t)slot : 0u;
            own[k] = F::one(on);
            for (int a = d - 1; a >= d - g.m; --a) {
                const uint32_t q = g.by_n.div(r);
                own[k] = F::merge(own[k], axis_factor<FAM, T>(axis, total, a * n + (int)(r - q * g.by_n.n)));
                r = q;
            }
        }
        if (L == 0) {
            acc = sum_entries<FAM, T, K>(own, tab, entries, (int)t0, (int)t1);
        } else {
            // row odometer: lane k of `dig` holds the digit of row axis k
            long long row = t0 / g.groups;
            int gi = (int)(t0 - row * g.groups);
            int dig = 0;
            for (int k = L - 1; k >= 0; --k) {
                const long long q = row / n;
                dig = lane == k ? (int)(row - q * n) : dig;
                row = q;
            }
            for (long long t = t0; t < t1;) {
                F rf = F::one(true);
                for (int k = 0; k < L; ++k)
                    rf = F::merge(rf, axis_factor<FAM, T>(axis, total, k * n + __builtin_amdgcn_readlane(dig, k)));
                F s[K];
#pragma unroll
                for (int k = 0; k < K; ++k) s[k] = F::merge(own[k], rf);
                const int left = g.groups - gi;
                const int ge = t1 - t < left ? gi + (int)(t1 - t) : g.groups;
                acc += sum_entries<FAM, T, K>(s, tab, entries, gi, ge);
                t += ge - gi;
                gi = 0;
                for (int k = L - 1; k >= 0; --k) {
                    const int dk = __builtin_amdgcn_readlane(dig, k) + 1;
                    const bool wrap = dk >= n;
                    dig = lane == k ? (wrap ? 0 : dk) : dig;
                    if (!wrap) break;
                }
            }
        }
    }
    double v;
    if (!sum_over_blocks(acc, A.sums, s_red, &v)) return;
    if (tid == 0) {
        double scale = A.c0;
        int exponent = 0;
        for (int k = 0; k < d; ++k) {
            scale *= s_scale[k];
            exponent += s_exp[k];
        }
        const double r = ldexp(v, exponent) * scale;
        if (A.out) *A.out = (T)r;
        if (A.out64) *A.out64 = r;
    }
}

// LDS of a merged (two-axis) loop table, and of all tables.
constexpr size_t kProductLoopLds = 40 * 1024;
constexpr size_t kProductLdsMax = 60 * 1024;

// Plan; false: the grid does not take this kernel.
static bool plan_product(const tq_grid_desc* gd, int C, int tsize, int cus, ProductGeom& G) {
    const int d = gd->dim, n = gd->n;
    if (d < 3 || n < 2) return false;
    G.d = d;
    G.n = n;
    G.rule = gd->rule;
    G.by_n = make_fast_div((uint32_t)n);
    if ((size_t)C * d * n * (sizeof(double) + tsize) > kProductLdsMax) return false;
    double P = 1.0;
    for (int k = 0; k < d; ++k) P *= n;
    // States per lane (they share the LDS reads of the loop entries) where
    // the grid still fills the chip: 2 from 8.4e6 points, 4 from 3.4e7, 8 (FP32
    // only) from 1.3e8.  d=5 n=65: 34.5 us with 8, 36 with 4; d=4 n=65 (1.8e7
    // points): 12 us with 2, 14 with 4 and 8.
    const int kmax = tsize == 4 ? 8 : 4;
    G.K = 1;
    while (G.K < kmax && P >= (double)(4 * G.K * G.K) * (1 << 21)) G.K *= 2;
    // Loop axes: two when their table fits and a lane axis remains, so the
    // per-row work (state merges, FP64 flush) comes once per n^2 points.
    G.q = (d >= 3 && (size_t)C * ((size_t)n * n + kGroup) * tsize <= kProductLoopLds) ? 2 : 1;
    // Lane axes: the fewest that fill 95 % of the 64 K slots of their waves,
    // else the best filling count.
    const int mmax = d - G.q;
    int m = 1;
    if (gd->lane_axes > 0) {
        m = gd->lane_axes < d ? gd->lane_axes : d - 1;
        if (m > mmax) G.q = 1;
    } else {
        double best = -1.0, c = 1.0;
        for (int k = 1; k <= mmax; ++k) {
            c *= n;
            if (c > (double)(1 << 30)) break;
            const double slots = (double)kWave * G.K;
            const double fill = c / (std::ceil(c / slots) * slots);
            if (fill > best) {
                best = fill;
                m = k;
            }
            if (fill >= 0.95) break;
        }
    }
    G.m = m;
    G.L = d - m - G.q;
    long long lc;
    if (ipow_checked(n, m, 1LL << 30, &lc) != 0) return false;
    G.lane_count = (int)lc;
    G.lane_groups = (int)((lc + kWave * G.K - 1) / (kWave * G.K));
    G.nl = G.q == 2 ? n * n : n;
    G.groups = (G.nl + kGroup - 1) / kGroup;
    if (product_lds_bytes(G, C, tsize) > kProductLdsMax) return false;
    long long rows;
    if (ipow_checked(n, G.L, (1LL << 62) / G.groups, &rows) != 0) return false;
    G.items = rows * G.groups;
    return true;
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
        long long per = waves / G.lane_groups;
        if (per < 1) per = 1;
        ipw = (G.items + per - 1) / per;
        if (ipw < kLeastItems) ipw = kLeastItems;
    }
    if (ipw > G.items) ipw = G.items;
    for (;; ipw *= 2) {
        G.ipw = ipw;
        G.num_waves = ((G.items + ipw - 1) / ipw) * (long long)G.lane_groups;
        G.blocks = (G.num_waves + kProductWaves - 1) / kProductWaves;
        if (G.blocks <= max_blocks || ipw >= G.items) return;
    }
}

template <typename T, int FAM>
static int launch_family(ProductGeom& G, ProductArgs<T>& A, hipStream_t st) {
    const size_t lds = product_lds_bytes(G, family_comps(FAM), (int)sizeof(T));
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
    if (cus <= 0 || !plan_product(gd, family_comps(f->family), (int)sizeof(T), cus, G)) return TQ_OK;
    const bool many = family_comps(f->family) * G.d * G.n > kManyFactors;
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
