// Parameter sweeps from factor tables (tq_product.hpp): one integral per
// blockIdx.y, its blocks and waves sharing (lane group, range of items) units.
//
// Forward: as the fused grid kernel.  Backward of the Gaussian and product
// peaks: besides F = sum W f the gradients need, per axis k, three sums
// sum W f h_i(k, node) of per-axis functions (Gaussian peak: t, t^2, t r;
// product peak: t g, g, t g r).  A lane keeps F per state; row axes multiply
// a row's F by the row node's h_i, lane axes a state's F by its nodes' h_i
// once per lane group.  Only the loop axis needs sums over its points: since
// they do not tell the states apart, the lane's states are added once per row
// and the sum meets the tables of W h_i -- for the Gaussian peak of W r and
// W r^2, from which the three follow (t = alpha r + gamma on an axis).
//
// 1024 Gaussian peaks of 32^4 FP32 points: forward 122 -> 31 us, backward
// 332 -> 62 us against one exponential per point (grad.hip, which keeps one
// axis, axes too long for the tables and the oscillatory backward).
#include "tq_grid_launch.hpp"
#include "tq_product.hpp"
#include "tq_sweep.hpp"

namespace tq {

// Waves of a block: at most, and for integrals of P points.  A block builds its
// tables and sums its waves; small integrals in waves that have next to nothing
// to do paid for both (1000 Gaussian peaks of 14^3 FP32 points: forward 12.3
// us with eight waves, 10.1 with four; backward 30 and 15.5).
constexpr int kSweepBlockWaves = 8;
constexpr int kSweepThreads = kSweepBlockWaves * kWave;
static int sweep_block_waves(long long P) { return P <= 1024 ? 1 : P <= 2048 ? 2 : P <= 4096 ? 4 : kSweepBlockWaves; }
constexpr size_t kSweepLdsMax = 60 * 1024;
// States per lane: the backward reads a loop entry's three or four tables per
// point from LDS, which eight FP32 states share.
template <typename T>
constexpr int kSweepStates = sizeof(T) == 4 ? 8 : 4;

// Units of one integral: every lane group, its items cut into `parts`.
struct SweepUnits {
    ProductSplit s;
    int rule;
    int parts;
    int block_waves;
    long long per;  // items per part
};

static bool plan_sweep_product(const tq_grid_desc* g, int C, int tsize, bool backward, long long blocks, SweepUnits& U) {
    const int d = g->dim, n = g->n, K = tsize == 4 ? 8 : 4;
    if (d < 2 || n < 2 || (long long)d * n > 8192) return false;
    // the backward's node tables (t, g and r) and moment tables beside the split's own
    const size_t extra = backward ? (size_t)(2 * d * n + n + 3 * (n + kGroup)) * tsize + 64 : 0;
    if (extra >= kSweepLdsMax) return false;
    const long long entries = backward ? n + kGroup : 8192 / ((long long)C * tsize);
    const int lane_axes = g->lane_axes > 0 ? (g->lane_axes < d ? g->lane_axes : d - 1) : 0;
    if (!split_product_axes(d, n, K, C, tsize, entries < n + kGroup ? n + kGroup : entries, 256, lane_axes,
                            kSweepLdsMax - extra, U.s, backward ? 1 : 2))
        return false;
    U.rule = g->rule;
    long long P;
    ipow_checked(n, d, 1LL << 62, &P);
    U.block_waves = sweep_block_waves(P);
    const long long waves = blocks * U.block_waves;
    long long parts = waves / U.s.lane_groups;
    if (parts < 1) parts = 1;
    if (parts > U.s.items) parts = U.s.items;
    U.per = (U.s.items + parts - 1) / parts;
    U.parts = (int)((U.s.items + U.per - 1) / U.per);
    return true;
}

// About 8192 waves (8 per SIMD) over the whole sweep, each with at least 4096
// points, and at most 256 blocks per integral (its final sum walks them).
long long sweep_product_blocks(const tq_grid_desc* g, int64_t B) {
    SweepUnits U;
    // the largest tables any family and direction needs
    const int tsize = g->dtype == TQ_F32 ? 4 : 8;
    if (!plan_sweep_product(g, 2, tsize, false, 1, U) || !plan_sweep_product(g, 1, tsize, true, 1, U)) return 0;
    if (g->items_per_wave > 0) return 0;  // a fixed split of the general kernels' items
    long long P;
    ipow_checked(g->n, g->dim, 1LL << 62, &P);
    long long waves = B > 0 ? (8192 + B - 1) / B : 8192;
    if (waves > P / 4096) waves = P / 4096;
    long long blocks = (waves + kSweepBlockWaves - 1) / kSweepBlockWaves;
    if (blocks < 1) blocks = 1;
    return blocks > 256 ? 256 : blocks;
}

template <typename T, int FAM, int K>
__global__ __launch_bounds__(kSweepThreads) void k_sweep_product_fwd(SweepUnits U, const T* a, const T* u,
                                                                     const T* dom, const double* glx,
                                                                     const double* glw, double* partials) {
    extern __shared__ __align__(16) unsigned char s_lds[];
    __shared__ Params<T> s_p;
    __shared__ Axis s_axis[TQ_MAX_DIM];
    __shared__ int s_exp[kExpSlots];
    __shared__ double s_red[kSweepBlockWaves];
    const ProductSplit& S = U.s;
    const long long b = blockIdx.y;
    const int tid = threadIdx.x;
    load_sweep_params<T, FAM>(S.d, S.n, U.rule, b, a, u, dom, &s_p, s_axis);
    __syncthreads();
    const ProductTables<T> tab = build_product_tables<FAM, T>(S, U.rule, s_axis, glx, glw, s_p, s_lds, s_exp);
    const int units = S.lane_groups * U.parts, waves = gridDim.x * U.block_waves;
    double acc = 0.0;
    Factor<FAM, T> own[K];
    double wl[K];
    for (int w = blockIdx.x * U.block_waves + __builtin_amdgcn_readfirstlane(tid >> 6); w < units; w += waves) {
        const int lg = w / U.parts, part = w - lg * U.parts;
        const long long t0 = part * U.per, t1 = t0 + U.per < S.items ? t0 + U.per : S.items;
        lane_states<FAM, T, K>(S, tab, lg * kWave + (tid & (kWave - 1)), own, wl);
        acc += sum_items<FAM, T, K>(S, tab, own, wl, t0, t1);
    }
    acc = block_sum(acc, s_red);
    if (tid == 0) partials[b * gridDim.x + blockIdx.x] = scale_back(FAM, acc, S.d, s_exp);
}

// Loop-axis sums kept beside F.
constexpr int sweep_moments(int fam) { return fam == TQ_FAM_GAUSSIAN_PEAK ? 2 : 3; }

// The per-axis functions at a node: t = x - u (rounded to T as the nodes
// are), g = 1 / (a^-2 + t^2) (product peak) and the normalised node r.
template <int FAM>
__device__ inline void sweep_functions(double t, double g, double r, double* h) {
    if constexpr (FAM == TQ_FAM_GAUSSIAN_PEAK) {
        h[0] = t;
        h[1] = t * t;
        h[2] = t * r;
    } else {
        h[0] = t * g;
        h[1] = g;
        h[2] = t * g * r;
    }
}

// partial layout per (integral, block): [F, h_0 sums of the D axes, h_1 .., h_2 ..]
template <typename T, int FAM, int K, int D>
__global__ __launch_bounds__(kSweepThreads) void k_sweep_product_bwd(SweepUnits U, const T* a, const T* u,
                                                                     const T* dom, const double* glx,
                                                                     const double* glw, double* partials) {
    using F = Factor<FAM, T>;
    constexpr int NM = sweep_moments(FAM);
    extern __shared__ __align__(16) unsigned char s_lds[];
    __shared__ Params<T> s_p;
    __shared__ Axis s_axis[TQ_MAX_DIM];
    __shared__ int s_exp[kExpSlots];
    const ProductSplit& S = U.s;
    const int n = S.n, L = S.L, groups = S.groups, entries = groups * kGroup;
    const long long b = blockIdx.y;
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    // not blockDim.x, with which the kernel holds 25 more registers (D = 4
    // product peak, FP32: 134 against 107, three waves per SIMD in place of four)
    const int stride = U.block_waves * kWave;
    load_sweep_params<T, FAM>(D, n, U.rule, b, a, u, dom, &s_p, s_axis);
    __syncthreads();
    // node tables and the loop axis's moment tables, after the split's own tables
    T* mom = reinterpret_cast<T*>(s_lds + round16(product_lds_bytes(S, 1, (int)sizeof(T))));
    T* s_t = mom + NM * entries;
    T* s_g = s_t + D * n;
    T* s_r = s_g + (FAM == TQ_FAM_PRODUCT_PEAK ? D * n : 0);
    for (int e = tid; e < D * n; e += stride) {
        const int k = (int)S.by_n.div((uint32_t)e), j = e - k * n;
        const T t = (T)node_of(s_axis[k], j, n, U.rule, glx) - s_p.u[k];
        s_t[e] = t;
        if (FAM == TQ_FAM_PRODUCT_PEAK) s_g[e] = (T)(1.0 / fma((double)t, (double)t, (double)s_p.b[k]));
        if (k == 0) s_r[j] = (T)node_r(j, n, U.rule, glx);
    }
    const ProductTables<T> tab = build_product_tables<FAM, T, false>(S, U.rule, s_axis, glx, glw, s_p, s_lds, s_exp);
    auto functions = [&](int k, int j, double* h) {
        sweep_functions<FAM>((double)s_t[k * n + j], FAM == TQ_FAM_PRODUCT_PEAK ? (double)s_g[k * n + j] : 0.0,
                             (double)s_r[j], h);
    };
    for (int e = tid; e < entries; e += stride) {
        double h[3] = {0.0, 0.0, 0.0};
        const double v = (double)tab.loop[e];  // zero past the last node
        const int j = e < n ? e : 0;
        if (FAM == TQ_FAM_GAUSSIAN_PEAK) {
            h[0] = (double)s_r[j];
            h[1] = h[0] * h[0];
        } else {
            functions(L, j, h);
        }
#pragma unroll
        for (int i = 0; i < NM; ++i) mom[i * entries + e] = (T)(v * h[i]);
    }
    __syncthreads();
    double accF = 0.0, acc[3][D], M[NM];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int k = 0; k < D; ++k) acc[i][k] = 0.0;
#pragma unroll
    for (int i = 0; i < NM; ++i) M[i] = 0.0;
    // acc of axis k (selected over the compile-time axes, so it stays in registers)
    auto add = [&](int axis, const double* h, double f) {
#pragma unroll
        for (int k = 0; k < D; ++k) {
            const double fk = k == axis ? f : 0.0;
#pragma unroll
            for (int i = 0; i < 3; ++i) acc[i][k] = fma(h[i], fk, acc[i][k]);
        }
    };
    const int units = S.lane_groups * U.parts, waves = gridDim.x * U.block_waves;
    for (int w = blockIdx.x * U.block_waves + __builtin_amdgcn_readfirstlane(tid >> 6); w < units; w += waves) {
        const int lg = w / U.parts, part = w - lg * U.parts;
        const long long t0 = part * U.per, t1 = t0 + U.per < S.items ? t0 + U.per : S.items;
        const int slot = lg * kWave + lane;
        F own[K];
        lane_states<FAM, T, K>(S, tab, slot, own, nullptr);
        double Fk[K];
#pragma unroll
        for (int k = 0; k < K; ++k) Fk[k] = 0.0;
        // row odometer: lane k of `dig` holds the digit of row axis k
        long long row = t0 / groups;
        int gi = (int)(t0 - row * groups);
        int dig = 0;
        for (int k = L - 1; k >= 0; --k) {
            const long long q = row / n;
            dig = lane == k ? (int)(row - q * n) : dig;
            row = q;
        }
        for (long long at = t0; at < t1;) {
            F rf = F::one(true);
            for (int k = 0; k < L; ++k)
                rf = F::merge(rf, axis_factor<FAM, T>(tab.axis, D * n, k * n + __builtin_amdgcn_readlane(dig, k)));
            T s[K];
#pragma unroll
            for (int k = 0; k < K; ++k) s[k] = own[k].v[0] * rf.v[0];
            const T all = (T)join_states<T, K>(s);
            const int left = groups - gi;
            const int ge = t1 - at < left ? gi + (int)(t1 - at) : groups;
            double Frow = 0.0;
            constexpr int kFlushGroups = kFlush / kGroup;
            for (int gb = gi; gb < ge; gb += kFlushGroups) {
                const int gend = gb + kFlushGroups < ge ? gb + kFlushGroups : ge;
                T fa[K];
#pragma unroll
                for (int k = 0; k < K; ++k) fa[k] = T(0);
                // the moments' FP32 partials stand for K points per entry
                constexpr int kMomentGroups = sizeof(T) == 4 ? kFlushGroups / K : kFlushGroups;
                for (int gm = gb; gm < gend; gm += kMomentGroups) {
                    const int gmend = gm + kMomentGroups < gend ? gm + kMomentGroups : gend;
                    T fm[NM];
#pragma unroll
                    for (int i = 0; i < NM; ++i) fm[i] = T(0);
                    for (int gq = gm; gq < gmend; ++gq) {
                        EntryGroup<TQ_FAM_CONSTANT, T> e, em[NM];
                        e.load(tab.loop, entries, gq);
#pragma unroll
                        for (int i = 0; i < NM; ++i) em[i].load(mom + i * entries, entries, gq);
#pragma unroll
                        for (int x = 0; x < kGroup; ++x) {
#pragma unroll
                            for (int k = 0; k < K; ++k) fa[k] = fma(s[k], e.v[0][x], fa[k]);
#pragma unroll
                            for (int i = 0; i < NM; ++i) fm[i] = fma(all, em[i].v[0][x], fm[i]);
                        }
                    }
#pragma unroll
                    for (int i = 0; i < NM; ++i) M[i] += (double)fm[i];
                }
#pragma unroll
                for (int k = 0; k < K; ++k) Fk[k] += (double)fa[k];
                Frow += join_states<T, K>(fa);
            }
            accF += Frow;
            // row axes: uniform nodes
#pragma unroll
            for (int k = 0; k < D - 1; ++k) {
                if (k < L) {
                    double h[3];
                    functions(k, __builtin_amdgcn_readlane(dig, k), h);
#pragma unroll
                    for (int i = 0; i < 3; ++i) acc[i][k] = fma(h[i], Frow, acc[i][k]);
                }
            }
            at += ge - gi;
            gi = 0;
            for (int k = L - 1; k >= 0; --k) {
                const int dk = __builtin_amdgcn_readlane(dig, k) + 1;
                const bool wrap = dk >= n;
                dig = lane == k ? (wrap ? 0 : dk) : dig;
                if (!wrap) break;
            }
        }
        // lane axes: the slot's inner nodes with the states' sum, the outer ones state by state
        double Fl = 0.0;
#pragma unroll
        for (int k = 0; k < K; ++k) Fl += Fk[k];
        uint32_t r = slot < S.slots ? (uint32_t)slot : 0u;
        for (int ax = D - 1; ax >= D - S.inner; --ax) {
            const uint32_t q = S.by_n.div(r);
            double h[3];
            functions(ax, (int)(r - q * S.by_n.n), h);
            add(ax, h, Fl);
            r = q;
        }
        const int o0 = L + S.q;
        double sum[2][3] = {{0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}};
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int f = (int)r + k * S.H < S.N ? (int)r + k * S.H : 0;  // states without a combination have Fk 0
            const int j1 = S.outer == 2 ? (int)S.by_n.div((uint32_t)f) : f;
            double h[3];
            functions(o0, j1, h);
#pragma unroll
            for (int i = 0; i < 3; ++i) sum[0][i] = fma(h[i], Fk[k], sum[0][i]);
            if (S.outer == 2) {
                functions(o0 + 1, f - j1 * n, h);
#pragma unroll
                for (int i = 0; i < 3; ++i) sum[1][i] = fma(h[i], Fk[k], sum[1][i]);
            }
        }
        add(o0, sum[0], 1.0);
        if (S.outer == 2) add(o0 + 1, sum[1], 1.0);
    }
    // loop axis
    if (FAM == TQ_FAM_GAUSSIAN_PEAK) {
        double alpha, beta;
        loop_axis_affine(s_axis[L], n, U.rule, &alpha, &beta);
        const double gam = beta - (double)s_p.u[L];
        const double h[3] = {alpha * M[0] + gam * accF, alpha * alpha * M[1] + 2.0 * alpha * gam * M[0] + gam * gam * accF,
                             alpha * M[1] + gam * M[0]};
        add(L, h, 1.0);
    } else {
        const double h[3] = {M[0], M[1], M[NM - 1]};
        add(L, h, 1.0);
    }
    // the waves' sums meet in LDS once, then a thread adds each value's (block sums one after the other: two barriers
    // and twelve LDS permutes for each of the 1 + 3 D)
    constexpr int V = 1 + 3 * D;
    __shared__ double s_sum[kSweepBlockWaves][V];
    const int wb = __builtin_amdgcn_readfirstlane(tid >> 6);
    auto put = [&](int i, double x) {
        x = wave_sum_last(x);
        if (lane == kWave - 1) s_sum[wb][i] = x;
    };
    put(0, accF);
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int k = 0; k < D; ++k) put(1 + i * D + k, acc[i][k]);
    __syncthreads();
    if (tid < V) {
        double x = 0.0;
        for (int q = 0; q < U.block_waves; ++q) x += s_sum[q][tid];
        partials[(b * gridDim.x + blockIdx.x) * V + tid] = scale_by(x, sum_exponents(s_exp));
    }
}

template <typename T, int FAM>
int launch_sweep_product_fwd(const tq_grid_desc* g, int64_t B, const void* a, const void* u, const void* dom,
                             double* partials, long long blocks, hipStream_t s) {
    SweepUnits U;
    const int C = family_comps(FAM);
    if (!plan_sweep_product(g, C, (int)sizeof(T), false, blocks, U)) return fail(TQ_E_ARG, "no product plan for the sweep");
    hipLaunchKernelGGL((k_sweep_product_fwd<T, FAM, kSweepStates<T>>), dim3((unsigned)blocks, (unsigned)B),
                       dim3(U.block_waves * kWave), product_lds_bytes(U.s, C, (int)sizeof(T)), s, U, (const T*)a, (const T*)u,
                       (const T*)dom, g->gl_nodes, g->gl_weights, partials);
    return check_launch("k_sweep_product_fwd");
}

template <typename T, int FAM, int D>
static void launch_bwd(const SweepUnits& U, const tq_grid_desc* g, int64_t B, const void* a, const void* u,
                       const void* dom, double* partials, long long blocks, hipStream_t s) {
    const int n = g->n, entries = U.s.groups * kGroup;
    const size_t lds = product_lds_bytes(U.s, 1, (int)sizeof(T)) + 16 +
                       ((size_t)sweep_moments(FAM) * entries + (size_t)2 * D * n + n) * sizeof(T);
    hipLaunchKernelGGL((k_sweep_product_bwd<T, FAM, kSweepStates<T>, D>), dim3((unsigned)blocks, (unsigned)B),
                       dim3(U.block_waves * kWave), lds, s, U, (const T*)a, (const T*)u, (const T*)dom, g->gl_nodes,
                       g->gl_weights, partials);
}

template <typename T, int FAM>
int launch_sweep_product_bwd(const tq_grid_desc* g, int64_t B, const void* a, const void* u, const void* dom,
                             double* partials, long long blocks, hipStream_t s) {
    SweepUnits U;
    if (!plan_sweep_product(g, 1, (int)sizeof(T), true, blocks, U)) return fail(TQ_E_ARG, "no product plan for the sweep");
    switch (g->dim) {
        case 2: launch_bwd<T, FAM, 2>(U, g, B, a, u, dom, partials, blocks, s); break;
        case 3: launch_bwd<T, FAM, 3>(U, g, B, a, u, dom, partials, blocks, s); break;
        case 4: launch_bwd<T, FAM, 4>(U, g, B, a, u, dom, partials, blocks, s); break;
        case 5: launch_bwd<T, FAM, 5>(U, g, B, a, u, dom, partials, blocks, s); break;
        case 6: launch_bwd<T, FAM, 6>(U, g, B, a, u, dom, partials, blocks, s); break;
        case 7: launch_bwd<T, FAM, 7>(U, g, B, a, u, dom, partials, blocks, s); break;
        default: launch_bwd<T, FAM, 8>(U, g, B, a, u, dom, partials, blocks, s); break;
    }
    return check_launch("k_sweep_product_bwd");
}

#define TQ_SWEEP_INST(T, FAM)                                                                                      \
    template int launch_sweep_product_fwd<T, FAM>(const tq_grid_desc*, int64_t, const void*, const void*,          \
                                                  const void*, double*, long long, hipStream_t);
TQ_SWEEP_INST(float, TQ_FAM_GAUSSIAN_PEAK)
TQ_SWEEP_INST(float, TQ_FAM_OSCILLATORY)
TQ_SWEEP_INST(float, TQ_FAM_PRODUCT_PEAK)
TQ_SWEEP_INST(double, TQ_FAM_GAUSSIAN_PEAK)
TQ_SWEEP_INST(double, TQ_FAM_OSCILLATORY)
TQ_SWEEP_INST(double, TQ_FAM_PRODUCT_PEAK)
#undef TQ_SWEEP_INST
#define TQ_SWEEP_INST(T, FAM)                                                                                      \
    template int launch_sweep_product_bwd<T, FAM>(const tq_grid_desc*, int64_t, const void*, const void*,          \
                                                  const void*, double*, long long, hipStream_t);
TQ_SWEEP_INST(float, TQ_FAM_GAUSSIAN_PEAK)
TQ_SWEEP_INST(float, TQ_FAM_PRODUCT_PEAK)
TQ_SWEEP_INST(double, TQ_FAM_GAUSSIAN_PEAK)
TQ_SWEEP_INST(double, TQ_FAM_PRODUCT_PEAK)
#undef TQ_SWEEP_INST

}  // namespace tq
