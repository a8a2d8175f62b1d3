// Tensor-product grid rules (Trapezoid, Simpson, Boole, Gauss-Legendre):
// the point-by-point fused kernel, which integrals of one or two axes and of
// axes too long for grid_product.hip's tables take (that kernel needs every
// axis's factors in FP64 first, which pays from three axes on; two axes here
// and there, Gaussian peak, trapezoid: FP32 n=101 7.4 and 7.4 us, n=1001 10.0
// and 12.2, n=2001 12.6 and 17.3; FP64 n=101 8.3 and 7.5, n=1001 11.9 and
// 12.1, n=2001 16.6 and 16.8; FP32 axes of more than 2048 nodes, which have no
// loop table here, are the exception: n=3001 47 and 22), and the kernels of
// user integrands.
//
// Index space.  The n^d grid points (ij order, last axis fastest, as
// IntegrationGrid.points in integration_grid.py:98-99) are split into
//   * lane axes  [d-m, d): one combination per lane, fixed for the lane's
//     lifetime (its partial fold and weight are computed once);
//   * loop axis  L = d-m-1: wave-uniform, iterated in the hot loop with its
//     nodes and weights read from an LDS table (broadcast reads);
//   * row axes   [0, L): wave-uniform, advanced by an odometer once per row.
// A wave owns one group of 64 lane combinations and a contiguous range of
// (row, loop-index) items.  Per point the kernel does: fold of the loop axis
// into the shared row+lane partial, the family's finish (transcendental),
// and one FMA into an FP32 partial that is flushed to FP64 at least every 128 points.
// Block partials are FP64 and the final sum runs in a fixed order, so the
// result is deterministic.
#include <mutex>

#include "tq_host.hpp"
#include "tq_grid_launch.hpp"
#include "tq_grid_tile.hpp"
#include "tq_values.hpp"

namespace tq {

constexpr int kMaxDimPoints = 64;  // point writer / weighted reduce

template <typename T>
struct GridArgs {
    GridGeom g;
    const T* domain;
    const double* glx;
    const double* glw;
    BlockSums sums;
    T* out;
    double* out64;
    double c0;
    Params<T> p;
};

static int check_grid_desc(const tq_grid_desc* g, int max_dim) {
    if (!g) return fail(TQ_E_NULL, "grid descriptor is NULL");
    if (g->dtype != TQ_F32 && g->dtype != TQ_F64) return fail(TQ_E_ARG, "dtype must be TQ_F32 or TQ_F64");
    if (g->dim < 1 || g->dim > max_dim) return fail(TQ_E_ARG, "grid dim out of range");
    switch (g->rule) {
        case TQ_RULE_TRAPEZOID:
            if (g->n < 2) return fail(TQ_E_ARG, "Trapezoid needs n >= 2 points per axis");
            break;
        case TQ_RULE_SIMPSON:
            if (g->n < 3 || (g->n % 2) != 1) return fail(TQ_E_ARG, "Simpson needs odd n >= 3");
            break;
        case TQ_RULE_BOOLE:
            if (g->n < 5 || ((g->n - 1) % 4) != 0) return fail(TQ_E_ARG, "Boole needs n = 1 + 4k >= 5");
            break;
        case TQ_RULE_GAUSS_LEGENDRE:
            if (g->n < 1) return fail(TQ_E_ARG, "Gauss-Legendre needs n >= 1");
            break;
        default: return fail(TQ_E_ARG, "unknown rule");
    }
    long long P;
    if (ipow_checked(g->n, g->dim, (1LL << 62), &P) != 0) return fail(TQ_E_ARG, "n^dim exceeds 2^62 points");
    return TQ_OK;
}

// Gauss-Legendre node/weight tables are needed wherever nodes or weights
// are formed (everything except unit-weight reductions).
static int check_gl_tables(const tq_grid_desc* g) {
    if (g->rule == TQ_RULE_GAUSS_LEGENDRE && (!g->gl_nodes || !g->gl_weights))
        return fail(TQ_E_NULL, "Gauss-Legendre needs node/weight tables");
    return TQ_OK;
}

// The point-by-point kernel's plan, which workspaces are sized by; the product
// kernel keeps its workgroups within the workspace it is given.
static int make_geom(const tq_grid_desc* gd, GridGeom& G) {
    return plan_geom(gd->dim, gd->n, gd->rule, gd->lane_axes, gd->items_per_wave, 16384, G);
}

// ---------------------------------------------------------------------------
// Fused kernel
// ---------------------------------------------------------------------------
// Dynamic LDS of the fused kernel: [row weights: L*n FP64][loop table:
// S*nl T][row contributions: slots*L*n T] (the row parts only when ROWTAB).
template <typename T, int FAM>
inline size_t fused_lds_bytes(const GridGeom& G, bool rowtab) {
    size_t b = (size_t)TabStride<FAM>::v * G.nl * sizeof(T);
    if (rowtab) b += (size_t)G.L * G.n * (sizeof(double) + StateSlots<FAM>::v * sizeof(T));
    return b;
}
constexpr size_t kFusedLdsMax = 48 * 1024;

// BW waves per block: 4, or 8 when a large loop table is shared by more
// waves (the LDS per block, not the registers, then bounds occupancy).
template <typename T, int FAM, bool TABLE, bool ROWTAB, int BW>
__global__ __launch_bounds__(BW * kWave) void k_grid_fused(GridArgs<T> A) {
    constexpr int NT = BW * kWave;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ Axis s_axis[TQ_MAX_DIM];
    __shared__ double s_red[BW];
    const GridGeom& g = A.g;
    const int tid = threadIdx.x;
    const int n = g.n, d = g.d, L = g.L, rule = g.rule;
    if (tid < d) s_axis[tid] = make_axis(A.domain, tid, n, rule);
    __syncthreads();
    double* s_rw = reinterpret_cast<double*>(smem_raw);
    T* s_tab = reinterpret_cast<T*>(smem_raw + (ROWTAB ? (size_t)L * n * sizeof(double) : 0));
    T* s_rt = s_tab + (size_t)TabStride<FAM>::v * g.nl;
    if (TABLE) {
        for (int j = tid; j < g.nl; j += NT)
            loop_table_entry<T, FAM>(s_tab, j, s_axis, L, n, rule, A.glx, A.glw, A.p);
        if (ROWTAB)
            for (int e = tid; e < L * n; e += NT) {
                const int k = e / n;
                row_table_entry<T, FAM>(s_rt, s_rw, k, e - k * n, s_axis[k], axis_c(A.p, k), n, rule, A.glx, A.glw,
                                        A.p);
            }
        __syncthreads();
    }
    // readfirstlane: the wave index is uniform, so the tile loop runs on SGPRs
    const long long wave = (long long)blockIdx.x * BW + __builtin_amdgcn_readfirstlane(tid >> 6);
    double acc = 0.0;
    if (wave < g.num_waves) {
        // wave < 2^31 (grid size limit): 32-bit division
        const unsigned uw = (unsigned)wave, ulw = (unsigned)g.lane_waves;
        const unsigned chunk = uw / ulw;
        const int lw = (int)(uw - chunk * ulw);
        const long long t0 = (long long)chunk * g.ipw;
        const long long t1 = (t0 + g.ipw < g.items) ? (t0 + g.ipw) : g.items;
        acc = grid_tile<T, FAM, TABLE, ROWTAB>(d, n, g.nl, g.m, L, rule, g.lane_count, A.p, s_axis, s_tab, A.glx,
                                               A.glw, lw, t0, t1, s_rt, s_rw);
    }
    double v;
    if (!sum_over_blocks(acc, A.sums, s_red, &v)) return;
    if (tid == 0) {
        double scale = A.c0;
        for (int k = 0; k < d; ++k)
            scale *= axis_scale((double)A.domain[2 * k], (double)A.domain[2 * k + 1], n, rule);
        const double r = v * scale;
        if (A.out) *A.out = (T)r;
        if (A.out64) *A.out64 = r;
    }
}

// Blocks of `kernel` (`threads` per block, `shmem` bytes of dynamic LDS)
// that stay resident on the current device at once, and the device's CU
// count; 0 if unknown.  Answers are kept per thread for the last few
// (device, kernel, shmem) keys, since the runtime query costs more than a
// small launch.
static long long resident_blocks(const void* kernel, int threads, size_t shmem, int* cus_out) {
    struct Entry {
        int dev;
        const void* kernel;
        size_t shmem;
        long long blocks;
        int cus;
    };
    constexpr int kEntries = 16;
    thread_local Entry cache[kEntries] = {};
    thread_local int next = 0;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    for (const Entry& e : cache)
        if (e.kernel == kernel && e.dev == dev && e.shmem == shmem) {
            *cus_out = e.cus;
            return e.blocks;
        }
    int cus = 0, per_cu = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, threads, shmem) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    const long long r = (long long)cus * per_cu;
    cache[next] = Entry{dev, kernel, shmem, r, cus};
    next = (next + 1) % kEntries;
    *cus_out = cus;
    return r;
}

// Workspace of the fused kernel, in block partials: at least this many, so
// that the automatic items per wave below can fill whole rounds.
constexpr long long kFusedMinBlocks = 8192;

// Launch-time model behind the automatic items per wave, fitted to the FP32
// Boole Gaussian-peak kernel on MI355X (d = 3..6, n = 17..129, items per
// wave 16..4096): a launch takes about
//   blocks x kBlockNs  (each workgroup's completion fence and counter, which
//                       the device serialises: 10112 workgroups of 16-item
//                       waves took 112 us for 3.9e7 evaluations)
//   + sum over rounds of ipw x kItemNs x (w + kItemLatency)
// where a round is one fill of the W resident waves and w its waves per
// SIMD: a wave's item (64 points) takes kItemNs (w + kItemLatency) when w
// waves share the SIMD -- latency-bound alone, issue-bound with many.
constexpr double kBlockNs = 10.0;
constexpr double kItemNs = 5.6;
constexpr double kItemLatency = 1.28;

// Relative time per item of a family and dtype (FP64 transcendentals are
// software sequences; the oscillatory cosine is a polynomial).
inline double item_scale(int fam, int tsize) {
    double s = fam == TQ_FAM_OSCILLATORY ? 1.5 : (fam == TQ_FAM_DOUBLE_GAUSSIAN ? 2.0 : 1.0);
    return tsize == 8 ? 6.0 * s : s;
}

// Automatic items per wave for a launch of `kernel`: the candidate with the
// least modelled time -- the counts that fill r = 1..16 resident rounds (each
// lane wave's items cut into floor(r W / lane_waves) chunks) and the powers
// of two up to the item count.  Keeps G as it is when the occupancy is unknown.
static void align_ipw(GridGeom& G, const void* kernel, int bw, size_t shmem, long long max_blocks, double scale) {
    int cus = 0;
    const long long W = resident_blocks(kernel, bw * kWave, shmem, &cus) * bw;
    if (W <= 0 || cus <= 0 || G.items <= 0) return;
    const double simds = 4.0 * cus;
    const double item_ns = kItemNs * scale;
    double best_t = -1.0;
    long long best_ipw = G.ipw;
    auto consider = [&](long long ipw) {
        if (ipw < 1) ipw = 1;
        if (ipw > G.items) ipw = G.items;
        const long long waves = ((G.items + ipw - 1) / ipw) * (long long)G.lane_waves;
        const long long blocks = (waves + bw - 1) / bw;
        if (blocks > max_blocks) return;
        const long long full = waves / W, rest = waves % W;
        double t = kBlockNs * (double)blocks + (double)full * (double)ipw * item_ns * ((double)W / simds + kItemLatency);
        if (rest > 0) t += (double)ipw * item_ns * ((double)rest / simds + kItemLatency);
        if (best_t < 0.0 || t < best_t) {
            best_t = t;
            best_ipw = ipw;
        }
    };
    for (long long r = 1; r <= 16; ++r) {
        long long per_lw = (r * W) / G.lane_waves;
        if (per_lw < 1) per_lw = 1;
        consider((G.items + per_lw - 1) / per_lw);
    }
    for (long long p = 16; p < G.items; p *= 2) consider(p);
    consider(G.items);
    G.ipw = best_ipw;
    G.chunks = (G.items + best_ipw - 1) / best_ipw;
    G.num_waves = G.chunks * (long long)G.lane_waves;
}

// Dynamic LDS above which 8-wave blocks share the tables.
constexpr size_t kWideBlockLds = 16 * 1024;

template <typename T, int FAM, bool TABLE, bool ROWTAB, int BW>
static void launch_fused(GridGeom& G, GridArgs<T>& A, size_t shmem, bool auto_ipw, long long max_blocks,
                         hipStream_t st) {
    const void* kern = (const void*)(k_grid_fused<T, FAM, TABLE, ROWTAB, BW>);
    if (auto_ipw) align_ipw(G, kern, BW, shmem, max_blocks, item_scale(FAM, (int)sizeof(T)));
    G.blocks = (G.num_waves + BW - 1) / BW;
    A.g = G;
    hipLaunchKernelGGL((k_grid_fused<T, FAM, TABLE, ROWTAB, BW>), dim3((unsigned)G.blocks), dim3(BW * kWave), shmem,
                       st, A);
}

template <typename T>
static int launch_grid(const tq_grid_desc* gd, const tq_integrand* f, const void* domain,
                       void* ws, size_t ws_bytes, void* out, double* out64, hipStream_t st) {
    GridGeom G;
    int rc = make_geom(gd, G);
    if (rc) return rc;
    const size_t need = kWsHeader + (size_t)G.blocks * sizeof(double);
    if (!ws || ws_bytes < need) return fail(TQ_E_WORKSPACE, "grid workspace too small");
    bool taken = false;
    rc = launch_grid_product<T>(gd, f, domain, ws, ws_bytes, out, out64, st, &taken);
    if (rc || taken) return rc;
    GridArgs<T> A;
    A.g = G;
    A.domain = (const T*)domain;
    A.glx = gd->gl_nodes;
    A.glw = gd->gl_weights;
    A.sums = block_sums(ws);
    A.out = (T*)out;
    A.out64 = out64;
    A.c0 = f->c0;
    A.p = make_params<T>(*f);
    const bool auto_ipw = gd->items_per_wave <= 0;
    const long long max_blocks = (long long)((ws_bytes - kWsHeader) / sizeof(double));
    TQ_DISPATCH_FAMILY(f->family, {
        const bool rowtab = G.use_table && G.L >= 1 && (fused_lds_bytes<T, FAM>(G, true)) <= kFusedLdsMax;
        const size_t shmem = (fused_lds_bytes<T, FAM>(G, rowtab));
        const bool wide = shmem > kWideBlockLds;
        if (rowtab && wide)
            (launch_fused<T, FAM, true, true, 8>)(G, A, shmem, auto_ipw, max_blocks, st);
        else if (rowtab)
            (launch_fused<T, FAM, true, true, kWavesPerBlock>)(G, A, shmem, auto_ipw, max_blocks, st);
        else if (G.use_table && wide)
            (launch_fused<T, FAM, true, false, 8>)(G, A, shmem, auto_ipw, max_blocks, st);
        else if (G.use_table)
            (launch_fused<T, FAM, true, false, kWavesPerBlock>)(G, A, shmem, auto_ipw, max_blocks, st);
        else
            (launch_fused<T, FAM, false, false, kWavesPerBlock>)(G, A, 0, auto_ipw, max_blocks, st);
    });
    return check_launch("k_grid_fused");
}

// ---------------------------------------------------------------------------
// Point writer (user integrands)
// ---------------------------------------------------------------------------
// h = x_1 - x_0 of an axis in the data type (integration_grid.py:90-93).
template <typename T>
__device__ inline T mesh_width(const Axis& ax, int n, int rule, const double* glx) {
    const T x0 = (T)node_of(ax, 0, n, rule, glx);
    const T x1 = (n > 1) ? (T)node_of(ax, 1, n, rule, glx) : x0;
    return x1 - x0;
}

// Any grid: one point per thread, coordinates stored one by one.  Used for
// more than 2^31 points, more axes than the staged writer's LDS holds and
// unaligned outputs.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_grid_points(const T* domain, int d, int n, int rule,
                                                        const double* glx, long long P, T* pts, T* h) {
    __shared__ Axis s_axis[kMaxDimPoints];
    for (int k = threadIdx.x; k < d; k += blockDim.x) {
        s_axis[k] = make_axis(domain, k, n, rule);
        if (h && blockIdx.x == 0) h[k] = mesh_width<T>(s_axis[k], n, rule, glx);
    }
    __syncthreads();
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x; p < P; p += stride) {
        unsigned long long rem = (unsigned long long)p;
        T* row = pts + p * d;
        for (int k = d - 1; k >= 0; --k) {
            const int j = (int)(rem % (unsigned long long)n);
            rem /= (unsigned long long)n;
            row[k] = (T)node_of(s_axis[k], j, n, rule, glx);
        }
    }
}

// Staged writer (write_stage): bound by the HBM writes of the points.  A
// point costs one multiply-high per axis for its digits and, with NODES, a
// read of the axis's node from an LDS table (else the node is formed where
// it is used).
constexpr size_t kNodeTableMax = 16 * 1024;

template <typename T, bool NODES, int PPL>
__global__ __launch_bounds__(kBlock) void k_grid_points_staged(const T* domain, int d, FastDiv by_n, int rule,
                                                               const double* glx, uint32_t P, uint32_t chunks,
                                                               T* pts, T* h) {
    extern __shared__ __align__(16) unsigned char s_raw[];
    __shared__ Axis s_axis[kMaxDimPoints];
    const int n = (int)by_n.n;
    for (int k = threadIdx.x; k < d; k += kBlock) {
        s_axis[k] = make_axis(domain, k, n, rule);
        if (h && blockIdx.x == 0) h[k] = mesh_width<T>(s_axis[k], n, rule, glx);
    }
    __syncthreads();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & (kWave - 1);
    constexpr int C = kWave * PPL;
    T* slice = reinterpret_cast<T*>(s_raw) + (size_t)wave * C * d;
    T* node = reinterpret_cast<T*>(s_raw) + (size_t)kWavesPerBlock * C * d;
    if (NODES) {
        for (int e = threadIdx.x; e < d * n; e += kBlock) {
            const int k = (int)by_n.div((uint32_t)e);
            node[e] = (T)node_of(s_axis[k], e - k * n, n, rule, glx);
        }
        __syncthreads();
    }
    const uint32_t stride = gridDim.x * kWavesPerBlock;
    for (uint32_t c = blockIdx.x * kWavesPerBlock + wave; c < chunks; c += stride) {
        const uint32_t first = c * C;
        const uint32_t left = P - first;
        const int points = left < (uint32_t)C ? (int)left : C;
        uint32_t r[PPL];
#pragma unroll
        for (int i = 0; i < PPL; ++i) {
            const int o = lane + kWave * i;
            r[i] = first + (uint32_t)(o < points ? o : 0);  // lanes past the end repeat a point that exists
        }
        for (int k = d - 1; k >= 0; --k) {
#pragma unroll
            for (int i = 0; i < PPL; ++i) {
                const uint32_t q = by_n.div(r[i]);
                const int j = (int)(r[i] - q * by_n.n);
                r[i] = q;
                slice[(lane + kWave * i) * d + k] =
                    NODES ? node[k * n + j] : (T)node_of(s_axis[k], j, n, rule, glx);
            }
        }
        wave_lds_fence();
        write_stage<T>(slice, pts, (long long)first, points, C, d);
        wave_lds_fence();  // the slice is read before the next chunk overwrites it
    }
}

template <typename T, int PPL>
static void launch_points_staged(const tq_grid_desc* g, const void* domain, long long P, void* points, void* h,
                                 hipStream_t st) {
    const FastDiv by_n = make_fast_div((uint32_t)g->n);
    const size_t nodes = (size_t)g->dim * g->n * sizeof(T);
    const uint32_t chunks = (uint32_t)((P + kWave * PPL - 1) / (kWave * PPL));
    // as many blocks as there is work for, at most 8 per CU: each builds the
    // node table once and then walks its chunks
    long long blocks = ((long long)chunks + kWavesPerBlock - 1) / kWavesPerBlock;
    if (blocks > 2048) blocks = 2048;
    // the node table where a block uses a node twice or more: 4000 points of
    // one axis took 4.5 us with it, 2.5 us without
    const bool table = nodes <= kNodeTableMax && P >= 2 * blocks * g->n;
    const size_t lds = stage_bytes(g->dim, sizeof(T), PPL) * kWavesPerBlock + (table ? nodes : 0);
    if (table)
        hipLaunchKernelGGL((k_grid_points_staged<T, true, PPL>), dim3((unsigned)blocks), dim3(kBlock), lds, st,
                           (const T*)domain, g->dim, by_n, g->rule, g->gl_nodes, (uint32_t)P, chunks, (T*)points,
                           (T*)h);
    else
        hipLaunchKernelGGL((k_grid_points_staged<T, false, PPL>), dim3((unsigned)blocks), dim3(kBlock), lds, st,
                           (const T*)domain, g->dim, by_n, g->rule, g->gl_nodes, (uint32_t)P, chunks, (T*)points,
                           (T*)h);
}

template <typename T>
static int launch_points(const tq_grid_desc* g, const void* domain, long long P, void* points, void* h,
                         hipStream_t st) {
    const int ppl = stage_ppl(g->dim, sizeof(T), P, 2048);
    if (P <= 0x7fffffffLL && stage_fits(g->dim, sizeof(T), ppl, points)) {
        if (ppl > 1)
            launch_points_staged<T, 16 / (int)sizeof(T)>(g, domain, P, points, h, st);
        else
            launch_points_staged<T, 1>(g, domain, P, points, h, st);
        return check_launch("k_grid_points_staged");
    }
    long long blocks = (P + kBlock - 1) / kBlock;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL((k_grid_points<T>), dim3((unsigned)blocks), dim3(kBlock), 0, st, (const T*)domain, g->dim,
                       g->n, g->rule, g->gl_nodes, P, (T*)points, (T*)h);
    return check_launch("k_grid_points");
}

template <typename T>
__global__ void k_grid_h(const T* domain, int d, int n, int rule, const double* glx, T* h) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= d) return;
    h[k] = mesh_width<T>(make_axis(domain, k, n, rule), n, rule, glx);
}

// ---------------------------------------------------------------------------
// Weighted reduction of user values f[P, S] (kernels in tq_values.hpp)
// ---------------------------------------------------------------------------
// Scale of the weighted reduction: Newton-Cotes uses the caller's mesh
// widths when given (hs[k]/c as _apply_composite_rule does), otherwise the
// domain's; Gauss-Legendre uses (b-a)/2 per axis.
template <typename T>
__device__ inline double reduce_scale(const T* domain, const T* hs, int d, int n, int rule, int unit) {
    double scale = 1.0;
    for (int k = 0; k < d; ++k) {
        const double a = (double)domain[2 * k], b = (double)domain[2 * k + 1];
        if (unit || rule == TQ_RULE_GAUSS_LEGENDRE) {
            scale *= 0.5 * (b - a);
        } else if (hs) {
            const double h = (double)hs[k];
            scale *= (rule == TQ_RULE_TRAPEZOID) ? h / 2.0 : (rule == TQ_RULE_SIMPSON) ? h / 3.0 : h / 22.5;
        } else {
            scale *= axis_scale(a, b, n, rule);
        }
    }
    return scale;
}

template <typename T>
struct GridScale {
    const T* domain;
    const T* hs;
    int d, n, rule, unit;
    __device__ double operator()() const { return reduce_scale(domain, hs, d, n, rule, unit); }
};

// Plan of the reduction; unit weights: every point weighs 1.
static int plan_reduce(const tq_grid_desc* g, long long S, int unit, ValuePlan& V) {
    long long P;
    ipow_checked(g->n, g->dim, 1LL << 62, &P);
    return plan_values(unit ? 0 : g->dim, g->n, g->rule, g->gl_weights, P, S, g->dtype == TQ_F32 ? 4 : 8, V);
}

// Backward of the weighted reduction: grad_f[p, s] = grad_out[s] * scale *
// W(p), a stream of writes.  Waves write contiguous ranges of `span` values
// (a multiple of 64 VEC), VEC per lane and store; a lane's values mostly
// share their point, so its weight is formed when the point changes (1e6
// values, d=4: 10.2 -> 5.4 us; [N, S] values were written one component at a
// time with lanes S elements apart).  One
// more block (when grad_domain is asked for) forms d/d domain, which only
// the scale depends on: -+ sum_s grad_out[s] out[s] / (b_k - a_k).
template <typename T, int VEC, int MODE>
__global__ __launch_bounds__(kBlock) void k_grid_reduce_backward(PointWeights w, GridScale<T> scale, const T* grad_out,
                                                                 FastDiv by_S, long long total, long long span,
                                                                 T* grad_f, const T* out, T* grad_domain) {
    extern __shared__ double s_w[];
    __shared__ double s_scale, s_red[kWavesPerBlock];
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int S = (int)by_S.n;
    if (grad_domain && blockIdx.x == gridDim.x - 1) {
        double v = 0.0;
        for (int s = tid; s < S; s += kBlock) v = fma((double)grad_out[s], (double)out[s], v);
        v = block_sum(v, s_red);
        if (tid == 0) s_scale = v;
        __syncthreads();
        for (int k = tid; k < scale.d; k += kBlock) {
            const double g = s_scale / ((double)scale.domain[2 * k + 1] - (double)scale.domain[2 * k]);
            grad_domain[2 * k] = (T)(-g);
            grad_domain[2 * k + 1] = (T)g;
        }
        return;
    }
    if (tid == 0) s_scale = scale();
    const WeightTables tab = build_weights<MODE>(w, s_w);
    __syncthreads();
    const double sc = s_scale;
    const long long wave = (long long)blockIdx.x * kWavesPerBlock + __builtin_amdgcn_readfirstlane(tid >> 6);
    const long long e0 = wave * span;
    if (e0 >= total) return;
    const uint32_t len = (uint32_t)(total - e0 < span ? total - e0 : span);
    uint32_t sub0 = 0, row0 = 0, in0 = 0;
    if (total <= 0x7fffffffLL) {  // every index fits the 32-bit divisions below
        if (S == 1) in0 = (uint32_t)e0;
        else sub0 = (uint32_t)e0;
    } else {
        const long long pt0 = S == 1 ? e0 : e0 / S;
        sub0 = S == 1 ? 0u : (uint32_t)(e0 - pt0 * S);
        in0 = (uint32_t)pt0;
        if (MODE != kUnitWeights && w.outer_axes > 0) {
            row0 = (uint32_t)(pt0 / w.inner);
            in0 = (uint32_t)(pt0 - (long long)row0 * w.inner);
        }
    }
    const double g0 = S == 1 ? (double)grad_out[0] : 0.0;
    T* dst = grad_f + e0;
    auto values = [&](uint32_t off, T* x, int count) {
        if (S == 1) {
            if (MODE == kUnitWeights || w.outer_axes == 0) {
                for (int i = 0; i < count; ++i)
                    x[i] = (T)(sc * point_weight<MODE>(w, tab, row0, in0, off + i) * g0);
                return;
            }
            // one outer weight per row
            const uint32_t p = in0 + off, r = w.by_inner.div(p);
            uint32_t in = p - r * w.inner;
            double wo = sc * outer_weight<MODE>(w, tab, row0 + r);
            for (int i = 0; i < count; ++i, ++in) {
                if (in == w.inner) {
                    in = 0;
                    wo = sc * outer_weight<MODE>(w, tab, row0 + r + 1);
                }
                x[i] = (T)(wo * inner_weight<MODE>(w, tab, in) * g0);
            }
            return;
        }
        uint32_t pt = by_S.div(sub0 + off), s = sub0 + off - pt * (uint32_t)S;
        double wp = sc * point_weight<MODE>(w, tab, row0, in0, pt);
        for (int i = 0; i < count; ++i, ++s) {
            if (s == (uint32_t)S) {
                s = 0;
                ++pt;
                wp = sc * point_weight<MODE>(w, tab, row0, in0, pt);
            }
            x[i] = (T)(wp * (double)grad_out[s]);
        }
    };
    uint32_t off = 0;
    constexpr uint32_t step = kWave * VEC;
    for (; off + step <= len; off += step) {
        T x[VEC];
        values(off + lane * VEC, x, VEC);
        if constexpr (VEC == 1) {
            dst[off + lane] = x[0];
        } else {
            using V = __attribute__((ext_vector_type(VEC))) T;
            V v;
#pragma unroll
            for (int i = 0; i < VEC; ++i) v[i] = x[i];
            *reinterpret_cast<V*>(dst + off + lane * VEC) = v;
        }
    }
    for (off += lane; off < len; off += kWave) values(off, dst + off, 1);
}

// Below kSmallBackward values a lane writes one, with the weights formed where
// they are used: the tables that a block would build first, and waves of 1024
// values on a few CUs, took longer than the launch (1.5e4 values, d=4, FP64:
// 6.7 us, now 3.5; 1e6 values, d=6, FP32: 6.4 us with tables, 9.7 without).
// Up to kMidBackward values waves of 256 still leave enough of them (7e5
// values, FP32: 4.0 us, 6.5 with 1024; 3e6: 10.2 and 9.5).
constexpr long long kSmallBackward = 1LL << 19, kMidBackward = 1LL << 21;

template <typename T>
static int launch_reduce_backward(const tq_grid_desc* g, const void* domain, const void* hs, int unit,
                                  const void* grad_out, long long S, void* grad_f, const void* out, void* grad_domain,
                                  hipStream_t st) {
    constexpr int VEC = 16 / (int)sizeof(T);
    ValuePlan V;  // for the weights; the values' split below is over P * S elements
    int rc = plan_reduce(g, 1, unit, V);
    if (rc) return rc;
    const long long total = V.P * S;
    const bool small = total < kSmallBackward;
    if (small && V.w.mode != kUnitWeights) direct_weights(g->dim, V);
    const GridScale<T> scale{(const T*)domain, (const T*)hs, g->dim, g->n, g->rule, unit};
    long long span = (total + 8191) / 8192;
    if (span < 1024) span = total < kMidBackward ? 256 : 1024;
    span = (span + kWave * VEC - 1) / (kWave * VEC) * (kWave * VEC);
    if (small) span = kWave;
    if (span > (1LL << 30)) return fail(TQ_E_ARG, "too many values for one launch");
    const long long per_block = span * kWavesPerBlock;
    const long long blocks = (grad_f ? (total + per_block - 1) / per_block : 0) + (grad_domain ? 1 : 0);
    if (blocks == 0) return TQ_OK;
    const bool vec = !small && ((uintptr_t)grad_f & 15) == 0 &&
                     (V.w.mode == kUnitWeights || S > 1 || V.w.inner >= (uint32_t)VEC);
    const FastDiv by_S = make_fast_div((uint32_t)S);
#define TQ_RB(VV, MODE)                                                                                             \
    hipLaunchKernelGGL((k_grid_reduce_backward<T, VV, MODE>), dim3((unsigned)blocks), dim3(kBlock), V.lds, st, V.w, \
                       scale, (const T*)grad_out, by_S, total, span, (T*)grad_f, (const T*)out, (T*)grad_domain)
#define TQ_RBV(MODE)                     \
    do {                                 \
        if (vec) TQ_RB(VEC, MODE);       \
        else TQ_RB(1, MODE);             \
    } while (0)
    if (V.w.mode == kUnitWeights) TQ_RBV(kUnitWeights);
    else if (V.w.mode == kTableWeights) TQ_RBV(kTableWeights);
    else TQ_RBV(kDirectWeights);
#undef TQ_RBV
#undef TQ_RB
    return check_launch("k_grid_reduce_backward");
}

// Backward of the point writer over grad_points[P, d], a stream of reads.
// A node is x = a (1 - t) + b t with t = j/(n-1), or (1 + r_j)/2 for
// Gaussian rules, so d/da = sum g (1 - t) and d/db = sum g t: two sums per
// axis.  64 / d points per wave and load, each lane on one axis, whose digit
// of the point index takes two multiply-highs; t comes from an LDS table
// when it fits.  With 64-bit divisions per element 1e6 points, d=4 took 28 us,
// 11 us so (21 MB read; the rest is launch, table and block sums).
constexpr int kNodeWeights = 2048;  // t values kept in LDS (16 KB)

// t of node j
__device__ inline double node_fraction(int j, int n, int rule, const double* glx) {
    if (rule == TQ_RULE_GAUSS_LEGENDRE) return 0.5 * (1.0 + glx[j]);
    return n > 1 ? (double)j / (double)(n - 1) : 0.0;
}

template <typename T, bool TABLE>
__global__ __launch_bounds__(kBlock) void k_grid_points_backward(int d, int n, int rule, const double* glx,
                                                                 long long P, long long span, const T* gp,
                                                                 double* partials /* [blocks][d][2] */) {
    __shared__ double s_t[TABLE ? kNodeWeights : 1];
    __shared__ double s_a[kBlock], s_b[kBlock];
    if (TABLE) {
        for (int j = threadIdx.x; j < n; j += kBlock) s_t[j] = node_fraction(j, n, rule, glx);
        __syncthreads();
    }
    const int lane = threadIdx.x & (kWave - 1);
    const int step = kWave / d, po = lane / d, k = lane - po * d;
    const long long wave = (long long)blockIdx.x * kWavesPerBlock + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long long p0 = wave * span, p1 = p0 + span < P ? p0 + span : P;
    double acc = 0.0, acc_t = 0.0;
    if (po < step && p0 < p1) {
        // digit of axis k: (p / n^(d-1-k)) mod n.  It repeats every n^(d-k) points, so the walk keeps p
        // modulo that period (when it is below 2^31) and divides 32-bit numbers.
        long long stride = 1;
        for (int q = k + 1; q < d; ++q) stride *= n;
        const bool small = stride <= 0x3fffffffLL / n;
        const long long period = stride * n;
        long long p = p0 + po;
        uint32_t r = small ? (uint32_t)(p % period) : 0u;
        const uint32_t st32 = small ? (uint32_t)stride : 1u;
        // multiply-high constants of this lane's stride (tq FastDiv)
        uint32_t m = 1u, sh = 0u;
        if (st32 > 1u) {
            const int l = 32 - __builtin_clz(st32 - 1u);
            sh = (uint32_t)l - 1u;
            m = (uint32_t)(((1ull << (31 + l)) + st32 - 1ull) / st32);
        }
        const uint32_t per32 = small ? (uint32_t)period : 0xffffffffu;
        // one step may pass several periods of a short axis
        const uint32_t adv = small ? (uint32_t)step % per32 : 0u;
        const T* src = gp + p0 * d + lane;
        const long long row = (long long)step * d;
        constexpr int U = 4;
        // t of this lane's axis at point q; then the walk's digit state moves one step on
        auto fraction = [&](long long q) {
            const int j = small ? (int)(st32 == 1u ? r : __umulhi(r, m) >> sh) : (int)((q / stride) % n);
            r += adv;
            if (r >= per32) r -= per32;
            return TABLE ? s_t[j] : node_fraction(j, n, rule, glx);
        };
        // (sum g - sum g t would lose the first where the gradients sit at the upper end)
        auto add = [&](double g, double t) {
            acc = fma(g, 1.0 - t, acc);
            acc_t = fma(g, t, acc_t);
        };
        for (; p + (long long)(U - 1) * step < p1; p += (long long)U * step, src += U * row) {
            T x[U];
#pragma unroll
            for (int u = 0; u < U; ++u) x[u] = src[u * row];
#pragma unroll
            for (int u = 0; u < U; ++u) add((double)x[u], fraction(p + (long long)u * step));
        }
        for (; p < p1; p += step, src += row) add((double)*src, fraction(p));
    }
    s_a[threadIdx.x] = acc;
    s_b[threadIdx.x] = acc_t;
    __syncthreads();
    if ((int)threadIdx.x < d) {
        double va = 0.0, vb = 0.0;
        for (int q = 0; q < kWavesPerBlock; ++q)
            for (int i = threadIdx.x; i < step * d; i += d) {
                va += s_a[q * kWave + i];
                vb += s_b[q * kWave + i];
            }
        partials[((long long)blockIdx.x * d + threadIdx.x) * 2] = va;
        partials[((long long)blockIdx.x * d + threadIdx.x) * 2 + 1] = vb;
    }
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_grid_points_backward_finalize(const double* partials, long long nb,
                                                                          int d, T* grad_domain) {
    __shared__ double s_red[kWavesPerBlock];
    const int e = blockIdx.x;  // (k, side)
    double v = 0.0;
    for (long long b = threadIdx.x; b < nb; b += blockDim.x) v += partials[b * d * 2 + e];
    v = block_sum(v, s_red);
    if (threadIdx.x == 0) grad_domain[e] = (T)v;
}

// Points per wave: at most about 4096 waves, at least 512 values each.
static void points_backward_shape(int d, long long P, long long* span, long long* nb) {
    const long long least = (512 + d - 1) / d;
    long long s = (P + 4095) / 4096;
    if (s < least) s = least;
    *span = s;
    *nb = (P + s * kWavesPerBlock - 1) / (s * kWavesPerBlock);
}

// ---------------------------------------------------------------------------
// Allocation-free entry point: the block partials live in a file-scope
// device array instead of a caller workspace.  Each device holds its own copy
// of the array; host code reaches it only through the address that
// hipGetSymbolAddress returns with that device current (the array's name is
// a host-side stand-in, not a device address).  Every block writes its
// partial before the last block reads it; the completion counter in the
// first bytes starts at zero (static storage) and every launch leaves it zero.
// ---------------------------------------------------------------------------
constexpr size_t kNoAllocScratchBytes = (size_t)1 << 20;  // the counters and (1 MiB - kWsHeader) / 8 block partials
constexpr int kMaxDevices = 64;

static __device__ __align__(256) double scratch[kNoAllocScratchBytes / sizeof(double)];

static std::mutex g_scratch_mu;
static void* g_scratch_ptr[kMaxDevices] = {};

// Device address of the current device's scratch array, looked up once per
// device (with that device current) and kept.
static int current_scratch(void** out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) {
        set_error("hipGetDevice: %s", hipGetErrorString(e));
        return (int)e;
    }
    if (dev < 0 || dev >= kMaxDevices) return fail(TQ_E_UNSUPPORTED, "device index beyond the scratch table");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            set_error("hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
            return e != hipSuccess ? (int)e : TQ_E_UNSUPPORTED;
        }
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return TQ_OK;
}

}  // namespace tq

using namespace tq;

extern "C" {

size_t tq_grid_workspace_size(const tq_grid_desc* g) {
    if (check_grid_desc(g, TQ_MAX_DIM)) return 0;
    GridGeom G;
    if (make_geom(g, G)) return 0;
    const long long blocks = G.blocks > kFusedMinBlocks ? G.blocks : kFusedMinBlocks;
    return kWsHeader + (size_t)blocks * sizeof(double);
}

int tq_grid_integrate(const tq_grid_desc* g, const tq_integrand* f, const void* domain, void* workspace,
                      size_t workspace_bytes, void* out, double* out_f64, void* stream) {
    int rc = check_grid_desc(g, TQ_MAX_DIM);
    if (rc) return rc;
    rc = check_gl_tables(g);
    if (rc) return rc;
    rc = check_integrand(f, g->dim);
    if (rc) return rc;
    if (!domain) return fail(TQ_E_NULL, "domain is NULL");
    if (!out && !out_f64) return fail(TQ_E_NULL, "no output pointer");
    if (g->dtype == TQ_F32)
        return launch_grid<float>(g, f, domain, workspace, workspace_bytes, out, out_f64, as_stream(stream));
    return launch_grid<double>(g, f, domain, workspace, workspace_bytes, out, out_f64, as_stream(stream));
}

int tq_grid_integrate_noalloc(const tq_grid_desc* g, const tq_integrand* f, const void* domain, void* out,
                              double* out_f64, void* stream) {
    int rc = check_grid_desc(g, TQ_MAX_DIM);
    if (rc) return rc;
    rc = check_gl_tables(g);
    if (rc) return rc;
    rc = check_integrand(f, g->dim);
    if (rc) return rc;
    if (!domain) return fail(TQ_E_NULL, "domain is NULL");
    if (!out && !out_f64) return fail(TQ_E_NULL, "no output pointer");
    // the same partial count as a workspace of tq_grid_workspace_size bytes,
    // so both entry points launch the same geometry
    const size_t need = tq_grid_workspace_size(g);
    if (need == 0) return fail(TQ_E_ARG, "invalid grid geometry");
    if (need > kNoAllocScratchBytes) {
        set_error("tq_grid_integrate_noalloc: %zu bytes of block partials exceed its %zu-byte scratch; use "
                  "tq_grid_integrate with a workspace",
                  need, kNoAllocScratchBytes);
        return TQ_E_WORKSPACE;
    }
    void* ws = nullptr;
    rc = current_scratch(&ws);
    if (rc) return rc;
    if (g->dtype == TQ_F32)
        return launch_grid<float>(g, f, domain, ws, need, out, out_f64, as_stream(stream));
    return launch_grid<double>(g, f, domain, ws, need, out, out_f64, as_stream(stream));
}

int tq_grid_points_h(const tq_grid_desc* g, const void* domain, void* points, void* h_out, void* stream) {
    int rc = check_grid_desc(g, kMaxDimPoints);
    if (rc) return rc;
    rc = check_gl_tables(g);
    if (rc) return rc;
    if (!domain || !points) return fail(TQ_E_NULL, "domain/points is NULL");
    long long P;
    ipow_checked(g->n, g->dim, 1LL << 62, &P);
    if (g->dtype == TQ_F32) return launch_points<float>(g, domain, P, points, h_out, as_stream(stream));
    return launch_points<double>(g, domain, P, points, h_out, as_stream(stream));
}

int tq_grid_points(const tq_grid_desc* g, const void* domain, void* points, void* stream) {
    return tq_grid_points_h(g, domain, points, nullptr, stream);
}

int tq_grid_h(const tq_grid_desc* g, const void* domain, void* h_out, void* stream) {
    int rc = check_grid_desc(g, kMaxDimPoints);
    if (rc) return rc;
    rc = check_gl_tables(g);
    if (rc) return rc;
    if (!domain || !h_out) return fail(TQ_E_NULL, "domain/h is NULL");
    const int blocks = (g->dim + 63) / 64;
    if (g->dtype == TQ_F32)
        hipLaunchKernelGGL((k_grid_h<float>), dim3(blocks), dim3(64), 0, as_stream(stream), (const float*)domain,
                           g->dim, g->n, g->rule, g->gl_nodes, (float*)h_out);
    else
        hipLaunchKernelGGL((k_grid_h<double>), dim3(blocks), dim3(64), 0, as_stream(stream), (const double*)domain,
                           g->dim, g->n, g->rule, g->gl_nodes, (double*)h_out);
    return check_launch("k_grid_h");
}

size_t tq_grid_reduce_workspace_size(const tq_grid_desc* g, int64_t S) {
    if (check_grid_desc(g, kMaxDimPoints) || S < 1) return 0;
    ValuePlan V;  // the same partial count with and without unit weights
    if (plan_reduce(g, S, 0, V)) return 0;
    return values_workspace(V);
}

int tq_grid_reduce(const tq_grid_desc* g, const void* domain, const void* hs, int32_t unit_weights,
                   const void* fvals, int64_t S, void* workspace, size_t workspace_bytes, void* out,
                   void* stream) {
    int rc = check_grid_desc(g, kMaxDimPoints);
    if (rc) return rc;
    if (!unit_weights) {
        rc = check_gl_tables(g);
        if (rc) return rc;
    }
    if (S < 1) return fail(TQ_E_ARG, "S must be >= 1");
    if (!domain || !fvals || !out) return fail(TQ_E_NULL, "domain/fvals/out is NULL");
    if (S > 65535) return fail(TQ_E_UNSUPPORTED, "more than 65535 integrand components");
    const int unit = unit_weights ? 1 : 0;
    ValuePlan V;
    rc = plan_reduce(g, S, unit, V);
    if (rc) return rc;
    if (!workspace || workspace_bytes < values_workspace(V)) return fail(TQ_E_WORKSPACE, "reduce workspace too small");
    hipStream_t st = as_stream(stream);
    if (g->dtype == TQ_F32)
        return launch_values<float>(V, (const float*)fvals, (double*)workspace,
                                    GridScale<float>{(const float*)domain, (const float*)hs, g->dim, g->n, g->rule, unit},
                                    (float*)out, st);
    return launch_values<double>(V, (const double*)fvals, (double*)workspace,
                                 GridScale<double>{(const double*)domain, (const double*)hs, g->dim, g->n, g->rule, unit},
                                 (double*)out, st);
}

int tq_grid_reduce_vjp(const tq_grid_desc* g, const void* domain, const void* hs, int32_t unit_weights,
                       const void* grad_out, const void* out, int64_t S, void* grad_f, void* grad_domain,
                       void* stream) {
    int rc = check_grid_desc(g, kMaxDimPoints);
    if (rc) return rc;
    if (!unit_weights) {
        rc = check_gl_tables(g);
        if (rc) return rc;
    }
    if (S < 1 || S > 0x3fffffff) return fail(TQ_E_ARG, "S out of range");
    if (!domain || !grad_out || (!grad_f && !grad_domain)) return fail(TQ_E_NULL, "domain/grad_out/grad_f is NULL");
    if (grad_domain && !out) return fail(TQ_E_NULL, "grad_domain needs the forward result");
    const int unit = unit_weights ? 1 : 0;
    if (grad_domain && hs && !unit && g->rule != TQ_RULE_GAUSS_LEGENDRE)
        return fail(TQ_E_ARG, "with mesh widths the result does not depend on the domain");
    if (g->dtype == TQ_F32)
        return launch_reduce_backward<float>(g, domain, hs, unit, grad_out, S, grad_f, out, grad_domain,
                                             as_stream(stream));
    return launch_reduce_backward<double>(g, domain, hs, unit, grad_out, S, grad_f, out, grad_domain,
                                          as_stream(stream));
}

int tq_grid_reduce_backward(const tq_grid_desc* g, const void* domain, const void* hs, int32_t unit_weights,
                            const void* grad_out, int64_t S, void* grad_f, void* stream) {
    if (!grad_f) return fail(TQ_E_NULL, "domain/grad_out/grad_f is NULL");
    return tq_grid_reduce_vjp(g, domain, hs, unit_weights, grad_out, nullptr, S, grad_f, nullptr, stream);
}

size_t tq_grid_points_backward_workspace_size(const tq_grid_desc* g) {
    if (check_grid_desc(g, kMaxDimPoints)) return 0;
    long long P, span, nb;
    ipow_checked(g->n, g->dim, 1LL << 62, &P);
    points_backward_shape(g->dim, P, &span, &nb);
    return (size_t)(nb * g->dim * 2) * sizeof(double);
}

}  // extern "C"

template <typename T>
static int launch_points_backward(const tq_grid_desc* g, const void* grad_points, void* ws, size_t ws_bytes,
                                  void* grad_domain, hipStream_t s) {
    long long P, span, nb;
    ipow_checked(g->n, g->dim, 1LL << 62, &P);
    points_backward_shape(g->dim, P, &span, &nb);
    if (!ws || ws_bytes < (size_t)(nb * g->dim * 2) * sizeof(double))
        return fail(TQ_E_WORKSPACE, "points backward workspace too small");
    if (g->n <= kNodeWeights)
        hipLaunchKernelGGL((k_grid_points_backward<T, true>), dim3((unsigned)nb), dim3(kBlock), 0, s, g->dim, g->n,
                           g->rule, g->gl_nodes, P, span, (const T*)grad_points, (double*)ws);
    else
        hipLaunchKernelGGL((k_grid_points_backward<T, false>), dim3((unsigned)nb), dim3(kBlock), 0, s, g->dim, g->n,
                           g->rule, g->gl_nodes, P, span, (const T*)grad_points, (double*)ws);
    const int rc = check_launch("k_grid_points_backward");
    if (rc) return rc;
    hipLaunchKernelGGL((k_grid_points_backward_finalize<T>), dim3(g->dim * 2), dim3(kBlock), 0, s, (const double*)ws,
                       nb, g->dim, (T*)grad_domain);
    return check_launch("k_grid_points_backward_finalize");
}

extern "C" {

int tq_grid_points_backward(const tq_grid_desc* g, const void* domain, const void* grad_points, void* workspace,
                            size_t workspace_bytes, void* grad_domain, void* stream) {
    int rc = check_grid_desc(g, kMaxDimPoints);
    if (rc) return rc;
    rc = check_gl_tables(g);
    if (rc) return rc;
    if (!domain || !grad_points || !grad_domain) return fail(TQ_E_NULL, "domain/grad_points/grad_domain is NULL");
    if (g->dtype == TQ_F32)
        return launch_points_backward<float>(g, grad_points, workspace, workspace_bytes, grad_domain,
                                             as_stream(stream));
    return launch_points_backward<double>(g, grad_points, workspace, workspace_bytes, grad_domain, as_stream(stream));
}

}  // extern "C"
