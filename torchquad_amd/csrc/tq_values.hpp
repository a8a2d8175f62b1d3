// Weighted sums of integrand values f[P, S] that the caller's function left
// in memory: the grid rules' tensor-product weights (P = n^d, ij order) and
// Monte Carlo's mean (weight 1).  All kernels are bound by reading f once;
// the weights come from the point index and the sums are FP64.
//
// A point p splits into an outer index (the leading axes) and an inner one
// (the last m axes, n^m <= kInnerMax points).  Each block builds the inner
// weights and the axis weights in LDS, so a point costs one multiply-high
// and two LDS reads plus one of each per outer axis.  Reading one value per
// lane with the weights of the outer axes formed by branches on the rule
// took 342 us for 6.9e7 FP32 values (d=5, n=37), 0.8 TB/s; this takes 67 us,
// 4.1 TB/s.  [10001, 200] values: 81 + 16 us with lanes over (point,
// component) pairs and 256 comparisons per component in every block, 4 + 4 us
// with k_values_cols; Monte Carlo's mean of 2e7 values 36 + 7 -> 14 + 5 us.
#pragma once
#include "tq_grid_tile.hpp"

namespace tq {

constexpr int kInnerMax = 2048;  // inner weights kept in LDS (16 KB)
constexpr int kFinalBlock = 1024;

// How the weights of points are formed.
enum { kUnitWeights = 0, kTableWeights = 1, kDirectWeights = 2 };

struct PointWeights {
    int mode, rule, n, outer_axes;
    uint32_t inner;  // points per outer index
    FastDiv by_inner, by_n;
    const double* glw;
};

struct ValuePlan {
    PointWeights w;
    long long P, S;
    long long span;    // points per wave
    long long blocks;  // rows of partials
    int vec;           // values per load (S == 1)
    size_t lds;        // weight tables
};

// Weight of node j where no table holds it (rule -1: 1).
__device__ inline double direct_weight(const PointWeights& w, uint32_t j) {
    return weight_of(w.rule, (int)j, w.n, w.glw);
}

struct WeightTables {
    double* in;  // inner weights
    double* ax;  // weights of one axis (== in when one axis is inner)
};

template <int MODE>
__device__ inline WeightTables build_weights(const PointWeights& w, double* lds) {
    WeightTables t{lds, lds};
    if constexpr (MODE == kTableWeights) {
        const bool one = (uint32_t)w.n == w.inner;
        if (!one) t.ax = lds + w.inner;
        for (int j = threadIdx.x; j < w.n; j += blockDim.x) t.ax[j] = weight_of(w.rule, j, w.n, w.glw);
        __syncthreads();
        if (!one) {
            for (uint32_t e = threadIdx.x; e < w.inner; e += blockDim.x) {
                double v = 1.0;
                uint32_t r = e;
                for (uint32_t left = w.inner; left > 1u; left = w.by_n.div(left)) {
                    const uint32_t q = w.by_n.div(r);
                    v *= t.ax[r - q * w.by_n.n];
                    r = q;
                }
                t.in[e] = v;
            }
            __syncthreads();
        }
    }
    return t;
}

template <int MODE>
__device__ inline double inner_weight(const PointWeights& w, const WeightTables& t, uint32_t i) {
    if constexpr (MODE == kTableWeights) return t.in[i];
    else if constexpr (MODE == kDirectWeights) return direct_weight(w, i);
    else return 1.0;
}

template <int MODE>
__device__ inline double outer_weight(const PointWeights& w, const WeightTables& t, uint32_t row) {
    double v = 1.0;
    if constexpr (MODE != kUnitWeights) {
        for (int k = 0; k < w.outer_axes; ++k) {
            const uint32_t q = w.by_n.div(row);
            const uint32_t j = row - q * w.by_n.n;
            v *= MODE == kTableWeights ? t.ax[j] : direct_weight(w, j);
            row = q;
        }
    }
    return v;
}

// Weight of the point `off` points after (row0, in0).
template <int MODE>
__device__ inline double point_weight(const PointWeights& w, const WeightTables& t, uint32_t row0, uint32_t in0,
                                      uint32_t off) {
    if constexpr (MODE == kUnitWeights) return 1.0;
    if (w.outer_axes == 0) return inner_weight<MODE>(w, t, in0 + off);
    const uint32_t p = in0 + off, r = w.by_inner.div(p);
    return outer_weight<MODE>(w, t, row0 + r) * inner_weight<MODE>(w, t, p - r * w.inner);
}

template <typename T, int VEC>
struct ValueVec {
    T v[VEC];
};

template <typename T, int VEC>
__device__ inline ValueVec<T, VEC> load_values(const T* p) {
    ValueVec<T, VEC> r;
    if constexpr (VEC == 1) {
        r.v[0] = *p;
    } else {
        using V = __attribute__((ext_vector_type(VEC))) T;
        const V x = *reinterpret_cast<const V*>(p);
#pragma unroll
        for (int i = 0; i < VEC; ++i) r.v[i] = x[i];
    }
    return r;
}

// Weighted sum of VEC consecutive values, the first `off` points after
// (row0, in0).  The values of one row share its outer weight; lanes whose
// values cross into the next row (VEC <= inner, so one crossing at most)
// send the whole wave through the two-row form.
template <typename T, int VEC, int MODE>
__device__ inline double weigh(const PointWeights& w, const WeightTables& t, uint32_t row0, uint32_t in0, uint32_t off,
                               const ValueVec<T, VEC>& x) {
    double r = 0.0;
    if constexpr (MODE == kUnitWeights) {
#pragma unroll
        for (int i = 0; i < VEC; ++i) r += (double)x.v[i];
        return r;
    } else {
        uint32_t row = 0, in = in0 + off;
        if (w.outer_axes > 0) {
            row = w.by_inner.div(in);
            in -= row * w.inner;
        }
        if (VEC == 1 || !__any(in + VEC > w.inner)) {
#pragma unroll
            for (int i = 0; i < VEC; ++i) r = fma(inner_weight<MODE>(w, t, in + i), (double)x.v[i], r);
            return w.outer_axes > 0 ? outer_weight<MODE>(w, t, row0 + row) * r : r;
        }
        double r2 = 0.0;
#pragma unroll
        for (int i = 0; i < VEC; ++i) {
            const bool next = in + i >= w.inner;
            const double y = inner_weight<MODE>(w, t, next ? in + i - w.inner : in + i) * (double)x.v[i];
            r += next ? 0.0 : y;
            r2 += next ? y : 0.0;
        }
        r *= outer_weight<MODE>(w, t, row0 + row);
        // a lane that does not cross may sit in the last row, whose successor does not exist
        return in + VEC > w.inner ? fma(outer_weight<MODE>(w, t, row0 + row + 1), r2, r) : r;
    }
}

// S == 1: waves stream contiguous ranges of `span` values (a multiple of
// 64 VEC), VEC values per lane and load, four loads in flight per lane.
template <typename T, int VEC, int MODE>
__global__ __launch_bounds__(kBlock) void k_values_flat(PointWeights w, const T* fv, long long P, long long span,
                                                        double* partials) {
    extern __shared__ double s_w[];
    __shared__ double s_red[kWavesPerBlock];
    const WeightTables tab = build_weights<MODE>(w, s_w);
    const int lane = threadIdx.x & (kWave - 1);
    const long long wave = (long long)blockIdx.x * kWavesPerBlock + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long long p0 = wave * span;
    double acc = 0.0;
    if (p0 < P) {
        const uint32_t len = (uint32_t)(P - p0 < span ? P - p0 : span);
        uint32_t row0 = 0, in0 = (uint32_t)p0;
        if (MODE != kUnitWeights && w.outer_axes > 0) {
            row0 = (uint32_t)(p0 / w.inner);
            in0 = (uint32_t)(p0 - (long long)row0 * w.inner);
        }
        const T* base = fv + p0;
        constexpr int U = 4;
        constexpr uint32_t step = kWave * VEC;
        uint32_t off = 0;
        for (; off + U * step <= len; off += U * step) {
            ValueVec<T, VEC> x[U];
#pragma unroll
            for (int u = 0; u < U; ++u) x[u] = load_values<T, VEC>(base + off + u * step + lane * VEC);
#pragma unroll
            for (int u = 0; u < U; ++u) acc += weigh<T, VEC, MODE>(w, tab, row0, in0, off + u * step + lane * VEC, x[u]);
        }
        for (off += lane; off < len; off += kWave)
            acc = fma(point_weight<MODE>(w, tab, row0, in0, off), (double)base[off], acc);
    }
    const double b = block_sum(acc, s_red);
    if (threadIdx.x == 0) partials[blockIdx.x] = b;
}

// 1 < S < 64: lanes 0 .. 64 - 64 mod S of a wave read consecutive values, so
// each keeps one component and the wave steps 64 / S points.
template <typename T, int MODE>
__global__ __launch_bounds__(kBlock) void k_values_narrow(PointWeights w, const T* fv, long long P, int S,
                                                          long long span, double* partials /* [blocks][S] */) {
    extern __shared__ double s_w[];
    __shared__ double s_acc[kBlock];
    const WeightTables tab = build_weights<MODE>(w, s_w);
    const int lane = threadIdx.x & (kWave - 1);
    const long long wave = (long long)blockIdx.x * kWavesPerBlock + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long long p0 = wave * span;
    const uint32_t step = (uint32_t)(kWave / S), po = (uint32_t)(lane / S);
    double acc = 0.0;
    if (p0 < P && po < step) {
        const uint32_t len = (uint32_t)(P - p0 < span ? P - p0 : span);
        uint32_t row0 = 0, in0 = (uint32_t)p0;
        if (MODE != kUnitWeights && w.outer_axes > 0) {
            row0 = (uint32_t)(p0 / w.inner);
            in0 = (uint32_t)(p0 - (long long)row0 * w.inner);
        }
        const T* base = fv + p0 * S + lane;
        constexpr int U = MODE == kUnitWeights ? 8 : 4;  // loads in flight; with weights, 4 take fewer registers
        uint32_t off = po;
        const uint32_t row = step * (uint32_t)S;  // values per step
        long long at = 0;
        for (; off + (U - 1) * step < len; off += U * step, at += (long long)U * row) {
            T x[U];
#pragma unroll
            for (int u = 0; u < U; ++u) x[u] = base[at + u * row];
#pragma unroll
            for (int u = 0; u < U; ++u)
                acc = fma(point_weight<MODE>(w, tab, row0, in0, off + u * step), (double)x[u], acc);
        }
        for (; off < len; off += step, at += row)
            acc = fma(point_weight<MODE>(w, tab, row0, in0, off), (double)base[at], acc);
    }
    s_acc[threadIdx.x] = acc;
    __syncthreads();
    if ((int)threadIdx.x < S) {
        double v = 0.0;
        for (int q = 0; q < kWavesPerBlock; ++q)
            for (int i = threadIdx.x; i < (int)step * S; i += S) v += s_acc[q * kWave + i];
        partials[(long long)blockIdx.x * S + threadIdx.x] = v;
    }
}

// S >= 64: a wave owns 64 components (its lanes) and `span` points.  The
// lanes form the weights of 64 points at once and hand them out one point
// at a time (readlane), so a value costs one load and one FMA.
template <typename T, int MODE>
__global__ __launch_bounds__(kBlock) void k_values_cols(PointWeights w, const T* fv, long long P, long long S,
                                                        long long span, double* partials /* [gridDim.y][S] */) {
    extern __shared__ double s_w[];
    __shared__ double s_acc[kWavesPerBlock][kWave];
    const WeightTables tab = build_weights<MODE>(w, s_w);
    const int lane = threadIdx.x & (kWave - 1), wb = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long long col = (long long)blockIdx.x * kWave + lane;
    const long long colc = col < S ? col : S - 1;  // lanes past the last component read it again
    const long long p0 = ((long long)blockIdx.y * kWavesPerBlock + wb) * span;
    double acc = 0.0;
    if (p0 < P) {
        const uint32_t len = (uint32_t)(P - p0 < span ? P - p0 : span);
        uint32_t row0 = 0, in0 = (uint32_t)p0;
        if (MODE != kUnitWeights && w.outer_axes > 0) {
            row0 = (uint32_t)(p0 / w.inner);
            in0 = (uint32_t)(p0 - (long long)row0 * w.inner);
        }
        const T* base = fv + p0 * S + colc;
        for (uint32_t b = 0; b < len; b += kWave) {
            const uint32_t cnt = len - b < (uint32_t)kWave ? len - b : (uint32_t)kWave;
            union {
                double d;
                int i[2];
            } pw;
            pw.d = point_weight<MODE>(w, tab, row0, in0, b + ((uint32_t)lane < cnt ? (uint32_t)lane : 0u));
            auto weight = [&](uint32_t q) {
                union {
                    double d;
                    int i[2];
                } r;
                r.i[0] = __builtin_amdgcn_readlane(pw.i[0], (int)q);
                r.i[1] = __builtin_amdgcn_readlane(pw.i[1], (int)q);
                return r.d;
            };
            const T* row = base + (long long)b * S;
            constexpr uint32_t U = 8;
            uint32_t q = 0;
            for (; q + U <= cnt; q += U) {
                T x[U];
#pragma unroll
                for (uint32_t u = 0; u < U; ++u) x[u] = row[(long long)(q + u) * S];
#pragma unroll
                for (uint32_t u = 0; u < U; ++u) acc = fma(weight(q + u), (double)x[u], acc);
            }
            for (; q < cnt; ++q) acc = fma(weight(q), (double)row[(long long)q * S], acc);
        }
    }
    s_acc[wb][lane] = acc;
    __syncthreads();
    if (wb == 0 && col < S) {
        double v = 0.0;
        for (int q = 0; q < kWavesPerBlock; ++q) v += s_acc[q][lane];
        partials[(long long)blockIdx.y * S + col] = v;
    }
}

// out[s] = scale * sum over the blocks' partials, in a fixed order.
// Few components: one block per component; many: 64 components per block,
// rows split over its waves so that reads are coalesced.
template <typename T, typename SCALE>
__global__ __launch_bounds__(kFinalBlock) void k_values_final(const double* partials, long long blocks, long long S,
                                                              SCALE scale, T* out) {
    __shared__ double s_red[kFinalBlock / kWave];
    __shared__ double s_col[kFinalBlock / kWave][kWave];
    if (S < kWave) {
        const long long s = blockIdx.x;
        double v = 0.0;
        for (long long b = threadIdx.x; b < blocks; b += blockDim.x) v += partials[b * S + s];
        v = block_sum(v, s_red);
        if (threadIdx.x == 0) out[s] = (T)(v * scale());
        return;
    }
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x >> 6;
    const long long col = (long long)blockIdx.x * kWave + lane;
    double v = 0.0;
    if (col < S)
#pragma unroll 4
        for (long long b = w; b < blocks; b += kFinalBlock / kWave) v += partials[b * S + col];
    s_col[w][lane] = v;
    __syncthreads();
    if (w == 0 && col < S) {
        v = 0.0;
        for (int q = 0; q < kFinalBlock / kWave; ++q) v += s_col[q][lane];
        out[col] = (T)(v * scale());
    }
}

// Plan for f[P, S] of the data type's size; d = 0: unit weights over P
// points.  Waves: at most about 8192 (32 per CU), each with at least 1024
// values (512 of several components below 2^20 of them), so small inputs still spread over the chip and the final sum
// stays short.  The block count does not depend on the buffer's alignment.
inline int plan_values(int d, int n, int rule, const double* glw, long long P, long long S, int tsize, ValuePlan& V) {
    V.P = P;
    V.S = S;
    PointWeights& w = V.w;
    w.rule = rule;
    w.n = n;
    w.glw = glw;
    w.mode = kUnitWeights;
    w.outer_axes = 0;
    w.inner = 1;
    w.by_n = make_fast_div(1);
    w.by_inner = make_fast_div(1);
    V.lds = 0;
    if (d > 0) {
        long long inner = n;
        int m = 1;
        while (m < d && n > 1 && inner * n <= kInnerMax) {  // one node per axis: the other axes stay outer ones
            inner *= n;
            ++m;
        }
        w.inner = (uint32_t)inner;
        w.outer_axes = d - m;
        w.by_n = make_fast_div((uint32_t)n);
        w.by_inner = make_fast_div(w.inner);
        if (P / inner > 0x7fffffffLL) return fail(TQ_E_ARG, "more than 2^31 rows of values");
        w.mode = inner <= kInnerMax ? kTableWeights : kDirectWeights;
        if (w.mode == kTableWeights) V.lds = ((size_t)inner + (m > 1 ? (size_t)n : 0)) * sizeof(double);
    }
    const int vec = 16 / tsize;
    V.vec = (S == 1 && (d == 0 || w.inner >= (uint32_t)vec)) ? vec : 1;
    const long long groups = S < kWave ? 1 : (S + kWave - 1) / kWave;
    const long long waves = 8192 / groups > 4 ? 8192 / groups : 4;
    long long span = (P + waves - 1) / waves;
    // points per wave
    const long long least = S == 1 ? 1024 : S < kWave ? (P * S < (1LL << 20) ? 512 : 1024) / S : 16;
    if (span < least) span = least;
    const long long round = S == 1 ? kWave * vec : 1;  // of the data type, whatever the weights allow
    span = (span + round - 1) / round * round;
    if (span > (1LL << 30)) return fail(TQ_E_ARG, "too many values for one launch");
    V.span = span;
    V.blocks = (P + span * kWavesPerBlock - 1) / (span * kWavesPerBlock);
    return TQ_OK;
}

// The plan's weights without tables: one inner axis, the others outer ones.
inline void direct_weights(int d, ValuePlan& V) {
    V.w.mode = kDirectWeights;
    V.w.inner = (uint32_t)V.w.n;
    V.w.outer_axes = d - 1;
    V.w.by_inner = V.w.by_n;
    V.lds = 0;
}

inline size_t values_workspace(const ValuePlan& V) { return (size_t)(V.blocks * V.S) * sizeof(double); }

template <typename T, int MODE>
static void launch_values_mode(const ValuePlan& V, const T* fv, double* partials, hipStream_t st) {
    if (V.S == 1) {
        constexpr int VEC = 16 / (int)sizeof(T);
        if (V.vec == VEC && ((uintptr_t)fv & 15) == 0)
            hipLaunchKernelGGL((k_values_flat<T, VEC, MODE>), dim3((unsigned)V.blocks), dim3(kBlock), V.lds, st, V.w,
                               fv, V.P, V.span, partials);
        else
            hipLaunchKernelGGL((k_values_flat<T, 1, MODE>), dim3((unsigned)V.blocks), dim3(kBlock), V.lds, st, V.w, fv,
                               V.P, V.span, partials);
    } else if (V.S < kWave) {
        hipLaunchKernelGGL((k_values_narrow<T, MODE>), dim3((unsigned)V.blocks), dim3(kBlock), V.lds, st, V.w, fv,
                           V.P, (int)V.S, V.span, partials);
    } else {
        const dim3 grid((unsigned)((V.S + kWave - 1) / kWave), (unsigned)V.blocks);
        hipLaunchKernelGGL((k_values_cols<T, MODE>), grid, dim3(kBlock), V.lds, st, V.w, fv, V.P, V.S, V.span,
                           partials);
    }
}

template <typename T, typename SCALE>
static int launch_values(const ValuePlan& V, const T* fv, double* partials, SCALE scale, T* out, hipStream_t st) {
    if (V.w.mode == kUnitWeights) launch_values_mode<T, kUnitWeights>(V, fv, partials, st);
    else if (V.w.mode == kTableWeights) launch_values_mode<T, kTableWeights>(V, fv, partials, st);
    else launch_values_mode<T, kDirectWeights>(V, fv, partials, st);
    const int rc = check_launch("k_values");
    if (rc) return rc;
    const long long fb = V.S < kWave ? V.S : (V.S + kWave - 1) / kWave;
    // (few partials: four waves start and meet sooner than sixteen)
    const int threads = V.S < kWave && V.blocks <= kBlock ? kBlock : kFinalBlock;
    hipLaunchKernelGGL((k_values_final<T, SCALE>), dim3((unsigned)fb), dim3(threads), 0, st, partials, V.blocks,
                       V.S, scale, out);
    return check_launch("k_values_final");
}

}  // namespace tq
