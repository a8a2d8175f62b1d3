// Integrand values of the built-in families as products of per-axis factors.
//
// Every built-in family's value at a grid point is a short sum of products
// of one number per axis:
//   Gaussian peak     prod 2^(-t_k^2)                     1 component
//   exp-linear        prod 2^(a_k x_k)                    1
//   product peak      prod 1 / (a_k^-2 + (x_k - u_k)^2)   1
//   oscillatory       Re prod e^(i a_k x_k)               2 (complex product)
//   sin-sum           eps part of prod (1 + eps s_k)      2 (dual numbers)
//   double Gaussian   sum of two products                 2
//   constant          1                                   1
// so a point costs one multiply-add per component from tables instead of a
// transcendental (FP32: an exp2 issues for 8.4 cycles per wave, the
// multiply-add for 2.7; FP64 transcendentals are sequences of some 40
// instructions).  Every point's value is still formed and added by itself.
//
// The factors are evaluated once per axis node in FP64 (node rounded to T,
// parameters as T holds them), multiplied by the node's weight, brought to
// at most 1 in magnitude per axis (an exact power of two, returned as an
// exponent for the result) and rounded to T once.  With factors of at most 1
// a partial product can only underflow when the point's own share of the sum
// is below 2^-126 (2^-1022) of the largest, so the form needs no range check
// and does not overflow where the sum of exponents did not.
#pragma once
#include "tq_grid_tile.hpp"

namespace tq {

constexpr bool family_exponential(int fam) { return fam == TQ_FAM_GAUSSIAN_PEAK || fam == TQ_FAM_EXP_LINEAR; }
constexpr int family_comps(int fam) {
    return (fam == TQ_FAM_OSCILLATORY || fam == TQ_FAM_SIN_SUM || fam == TQ_FAM_DOUBLE_GAUSSIAN) ? 2 : 1;
}

// log2 of an exponential family's factor; the constant term goes to axis 0.
// Kept within +-1e8, far outside any result, so that the exponents of 16 axes
// add up in 32 bits and overflow to infinity only in the result (NaN stays).
template <int FAM, typename T>
__device__ inline double factor_exponent(int k, T x, const Params<T>& p) {
    double e;
    if constexpr (FAM == TQ_FAM_GAUSSIAN_PEAK) {
        const double t = fma((double)x, (double)p.a[k], (double)p.b[k]);
        e = -t * t;
    } else {
        e = (double)p.a[k] * (double)x;
        if (k == 0) e += (double)p.c1;
    }
    return e > 1e8 ? 1e8 : (e < -1e8 ? -1e8 : e);
}

// Weighted factor of a family that is not exponential.
template <int FAM, typename T>
__device__ inline void factor_comps(int k, T x, double w, const Params<T>& p, double* v) {
    if constexpr (FAM == TQ_FAM_PRODUCT_PEAK) {
        const double t = (double)x - (double)p.u[k];
        v[0] = w / fma(t, t, (double)p.b[k]);
    } else if constexpr (FAM == TQ_FAM_OSCILLATORY) {
        double s, c;
        double phase = (double)p.a[k] * (double)x;  // FP32: revolutions, FP64: radians
        if (k == 0) phase += (double)p.c2;
        if (sizeof(T) == 4) sincospi(2.0 * phase, &s, &c);
        else sincos(phase, &s, &c);
        v[0] = w * c;
        v[1] = w * s;
    } else if constexpr (FAM == TQ_FAM_SIN_SUM) {
        v[0] = w;
        v[1] = w * sin(fma((double)p.a[k], (double)x, (double)p.u[k]));
    } else if constexpr (FAM == TQ_FAM_DOUBLE_GAUSSIAN) {
        const double t1 = (double)x - (double)p.c1, t2 = (double)x - (double)p.c2, c = -(double)p.c3;
        v[0] = w * exp2(c * t1 * t1);
        v[1] = w * exp2(c * t2 * t2);
    } else {
        v[0] = w;
    }
}

template <int FAM, typename T>
struct Factor {
    static constexpr int C = family_comps(FAM);
    T v[C];

    // identity of merge
    __device__ static inline Factor one(bool on) {
        Factor r;
        r.v[0] = on ? T(1) : T(0);
        if constexpr (C == 2) r.v[1] = FAM == TQ_FAM_DOUBLE_GAUSSIAN ? r.v[0] : T(0);
        return r;
    }
    // factor of the union of two disjoint sets of axes
    __device__ static inline Factor merge(const Factor& a, const Factor& b) {
        Factor r;
        if constexpr (FAM == TQ_FAM_OSCILLATORY) {
            r.v[0] = fma(a.v[0], b.v[0], -(a.v[1] * b.v[1]));
            r.v[1] = fma(a.v[0], b.v[1], a.v[1] * b.v[0]);
        } else if constexpr (FAM == TQ_FAM_SIN_SUM) {
            r.v[0] = a.v[0] * b.v[0];
            r.v[1] = fma(a.v[0], b.v[1], a.v[1] * b.v[0]);
        } else {
#pragma unroll
            for (int c = 0; c < C; ++c) r.v[c] = a.v[c] * b.v[c];
        }
        return r;
    }
    // the form in which an entry meets a state: value(merge(a, b)) = sum_c a.v[c] * b.dual().v[c]
    __device__ inline Factor dual() const {
        Factor r = *this;
        if constexpr (FAM == TQ_FAM_OSCILLATORY) r.v[1] = -v[1];
        if constexpr (FAM == TQ_FAM_SIN_SUM) {
            r.v[0] = v[1];
            r.v[1] = v[0];
        }
        return r;
    }
};

// Exponent (as frexp) of |v|, or the smallest int for 0 and non-finite v.
__device__ inline int mag_exp(double v) {
    const int e = (int)((__double_as_longlong(v) >> 52) & 0x7ff);
    if (e == 0x7ff || v == 0.0) return -0x7fffffff;
    return e == 0 ? -1022 : e - 1022;
}
__device__ inline int exp_or_zero(int e) { return e == -0x7fffffff ? 0 : e; }

// Largest value of the wave's lanes, in every lane (DPP, no LDS).
__device__ inline int wave_max(int v) {
    auto step = [&](int o) { v = o > v ? o : v; };
    step(__builtin_amdgcn_update_dpp(v, v, 0x111, 0xF, 0xF, false));  // row_shr 1, 2, 4, 8
    step(__builtin_amdgcn_update_dpp(v, v, 0x112, 0xF, 0xF, false));
    step(__builtin_amdgcn_update_dpp(v, v, 0x114, 0xF, 0xF, false));
    step(__builtin_amdgcn_update_dpp(v, v, 0x118, 0xF, 0xF, false));
    step(__builtin_amdgcn_update_dpp(v, v, 0x142, 0xA, 0xF, false));  // row_bcast15 into rows 1 and 3
    step(__builtin_amdgcn_update_dpp(v, v, 0x143, 0xC, 0xF, false));  // row_bcast31 into rows 2 and 3
    return __builtin_amdgcn_readlane(v, kWave - 1);
}

// The integer above an exponent, or the smallest int for NaN.
__device__ inline int exp_ceil(double x) { return x == x ? (int)ceil(x) : -0x7fffffff; }

// Weighted factor of node j on axis k; top: the axis's largest exponent (exponential families).  Returns the
// exponent of the value that the axis is scaled by.
template <int FAM, typename T>
__device__ inline int weighted_factor(int k, T x, double ex, int top, double w, const Params<T>& p, double* v) {
    if constexpr (family_exponential(FAM)) {
        v[0] = w * exp2(ex - (double)exp_or_zero(top));
        return mag_exp(v[0]);
    } else {
        factor_comps<FAM, T>(k, x, w, p, v);
        return mag_exp(FAM == TQ_FAM_PRODUCT_PEAK ? v[0] : w);
    }
}

// Axis tables of a whole block: component c of axis k's node j goes to
// axis[c * d * n + k * n + j], the power of two taken out of axis k to
// s_exp[k].  Axes of up to 128 nodes: one wave per axis, two nodes per lane,
// in registers.  Longer ones: the block walks all nodes, with 8-byte copies
// of the entries in `tmp` until they are scaled (s_top: [d] ints).  Ends with
// a barrier.
constexpr int kWaveAxis = 2 * kWave;

template <int FAM, typename T>
__device__ inline void build_axis_factors(int d, int n, int rule, const Axis* ax, const double* glx,
                                          const double* glw, const Params<T>& p, FastDiv by_n, T* axis, double* tmp,
                                          int* s_top, int* s_exp) {
    constexpr int C = family_comps(FAM);
    constexpr bool EXP = family_exponential(FAM);
    const int tid = threadIdx.x, nt = blockDim.x, total = d * n;
    if (n <= kWaveAxis) {
        const int lane = tid & (kWave - 1), waves = nt >> 6;
        for (int k = __builtin_amdgcn_readfirstlane(tid >> 6); k < d; k += waves) {
            double ex[2] = {0.0, 0.0}, w[2], v[2][C];
            T x[2];
            int top = -0x7fffffff, m = -0x7fffffff;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                if (i * kWave >= n) continue;
                const int j = lane + i * kWave, jc = j < n ? j : n - 1;  // lanes past the end repeat the last node
                x[i] = (T)node_of(ax[k], jc, n, rule, glx);
                w[i] = weight_of(rule, jc, n, glw);
                if constexpr (EXP) {
                    ex[i] = factor_exponent<FAM, T>(k, x[i], p);
                    const int e = exp_ceil(ex[i]);
                    top = e > top ? e : top;
                }
            }
            if (EXP) top = wave_max(top);
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                if (i * kWave >= n) continue;
                const int e = weighted_factor<FAM, T>(k, x[i], ex[i], top, w[i], p, v[i]);
                m = e > m ? e : m;
            }
            m = exp_or_zero(wave_max(m));
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int j = lane + i * kWave;
                if (j < n)
#pragma unroll
                    for (int c = 0; c < C; ++c) axis[c * total + k * n + j] = (T)ldexp(v[i][c], -m);
            }
            if (lane == 0) s_exp[k] = m + (EXP ? exp_or_zero(top) : 0);
        }
        __syncthreads();
        return;
    }
    if (tid < d) {
        s_top[tid] = -0x7fffffff;
        s_exp[tid] = -0x7fffffff;
    }
    __syncthreads();
    if (EXP) {
        for (int e = tid; e < total; e += nt) {
            const int k = (int)by_n.div((uint32_t)e), j = e - k * n;
            tmp[e] = factor_exponent<FAM, T>(k, (T)node_of(ax[k], j, n, rule, glx), p);
            atomicMax(&s_top[k], exp_ceil(tmp[e]));
        }
        __syncthreads();
    }
    for (int e = tid; e < total; e += nt) {
        const int k = (int)by_n.div((uint32_t)e), j = e - k * n;
        double v[C];
        const T x = EXP ? T(0) : (T)node_of(ax[k], j, n, rule, glx);
        const int m = weighted_factor<FAM, T>(k, x, EXP ? tmp[e] : 0.0, EXP ? s_top[k] : 0,
                                              weight_of(rule, j, n, glw), p, v);
#pragma unroll
        for (int c = 0; c < C; ++c) tmp[c * total + e] = v[c];
        atomicMax(&s_exp[k], m);
    }
    __syncthreads();
    for (int e = tid; e < total; e += nt) {
        const int m = exp_or_zero(s_exp[by_n.div((uint32_t)e)]);
#pragma unroll
        for (int c = 0; c < C; ++c) axis[c * total + e] = (T)ldexp(tmp[c * total + e], -m);
    }
    __syncthreads();
    if (tid < d) s_exp[tid] = exp_or_zero(s_exp[tid]) + (EXP ? exp_or_zero(s_top[tid]) : 0);
    __syncthreads();
}

template <int FAM, typename T>
__device__ inline Factor<FAM, T> axis_factor(const T* axis, int total, int e) {
    Factor<FAM, T> f;
#pragma unroll
    for (int c = 0; c < Factor<FAM, T>::C; ++c) f.v[c] = axis[c * total + e];
    return f;
}

// Entries are read four at a time (16-byte LDS reads), so a loop of nl
// points is stored as ceil(nl / 4) groups, zeros after the last point.
constexpr int kGroup = 4;

template <int FAM, typename T>
struct EntryGroup {
    T v[Factor<FAM, T>::C][kGroup];
    __device__ inline void load(const T* tab, int entries, int g) {
        constexpr int V = 16 / (int)sizeof(T);
        using VT = __attribute__((ext_vector_type(V))) T;
#pragma unroll
        for (int c = 0; c < Factor<FAM, T>::C; ++c)
#pragma unroll
            for (int i = 0; i < kGroup / V; ++i) {
                const VT x = *reinterpret_cast<const VT*>(tab + (size_t)c * entries + g * kGroup + i * V);
#pragma unroll
                for (int j = 0; j < V; ++j) v[c][i * V + j] = x[j];
            }
    }
};

// Sum over the entries of groups [g0, g1) and the K states of a lane of
// their values, FP32 partials of at most 128 entries per state added to FP64.
// K states share each entry that is read from LDS: with one state the four
// SIMDs' reads of a 4-byte entry take 8 cycles of the CU's LDS against 2.7
// cycles of multiply-add, with four they take less than the arithmetic.
template <int FAM, typename T, int K>
__device__ inline double sum_entries(const Factor<FAM, T>* s, const T* tab, int entries, int g0, int g1) {
    constexpr int C = Factor<FAM, T>::C;
    constexpr int kFlushGroups = kFlush / kGroup;
    double acc = 0.0;
    for (int gb = g0; gb < g1; gb += kFlushGroups) {
        const int ge = gb + kFlushGroups < g1 ? gb + kFlushGroups : g1;
        T fa[K];
#pragma unroll
        for (int k = 0; k < K; ++k) fa[k] = T(0);
#pragma unroll 2
        for (int g = gb; g < ge; ++g) {
            EntryGroup<FAM, T> e;
            e.load(tab, entries, g);
#pragma unroll
            for (int i = 0; i < kGroup; ++i)
#pragma unroll
                for (int k = 0; k < K; ++k)
#pragma unroll
                    for (int c = 0; c < C; ++c) fa[k] = fma(s[k].v[c], e.v[c][i], fa[k]);
        }
#pragma unroll
        for (int w = K / 2; w > 0; w >>= 1)
#pragma unroll
            for (int k = 0; k < w; ++k) fa[k] += fa[k + w];
        acc += (double)fa[0];
    }
    return acc;
}

// ---- planning --------------------------------------------------------------
struct ProductGeom {
    int d, n, m, q, L;  // row axes [0, L), loop axes [L, L + q), lane axes [d - m, d)
    int rule, K;
    int nl, groups;     // loop points n^q and their groups of four
    int lane_count;     // n^m
    int lane_groups;    // ceil(n^m / (64 K))
    FastDiv by_n;
    long long items;    // rows * groups
    long long ipw;      // items per wave
    long long num_waves, blocks;
};

inline size_t product_axis_bytes(const ProductGeom& G, int C, int tsize) {
    return ((size_t)C * G.d * G.n * tsize + 15) & ~(size_t)15;
}
inline size_t product_lds_bytes(const ProductGeom& G, int C, int tsize) {
    const size_t tmp = G.n > kWaveAxis ? (size_t)C * G.d * G.n * sizeof(double) : 0;
    const size_t loop = (size_t)C * G.groups * kGroup * tsize;
    return product_axis_bytes(G, C, tsize) + (tmp > loop ? tmp : loop);
}

}  // namespace tq
