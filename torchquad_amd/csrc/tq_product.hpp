// Integrand values of the built-in families as products of per-axis factors.
//
// Every built-in family's value at a grid point is a short sum of products
// of one number per axis:
//   Gaussian peak     prod 2^(-t_k^2)                     1 component
//   exp-linear        prod 2^(a_k x_k)                    1
//   product peak      prod 1 / (a_k^-2 + (x_k - u_k)^2)   1
//   oscillatory       Re prod e^(i a_k x_k)               2 (complex product)
//   sin-sum           sum s_k                             2 (weight, sum)
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
// exponent for the result) and rounded to T once.  The largest factor of an
// axis is then in (1/4, 1]: of a family with one positive component and, each
// component by itself, of the double Gaussian (the smaller component's share
// goes to the first axis).  A partial product underflows only when the point
// is below 2^(2d - 126) (FP64: 2^(2d - 1022)) of the largest, so the form
// needs no range check and does not overflow where the sum of exponents did
// not.  The oscillatory and the sin-sum factors are scaled by the weights
// alone, which bound them.
#pragma once
#include "tq_grid_tile.hpp"

namespace tq {

constexpr bool family_exponential(int fam) { return fam == TQ_FAM_GAUSSIAN_PEAK || fam == TQ_FAM_EXP_LINEAR; }
// Exponents that a family's factors have by themselves: one, the double Gaussian one per component.
constexpr int family_exponents(int fam) { return family_exponential(fam) ? 1 : (fam == TQ_FAM_DOUBLE_GAUSSIAN ? 2 : 0); }
constexpr int family_comps(int fam) {
    return (fam == TQ_FAM_OSCILLATORY || fam == TQ_FAM_SIN_SUM || fam == TQ_FAM_DOUBLE_GAUSSIAN) ? 2 : 1;
}

// The sin-sum keeps the weights of row and lane axes out of its factors, in
// FP64, as the point-by-point kernel does; only the loop table carries its
// weights in T.  Rounded into FP32 factors, the weights of a Gauss-Legendre
// rule are off alike on every axis (error / sum |w f|, rms over d = 3..7:
// 3.3e-8 so, 0.7e-8 apart, 0.9e-8 point by point).  The other families'
// rounding errors differ from axis to axis and stay where the point-by-point
// kernel's are, and most need the weights inside for their range: weights may
// fall as fast as the factors rise.
constexpr bool weights_apart(int fam) { return fam == TQ_FAM_SIN_SUM; }

// log2 of an exponential family's factor; the constant term goes to axis 0.
// Kept within a 32-bit integer, far outside any result, so that exponents
// that cancel between axes do and overflow to infinity happens only in the
// result (NaN stays).
__device__ inline double bound_exponent(double e) { return e > 2e9 ? 2e9 : (e < -2e9 ? -2e9 : e); }
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
    return bound_exponent(e);
}

// Denominator of the product peak's factor on axis k.
template <typename T>
__device__ inline double peak_denominator(int k, T x, const Params<T>& p) {
    const double t = (double)x - (double)p.u[k];
    return fma(t, t, (double)p.b[k]);
}

// A node on which the product peak has a pole (a denominator of zero, or one
// whose reciprocal may leave the FP64 range).  Stored as it is, the infinite
// factor would meet the zeros of lanes and loop entries past the end and make
// NaN of an integral that is infinite; so its axis keeps the signs of the
// poles' weights alone, everything else on it counting for nothing beside
// them, and an exponent that takes any sum but 0 out of the range.
constexpr int kPoleExp = 1 << 27;  // above the product peak's other exponents
__device__ inline bool is_pole(double denominator) { return fabs(denominator) < 0x1.0p-1022; }

// log2 of the double Gaussian's factors, kept in range as factor_exponent's.
template <typename T>
__device__ inline void gauss_exponents(T x, const Params<T>& p, double* ex) {
    const double t1 = (double)x - (double)p.c1, t2 = (double)x - (double)p.c2, c = -(double)p.c3;
    ex[0] = bound_exponent(c * t1 * t1);
    ex[1] = bound_exponent(c * t2 * t2);
}

// Weighted factor of a family without exponents.
template <int FAM, typename T>
__device__ inline void factor_comps(int k, T x, double w, const Params<T>& p, double* v) {
    if constexpr (FAM == TQ_FAM_PRODUCT_PEAK) {
        v[0] = w / peak_denominator(k, x, p);
    } else if constexpr (FAM == TQ_FAM_OSCILLATORY) {
        double s, c;
        double phase = (double)p.a[k] * (double)x;  // FP32: revolutions, FP64: radians
        if (k == 0) phase += (double)p.c2;
        if (sizeof(T) == 4) sincospi(2.0 * phase, &s, &c);
        else sincos(phase, &s, &c);
        v[0] = w * c;
        v[1] = w * s;
    } else if constexpr (FAM == TQ_FAM_SIN_SUM) {
        v[0] = 1.0;
        v[1] = sin(fma((double)p.a[k], (double)x, (double)p.u[k]));
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
            r.v[0] = T(1);
            r.v[1] = a.v[1] + b.v[1];
        } else {
#pragma unroll
            for (int c = 0; c < C; ++c) r.v[c] = a.v[c] * b.v[c];
        }
        return r;
    }
    // the form in which an entry (of weight w, where that is kept apart) meets a state: value(merge(a, b)) =
    // sum_c a.v[c] * b.entry(w).v[c]; sin-sum: b.entry(w).v[0] * (a.v[1] + b.entry(w).v[1])
    __device__ inline Factor entry(double w) const {
        Factor r = *this;
        if constexpr (FAM == TQ_FAM_OSCILLATORY) r.v[1] = -v[1];
        if constexpr (FAM == TQ_FAM_SIN_SUM) r.v[0] = (T)w;
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

// Exponent that a node's weighted factor does not exceed by more than one,
// without evaluating the factor: the power of two that its axis is scaled by
// is the largest of these.
template <int FAM, typename T, bool POLES>
__device__ inline int factor_scale(int k, T x, double w, double ex, const Params<T>& p) {
    const int m = mag_exp(w);
    if (m == -0x7fffffff) return m;
    if constexpr (family_exponents(FAM) > 0) {
        return ex == ex ? m + (int)ceil(ex) : -0x7fffffff;
    } else if constexpr (FAM == TQ_FAM_PRODUCT_PEAK) {
        const double den = peak_denominator(k, x, p);
        if (POLES && is_pole(den)) return kPoleExp;
        const int e = mag_exp(den);
        return e == -0x7fffffff ? e : m - e + 1;
    } else {
        return m;
    }
}

// Powers of two taken out of the axes: s_exp[k] of axis k, of the double
// Gaussian's second component s_exp[TQ_MAX_DIM + k]; slots without an axis
// count as 0, so that a sum reads them all at once (axis by axis it waits for
// LDS d times: double Gaussian, 13^7 FP32 points, 16.2 us, 15.4 so).
constexpr int kExpSlots = 2 * TQ_MAX_DIM;
__device__ inline long long sum_exponents(const int* s_exp) {
    long long e = 0;
#pragma unroll
    for (int k = 0; k < TQ_MAX_DIM; ++k) e += exp_or_zero(s_exp[k]);
    return e;
}
__device__ inline double scale_by(double v, long long e) {
    return ldexp(v, (int)(e > (1 << 30) ? (1 << 30) : (e < -(1 << 30) ? -(1 << 30) : e)));
}

// A block's sum v with the powers of two put back that were taken out of its
// axes.  A pole on every axis: NaN, as from a sum over 0 times infinity.
__device__ inline double scale_back(int fam, double v, int d, const int* s_exp) {
    long long e = sum_exponents(s_exp);
    if (fam == TQ_FAM_DOUBLE_GAUSSIAN) {
        const long long e2 = sum_exponents(s_exp + TQ_MAX_DIM);
        if (e2 > e) e = e2;
    }
    if (fam == TQ_FAM_PRODUCT_PEAK) {
        int poles = 0;
#pragma unroll
        for (int k = 0; k < TQ_MAX_DIM; ++k) poles += s_exp[k] >= kPoleExp ? 1 : 0;
        if (poles == d) return __longlong_as_double(0x7ff8000000000000ll);
    }
    return scale_by(v, e);
}

// An axis's weights where they are kept apart, in the place of the component
// that is not stored (n FP64 numbers; d >= 2 axes of n numbers of T).
template <typename T>
__device__ inline double* apart_weights(const T* axis) {
    return const_cast<double*>(reinterpret_cast<const double*>(axis));
}

// Axis tables of a whole block: component c of axis k's node j goes to
// axis[c * d * n + k * n + j], the power of two taken out of axis k to
// s_exp[k].  The d n nodes are spread over the block's threads; the scales
// come from a first pass over them that evaluates no transcendental (an
// earlier form, one wave per axis with the factors in registers, left most
// lanes idle on short axes and evaluated long ones up to three times).  Ends
// with a barrier.
template <int FAM, typename T, bool POLES>
__device__ inline void build_axis_factors(int d, int n, int rule, const Axis* ax, const double* glx,
                                          const double* glw, const Params<T>& p, FastDiv by_n, T* axis, int* s_exp) {
    constexpr int C = family_comps(FAM);
    const int tid = threadIdx.x, nt = blockDim.x, total = d * n;
    constexpr int E = family_exponents(FAM);
    if (tid < kExpSlots) s_exp[tid] = -0x7fffffff;
    __syncthreads();
    struct Node {
        int k;
        T x;
        double w, ex[2];
    };
    auto node = [&](int e) {
        Node v;
        v.k = (int)by_n.div((uint32_t)e);
        const int j = e - v.k * n;
        v.x = (T)node_of(ax[v.k], j, n, rule, glx);
        v.w = weights_apart(FAM) ? 1.0 : weight_of(rule, j, n, glw);
        v.ex[0] = v.ex[1] = 0.0;
        if constexpr (E == 1) v.ex[0] = factor_exponent<FAM, T>(v.k, v.x, p);
        if constexpr (E == 2) gauss_exponents<T>(v.x, p, v.ex);
        return v;
    };
    auto scale = [&](const Node& v) {
        atomicMax(&s_exp[v.k], factor_scale<FAM, T, POLES>(v.k, v.x, v.w, v.ex[0], p));
        if constexpr (E == 2)
            atomicMax(&s_exp[TQ_MAX_DIM + v.k], factor_scale<FAM, T, POLES>(v.k, v.x, v.w, v.ex[1], p));
    };
    auto store = [&](const Node& nd, int e) {
        const int m = exp_or_zero(s_exp[nd.k]);
        double v[C];
        if constexpr (E == 1) {
            v[0] = nd.w * exp2(nd.ex[0] - (double)m);
        } else if constexpr (E == 2) {
            const int m2 = exp_or_zero(s_exp[TQ_MAX_DIM + nd.k]);
            // the first axis brings the components to the larger one's power of two
            const double behind = nd.k == 0 ? (double)(sum_exponents(s_exp) - sum_exponents(s_exp + TQ_MAX_DIM)) : 0.0;
            v[0] = nd.w * exp2(nd.ex[0] - (double)m + fmin(behind, 0.0));
            v[1] = nd.w * exp2(nd.ex[1] - (double)m2 - fmax(behind, 0.0));
        } else {
            factor_comps<FAM, T>(nd.k, nd.x, nd.w, p, v);
            if (FAM == TQ_FAM_PRODUCT_PEAK && POLES && m >= kPoleExp) {
                if (is_pole(peak_denominator(nd.k, nd.x, p))) v[0] = copysign(1.0, v[0]);
                else if (v[0] == v[0]) v[0] = 0.0;
            } else {
#pragma unroll
                for (int c = 0; c < C; ++c) v[c] = ldexp(v[c], -m);
            }
        }
#pragma unroll
        for (int c = FAM == TQ_FAM_SIN_SUM ? 1 : 0; c < C; ++c) axis[c * total + e] = (T)v[c];
    };
    // the thread's first node is kept over the barrier, later ones are formed again
    Node first = node(tid < total ? tid : total - 1);
    if constexpr (!weights_apart(FAM)) {
        if (tid < total) scale(first);
        for (int e = tid + nt; e < total; e += nt) scale(node(e));
        __syncthreads();
    }
    if (tid < total) store(first, tid);
    for (int e = tid + nt; e < total; e += nt) store(node(e), e);
    if constexpr (weights_apart(FAM))
        for (int j = tid; j < n; j += nt) apart_weights(axis)[j] = weight_of(rule, j, n, glw);
    __syncthreads();
}

template <int FAM, typename T>
__device__ inline Factor<FAM, T> axis_factor(const T* axis, int total, int e) {
    Factor<FAM, T> f = Factor<FAM, T>::one(true);
#pragma unroll
    for (int c = FAM == TQ_FAM_SIN_SUM ? 1 : 0; c < Factor<FAM, T>::C; ++c) f.v[c] = axis[c * total + e];
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

// The states' partial sums, joined in FP64 (joined in FP32, one rounding there
// would stand for 128 K points).
// w: the states' weights, where they are kept apart.
template <typename T, int K>
__device__ inline double join_states(const T* fa, const double* w = nullptr) {
    double r[K];
#pragma unroll
    for (int k = 0; k < K; ++k) r[k] = w ? w[k] * (double)fa[k] : (double)fa[k];
#pragma unroll
    for (int w = K / 2; w > 0; w >>= 1)
#pragma unroll
        for (int k = 0; k < w; ++k) r[k] += r[k + w];
    return r[0];
}

// Sum over the entries of groups [g0, g1) and the K states of a lane of
// their values, FP32 partials of at most 128 entries per state added to FP64.
// K states share each entry that is read from LDS: with one state the four
// SIMDs' reads of a 4-byte entry take 8 cycles of the CU's LDS against 2.7
// cycles of multiply-add, with four they take less than the arithmetic.
// Sin-sum: a value is formed before it is added.  As a sum of two products,
// weight and sine each multiplied through, one component is the same power of
// two on most entries and repeats one rounding along the loop, so the errors
// do not average out (FP32 Newton-Cotes rules, as above: 4e-8 so, 0.6e-8 here).
template <int FAM, typename T, int K>
__device__ inline double sum_entries(const Factor<FAM, T>* s, const double* wl, const T* tab, int entries, int g0,
                                     int g1) {
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
                for (int k = 0; k < K; ++k) {
                    if constexpr (FAM == TQ_FAM_SIN_SUM) {
                        fa[k] = fma(e.v[0][i], s[k].v[1] + e.v[1][i], fa[k]);
                    } else {
#pragma unroll
                        for (int c = 0; c < C; ++c) fa[k] = fma(s[k].v[c], e.v[c][i], fa[k]);
                    }
                }
        }
        if constexpr (weights_apart(FAM)) {
            acc += join_states<T, K>(fa, wl);
        } else {
            acc += join_states<T, K>(fa);
        }
    }
    return acc;
}

// Table of the combined factors of axes A .. A + q - 1 (q = 2: entry
// j1 n + j2), `count` of them, zeros from there to `entries`; LOOP: in the
// form that meets a state (Factor::entry).  Four entries per thread and trip: their reads go
// out together.  The caller's next barrier publishes it.
template <int FAM, typename T, bool LOOP>
__device__ inline void build_table(const T* axis, int total, int n, int A, int q, int count, int entries, FastDiv by_n,
                                   T* tab) {
    using F = Factor<FAM, T>;
    const int nt = blockDim.x;
    for (int e0 = threadIdx.x; e0 < entries; e0 += 4 * nt) {
        F f[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int e = e0 + i * nt;
            f[i] = F::one(false);
            if (e < count) {
                double w = 1.0;
                if (q == 2) {
                    const int j1 = (int)by_n.div((uint32_t)e);
                    if (LOOP && weights_apart(FAM)) w = apart_weights(axis)[j1] * apart_weights(axis)[e - j1 * n];
                    f[i] = F::merge(axis_factor<FAM, T>(axis, total, A * n + j1),
                                    axis_factor<FAM, T>(axis, total, (A + 1) * n + e - j1 * n));
                } else {
                    if (LOOP && weights_apart(FAM)) w = apart_weights(axis)[e];
                    f[i] = axis_factor<FAM, T>(axis, total, A * n + e);
                }
                if (LOOP) f[i] = f[i].entry(w);
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int c = 0; c < F::C; ++c)
                if (e0 + i * nt < entries) tab[c * entries + e0 + i * nt] = f[i].v[c];
    }
}

// How an integral's axes are split: row axes [0, L), loop axes [L, L + q),
// lane axes [L + q, d).  The outer one or two lane axes (`outer` of them, N
// combinations) are cut into K parts of H: a lane holds one combination of
// the inner lane axes and K of the outer ones, f, f + H, f + 2 H, ..., so its
// states share everything but one table entry.  (Spreading the K states over
// consecutive combinations cost digits for every state and axis: an eighth of
// the instructions of an 8192-integral batch.)
struct ProductSplit {
    int d, n, L, q;
    int outer, inner;   // lane axes: outer (1 or 2) and inner ones
    int N, H;           // outer combinations, and per state
    int nl, groups;     // loop points n^q and their groups of four
    int slots;          // H * n^inner
    int lane_groups;    // ceil(slots / 64)
    FastDiv by_n;
    long long items;    // rows * groups
};

// LDS tables of a split: every axis's factors, the loop table, and the outer
// table when two axes are combined there.
template <typename T>
struct ProductTables {
    T* axis;
    T* loop;
    T* outer;  // component c of outer combination f: outer[c * outer_stride + f]
    int outer_stride;
};

__host__ __device__ inline size_t round16(size_t b) { return (b + 15) & ~(size_t)15; }
__host__ __device__ inline size_t product_lds_bytes(const ProductSplit& S, int C, int tsize) {
    return round16((size_t)C * S.d * S.n * tsize) + round16((size_t)C * S.groups * kGroup * tsize) +
           (S.outer == 2 ? (size_t)C * S.N * tsize : 0);
}

// Builds them (all threads of the block; ends with a barrier).  POLES: an
// infinite factor as the sign of its weight (kPoleExp), for scale_back.
template <int FAM, typename T, bool POLES = true>
__device__ inline ProductTables<T> build_product_tables(const ProductSplit& S, int rule, const Axis* ax,
                                                        const double* glx, const double* glw, const Params<T>& p,
                                                        unsigned char* lds, int* s_exp) {
    constexpr int C = family_comps(FAM);
    const int total = S.d * S.n, entries = S.groups * kGroup;
    ProductTables<T> t;
    t.axis = reinterpret_cast<T*>(lds);
    const size_t a = ((size_t)C * total * sizeof(T) + 15) & ~(size_t)15;
    t.loop = reinterpret_cast<T*>(lds + a);
    build_axis_factors<FAM, T, POLES>(S.d, S.n, rule, ax, glx, glw, p, S.by_n, t.axis, s_exp);
    build_table<FAM, T, true>(t.axis, total, S.n, S.L, S.q, S.nl, entries, S.by_n, t.loop);
    if (S.outer == 2) {
        t.outer = reinterpret_cast<T*>(lds + a + (((size_t)C * entries * sizeof(T) + 15) & ~(size_t)15));
        t.outer_stride = S.N;
        build_table<FAM, T, false>(t.axis, total, S.n, S.L + S.q, 2, S.N, S.N, S.by_n, t.outer);
    } else {
        t.outer = t.axis + (S.L + S.q) * S.n;
        t.outer_stride = total;
    }
    __syncthreads();
    return t;
}

// The K states of lane slot `slot`, and their weights where they are kept
// apart; zeros where there is no combination.
template <int FAM, typename T, int K>
__device__ inline void lane_states(const ProductSplit& S, const ProductTables<T>& t, int slot, Factor<FAM, T>* own,
                                   double* wl) {
    using F = Factor<FAM, T>;
    const bool on = slot < S.slots;
    uint32_t r = on ? (uint32_t)slot : 0u;
    F common = F::one(true);
    double w = 1.0;
    for (int a = S.d - 1; a >= S.d - S.inner; --a) {
        const uint32_t q = S.by_n.div(r);
        const int j = (int)(r - q * S.by_n.n);
        common = F::merge(common, axis_factor<FAM, T>(t.axis, S.d * S.n, a * S.n + j));
        if constexpr (weights_apart(FAM)) w *= apart_weights(t.axis)[j];
        r = q;
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int f = (int)r + k * S.H;
        const bool has = on && f < S.N;
        F o = axis_factor<FAM, T>(t.outer, t.outer_stride, has ? f : 0);
        o = F::merge(common, o);
#pragma unroll
        for (int c = 0; c < F::C; ++c) own[k].v[c] = has ? o.v[c] : T(0);
        if constexpr (weights_apart(FAM)) {
            const int j1 = S.outer == 2 ? (int)S.by_n.div((uint32_t)(has ? f : 0)) : (has ? f : 0);
            double wo = apart_weights(t.axis)[j1];
            if (S.outer == 2) wo *= apart_weights(t.axis)[(has ? f : 0) - j1 * S.n];
            wl[k] = has ? w * wo : 0.0;
        }
    }
}

// Sum over the wave-uniform items [t0, t1) of the K states' values: item t is
// group t mod `groups` of the loop table on row t / groups, whose factor (of
// the axes [0, L)) is merged into the states.
template <int FAM, typename T, int K>
__device__ inline double sum_items(const ProductSplit& S, const ProductTables<T>& t, const Factor<FAM, T>* own,
                                   const double* wl, long long t0, long long t1) {
    using F = Factor<FAM, T>;
    const int lane = threadIdx.x & (kWave - 1), n = S.n, L = S.L, groups = S.groups, entries = groups * kGroup;
    if (L == 0) return sum_entries<FAM, T, K>(own, wl, t.loop, entries, (int)t0, (int)t1);
    // row odometer: lane k of `dig` holds the digit of row axis k
    long long row = t0 / groups;
    int gi = (int)(t0 - row * groups);
    int dig = 0;
    for (int k = L - 1; k >= 0; --k) {
        const long long q = row / n;
        dig = lane == k ? (int)(row - q * n) : dig;
        row = q;
    }
    double acc = 0.0;
    for (long long at = t0; at < t1;) {
        F rf = F::one(true);
        double rw = 1.0;
        for (int k = 0; k < L; ++k) {
            const int j = __builtin_amdgcn_readlane(dig, k);
            rf = F::merge(rf, axis_factor<FAM, T>(t.axis, S.d * n, k * n + j));
            if constexpr (weights_apart(FAM)) rw *= apart_weights(t.axis)[j];
        }
        F s[K];
#pragma unroll
        for (int k = 0; k < K; ++k) s[k] = F::merge(own[k], rf);
        const int left = groups - gi;
        const int ge = t1 - at < left ? gi + (int)(t1 - at) : groups;
        const double part = sum_entries<FAM, T, K>(s, wl, t.loop, entries, gi, ge);
        if constexpr (weights_apart(FAM)) acc = fma(rw, part, acc);
        else acc += part;
        at += ge - gi;
        gi = 0;
        for (int k = L - 1; k >= 0; --k) {
            const int dk = __builtin_amdgcn_readlane(dig, k) + 1;
            const bool wrap = dk >= n;
            dig = lane == k ? (wrap ? 0 : dk) : dig;
            if (!wrap) break;
        }
    }
    return acc;
}

// The split of a d-axis integral with K states per lane that has the least
// work, counted in instructions per wave: the multiply-adds of the (padded)
// groups, the states' set-up once per lane group, and the merges, digits and
// flush once per row.  max_entries: longest loop table; max_outer: longest
// combined outer table; lane_axes > 0 fixes the number of lane axes; max_q:
// loop axes at most.  False: no split fits lds_max bytes of tables.
inline bool split_product_axes(int d, int n, int K, int C, int tsize, long long max_entries, long long max_outer,
                               int lane_axes, size_t lds_max, ProductSplit& S, int max_q = 2) {
    if (d < 2 || n < 2) return false;
    double best = -1.0;
    double power[TQ_MAX_DIM + 1];  // n^i (the host plans thousands of integrals a batch: no libm calls here)
    power[0] = 1.0;
    for (int i = 1; i <= d; ++i) power[i] = power[i - 1] * n;
    for (int q = 1; q <= max_q && q < d; ++q) {
        const long long nl = q == 2 ? (long long)n * n : n, groups = (nl + kGroup - 1) / kGroup;
        if (groups * kGroup > max_entries) break;
        for (int m = 1; m <= d - q; ++m) {
            if (lane_axes > 0 && m != lane_axes) continue;
            for (int outer = 1; outer <= 2 && outer <= m; ++outer) {
                const long long N = outer == 2 ? (long long)n * n : n;
                if (outer == 2 && N > max_outer) break;
                const long long H = (N + K - 1) / K;
                if ((double)H * power[m - outer] > (double)(1 << 30)) break;
                const long long slots = H * (long long)power[m - outer], lane_groups = (slots + kWave - 1) / kWave;
                const int L = d - q - m;
                constexpr int kFlushGroups = kFlush / kGroup;
                const long long row = groups * kGroup * K * C + (L > 0 ? 30 + 8 * L + 2 * K * C : 0) +
                                      (groups + kFlushGroups - 1) / kFlushGroups * 8;
                const long long init = 20 + 12 * (m - outer) + K * (5 + 3 * C);
                const double work = (double)lane_groups * ((double)init + power[L] * (double)row);
                if (best >= 0.0 && work >= best) continue;
                ProductSplit X;
                X.d = d;
                X.n = n;
                X.L = L;
                X.q = q;
                X.outer = outer;
                X.inner = m - outer;
                X.N = (int)N;
                X.H = (int)H;
                X.nl = (int)nl;
                X.groups = (int)groups;
                if (product_lds_bytes(X, C, tsize) > lds_max) continue;
                X.slots = (int)slots;
                X.lane_groups = (int)lane_groups;
                long long r;
                if (ipow_checked(n, L, (1LL << 62) / X.groups, &r) != 0) continue;
                X.items = r * X.groups;
                best = work;
                S = X;
            }
        }
    }
    S.by_n = make_fast_div((uint32_t)n);
    return best >= 0.0;
}

}  // namespace tq
