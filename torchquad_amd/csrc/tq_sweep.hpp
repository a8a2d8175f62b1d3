// What the parameter-sweep kernels share (grad.hip, sweep_product.hip).
#pragma once
#include "tq_grid_tile.hpp"

namespace tq {

constexpr int kSweepMaxD = 8;

// Parameters of integral b in the family's Params layout (as make_params
// builds them for one integrand): Gaussian peak a[b][d], u[b][d]; product
// peak a[b][d], u[b][d] (b_k = a_k^-2); oscillatory c[b][d] in a and w[b]
// in u (FP32 phase in revolutions, FP64 in radians).
template <typename T, int FAM>
__device__ inline void load_sweep_params(int d, int n, int rule, long long b, const T* a, const T* u, const T* dom,
                                         Params<T>* p, Axis* ax) {
    const double sl2e = 1.2011224087864498;  // sqrt(log2 e), as in make_params
    const int tid = threadIdx.x;
    if (tid < TQ_MAX_DIM) {
        T pa = T(0), pb = T(0), pu = T(0);
        if (tid < d) {
            const double ak = (double)a[b * d + tid];
            if (FAM == TQ_FAM_GAUSSIAN_PEAK) {
                const double uk = (double)u[b * d + tid];
                pa = (T)(ak * sl2e);
                pb = (T)(-ak * uk * sl2e);
                pu = (T)uk;
            } else if (FAM == TQ_FAM_PRODUCT_PEAK) {
                pa = (T)ak;
                pb = (T)(ak != 0.0 ? 1.0 / (ak * ak) : 0.0);
                pu = u[b * d + tid];
            } else {  // oscillatory
                pa = (T)(sizeof(T) == 4 ? ak / (2.0 * M_PI) : ak);
            }
            ax[tid] = make_axis(dom + b * 2 * d, tid, n, rule);
        }
        p->a[tid] = pa;
        p->b[tid] = pb;
        p->u[tid] = pu;
    }
    if (tid == 0) {
        p->c0 = T(1);
        p->c1 = p->c3 = T(0);
        p->c2 = T(0);
        if (FAM == TQ_FAM_OSCILLATORY) {
            const double w = (double)u[b];
            p->c2 = (T)(sizeof(T) == 4 ? w : 2.0 * M_PI * w);
        }
    }
}

// normalised node coordinate r in [-1, 1]
__device__ inline double node_r(int j, int n, int rule, const double* glx) {
    if (rule == TQ_RULE_GAUSS_LEGENDRE) return glx[j];
    return (n > 1) ? 2.0 * (double)j / (double)(n - 1) - 1.0 : 0.0;
}

// x = alpha r + beta on an axis (r the normalised node of node_r).
__device__ inline void loop_axis_affine(const Axis& ax, int n, int rule, double* alpha, double* beta) {
    if (rule == TQ_RULE_GAUSS_LEGENDRE) {
        *alpha = ax.a;
        *beta = ax.h;
    } else {
        *alpha = 0.5 * (ax.b - ax.a);
        *beta = 0.5 * (ax.b + ax.a);
    }
}

// Block partials per integral of the backward: Gaussian and product peak
// [F, three sums per axis], oscillatory [F, G, R_k].
inline int sweep_values(int family, int D) { return family == TQ_FAM_OSCILLATORY ? 2 + D : 1 + 3 * D; }

// sweep_product.hip: the factor-table form of the sweeps.  Blocks per
// integral (0: dimension, n or table sizes it does not take), the same for
// every family, so that one workspace size covers both directions.
long long sweep_product_blocks(const tq_grid_desc* g, int64_t B);
template <typename T, int FAM>
int launch_sweep_product_fwd(const tq_grid_desc* g, int64_t B, const void* a, const void* u, const void* dom,
                             double* partials, long long blocks, hipStream_t s);
// Gaussian and product peaks.
template <typename T, int FAM>
int launch_sweep_product_bwd(const tq_grid_desc* g, int64_t B, const void* a, const void* u, const void* dom,
                             double* partials, long long blocks, hipStream_t s);

}  // namespace tq
