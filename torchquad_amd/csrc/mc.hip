// Monte Carlo: counter-based sampling fused with the integrand and a block
// reduction of (sum f, sum f^2).  No sample ever touches HBM on the fused
// path; the point writer produces the identical stream for user integrands.
#include "tq_host.hpp"
#include "tq_values.hpp"

namespace tq {

constexpr int kMcFlush = 32;

template <typename T>
struct McArgs {
    int d;
    long long N;
    long long spt;  // samples per thread
    uint64_t seed, offset;
    const uint64_t* offset_dev;  // when set, the first counter is read from here
    const T* domain;
    double* partials;  // [blocks][2]
    Params<T> p;
};

// x[k] = lo + size u[k] of one sample.  FOLD (FP32): u[k] stays the integer
// u 2^24 and the size carries the 2^-24: the same product, one multiply per
// coordinate less.
template <int D, bool FOLD>
__device__ inline void mc_point(uint64_t seed, uint32_t c_lo, uint32_t c_hi, const float* lo, const float* sz,
                                float* x) {
#pragma unroll
    for (int k = 0; k < D; k += 4) {
        const u32x4 r = philox_block(seed, c_lo, c_hi, (uint32_t)(k / 4));
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (k + i < D) x[k + i] = fmaf(FOLD ? (float)(r.v[i] >> 8) : u01f(r.v[i]), sz[k + i], lo[k + i]);
    }
}
template <int D, bool FOLD>
__device__ inline void mc_point(uint64_t seed, uint32_t c_lo, uint32_t c_hi, const double* lo, const double* sz,
                                double* x) {
#pragma unroll
    for (int k = 0; k < D; k += 2) {
        const u32x4 r = philox_block(seed, c_lo, c_hi, (uint32_t)(k / 2));
#pragma unroll
        for (int i = 0; i < 2; ++i)
            if (k + i < D) x[k + i] = fma(u01d(r.v[2 * i], r.v[2 * i + 1]), sz[k + i], lo[k + i]);
    }
}

// The samples s0 .. s1-1 of a thread, in runs of one high counter word: the
// Philox products of that word leave the loop.
template <typename T, int FAM, int D, bool FOLD>
__device__ inline void mc_samples(const McArgs<T>& A, const T* lo, const T* sz, long long s0, long long s1,
                                  double& acc, double& acc2) {
    const uint64_t base = A.offset_dev ? *A.offset_dev : A.offset;
    while (s0 < s1) {
        const uint64_t c = base + (uint64_t)s0;
        const uint32_t c_lo = (uint32_t)c, c_hi = (uint32_t)(c >> 32);
        const uint32_t left = 0u - c_lo;  // samples to the next high word, 0: all 2^32
        int n = s1 - s0 < kMcFlush ? (int)(s1 - s0) : kMcFlush;
        if (left && left < (uint32_t)n) n = (int)left;
        T fa = T(0), fa2 = T(0);
        for (int i = 0; i < n; ++i) {
            T x[D];
            mc_point<D, FOLD>(A.seed, c_lo + (uint32_t)i, c_hi, lo, sz, x);
            const T f = eval_point<FAM, T, D>(x, D, A.p);
            fa += f;
            fa2 = fma(f, f, fa2);
        }
        acc += (double)fa;
        acc2 += (double)fa2;
        s0 += n;
    }
}

// D is exact (a bound of 4, 8 or 16 with run-time predicates cost two selects
// per coordinate).  Bound by the vector unit: 36 Philox multiplies at about 7
// cycles a wave and some 100 other operations per sample at d = 8.
// Dimensions above eight gain as well (4e6 samples: FP32 d = 12 41 -> 29 us, d =
// 16 49 -> 35 us; FP64 d = 16 111 -> 80 us).
// Oscillatory, d = 8, FP32, 1e8 samples: 400 us before, 285 us now (3-input xors, exact D, the high
// word's products and the 2^-24 out of the loop).
template <typename T, int FAM, int D>
__global__ __launch_bounds__(kBlock) void k_mc(McArgs<T> A) {
    __shared__ double s_red[kWavesPerBlock];
    T lo[D], sz[D];
    bool fold = sizeof(T) == 4;
#pragma unroll
    for (int k = 0; k < D; ++k) {
        lo[k] = A.domain[2 * k];
        sz[k] = A.domain[2 * k + 1] - A.domain[2 * k];
        // the scaled size is exact unless it leaves the normal range
        if constexpr (sizeof(T) == 4) fold = fold && sz[k] * 0x1.0p-24f * 0x1.0p24f == sz[k];
    }
    const long long gt = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long s0 = gt * A.spt;
    const long long s1 = (s0 + A.spt < A.N) ? (s0 + A.spt) : A.N;
    double acc = 0.0, acc2 = 0.0;
    if constexpr (sizeof(T) == 8) {
        mc_samples<T, FAM, D, false>(A, lo, sz, s0, s1, acc, acc2);
    } else if (fold) {
#pragma unroll
        for (int k = 0; k < D; ++k) sz[k] *= T(0x1.0p-24f);
        mc_samples<T, FAM, D, true>(A, lo, sz, s0, s1, acc, acc2);
    } else {
        mc_samples<T, FAM, D, false>(A, lo, sz, s0, s1, acc, acc2);
    }
    const double b1 = block_sum(acc, s_red);
    const double b2 = block_sum(acc2, s_red);
    if (threadIdx.x == 0) {
        A.partials[2 * blockIdx.x] = b1;
        A.partials[2 * blockIdx.x + 1] = b2;
    }
}

template <typename T>
__global__ __launch_bounds__(1024) void k_mc_finalize(const double* partials, long long nb, const T* domain,
                                                       int d, long long N, double c0, T* out, double* stats) {
    __shared__ double s_red[1024 / kWave];
    double v1 = 0.0, v2 = 0.0;
    for (long long i = threadIdx.x; i < nb; i += blockDim.x) {
        v1 += partials[2 * i];
        v2 += partials[2 * i + 1];
    }
    v1 = block_sum(v1, s_red);
    v2 = block_sum(v2, s_red);
    if (threadIdx.x == 0) {
        double vol = 1.0;
        for (int k = 0; k < d; ++k) vol *= (double)domain[2 * k + 1] - (double)domain[2 * k];
        const double r = c0 * vol * v1 / (double)N;
        if (out) *out = (T)r;
        if (stats) {
            stats[0] = c0 * vol * v1;
            stats[1] = c0 * c0 * vol * vol * v2;
            stats[2] = (double)N;
        }
    }
}

// The fused kernel's samples as [N, d] points.  MAXD: compile-time bound on
// the dimension, as in k_mc.  Staged writer (write_stage): the HBM writes
// bound it (d=7, FP32, 2e7 samples: 299 us with lane-strided 4-byte stores,
// 92 us or 6.1 TB/s so).
template <typename T, int MAXD>
__global__ __launch_bounds__(kBlock) void k_mc_points(const T* domain, int d, long long N, uint64_t seed,
                                                      uint64_t offset, int ppl, T* pts) {
    extern __shared__ __align__(16) unsigned char s_raw[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & (kWave - 1);
    const int C = kWave * ppl;
    T* slice = reinterpret_cast<T*>(s_raw) + (size_t)wave * C * d;
    T lo[MAXD], sz[MAXD];
#pragma unroll
    for (int k = 0; k < MAXD; ++k) {
        lo[k] = k < d ? domain[2 * k] : T(0);
        sz[k] = k < d ? domain[2 * k + 1] - lo[k] : T(0);
    }
    const long long chunks = (N + C - 1) / C;
    const long long stride = (long long)gridDim.x * kWavesPerBlock;
    for (long long c = (long long)blockIdx.x * kWavesPerBlock + wave; c < chunks; c += stride) {
        const long long first = c * C;
        const int points = N - first < C ? (int)(N - first) : C;
        for (int i = 0; i < ppl; ++i) {
            T u[MAXD];
            const int o = lane + kWave * i;
            Uniform<T>::template draw<MAXD>(seed, offset + (uint64_t)(first + o), d, u);
#pragma unroll
            for (int k = 0; k < MAXD; ++k)
                if (k < d) slice[o * d + k] = fma(u[k], sz[k], lo[k]);
        }
        wave_lds_fence();
        write_stage<T>(slice, pts, first, points, C, d);
        wave_lds_fence();  // the slice is read before the next chunk overwrites it
    }
}

// Unaligned outputs and few samples of one or two axes: one sample per
// thread, stored coordinate by coordinate.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_mc_points_any(const T* domain, int d, long long N, uint64_t seed,
                                                          uint64_t offset, T* pts) {
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (long long s = (long long)blockIdx.x * blockDim.x + threadIdx.x; s < N; s += stride) {
        T u[TQ_MAX_DIM];
        Uniform<T>::template draw<TQ_MAX_DIM>(seed, offset + (uint64_t)s, d, u);
#pragma unroll
        for (int k = 0; k < TQ_MAX_DIM; ++k) {
            if (k < d) {
                const T lo = domain[2 * k];
                const T sz = domain[2 * k + 1] - lo;
                pts[s * d + k] = fma(u[k], sz, lo);
            }
        }
    }
}

template <typename T>
static int launch_mc_points(const tq_mc_desc* m, const void* domain, void* points, hipStream_t st) {
    long long blocks = (m->N + kBlock - 1) / kBlock;
    const int ppl = stage_ppl(m->dim, sizeof(T), m->N, 1024);
    // one point per lane of one or two coordinates is as good as contiguous (1000 points, FP32: 2.3 us, staged 2.5)
    if ((ppl == 1 && m->dim <= 2) || !stage_fits(m->dim, sizeof(T), ppl, points)) {
        if (blocks > 65536) blocks = 65536;
        hipLaunchKernelGGL((k_mc_points_any<T>), dim3((unsigned)blocks), dim3(kBlock), 0, st, (const T*)domain,
                           m->dim, m->N, m->seed, m->offset, (T*)points);
        return check_launch("k_mc_points_any");
    }
    blocks = (blocks + ppl - 1) / ppl;
    if (blocks > 4096) blocks = 4096;
    const size_t lds = stage_bytes(m->dim, sizeof(T), ppl) * kWavesPerBlock;
#define TQ_MC_POINTS(MAXD)                                                                                        \
    hipLaunchKernelGGL((k_mc_points<T, MAXD>), dim3((unsigned)blocks), dim3(kBlock), lds, st, (const T*)domain,   \
                       m->dim, (long long)m->N, m->seed, m->offset, ppl, (T*)points)
    if (m->dim <= 4) TQ_MC_POINTS(4);
    else if (m->dim <= 8) TQ_MC_POINTS(8);
    else TQ_MC_POINTS(TQ_MAX_DIM);
#undef TQ_MC_POINTS
    return check_launch("k_mc_points");
}

// Generic-width uniform stream: row r, column c.
template <typename T>
__device__ inline T uniform_at(uint64_t seed, uint64_t row, int c);
template <>
__device__ inline float uniform_at<float>(uint64_t seed, uint64_t row, int c) {
    const u32x4 r = philox_block(seed, row, (uint32_t)(c >> 2));
    return u01f(r.v[c & 3]);
}
template <>
__device__ inline double uniform_at<double>(uint64_t seed, uint64_t row, int c) {
    const u32x4 r = philox_block(seed, row, (uint32_t)(c >> 1));
    return (c & 1) ? u01d(r.v[2], r.v[3]) : u01d(r.v[0], r.v[1]);
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_uniform(uint64_t seed, uint64_t offset, long long rows, int cols,
                                                    T* out) {
    const long long total = rows * (long long)cols;
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += stride) {
        const long long r = e / cols;
        const int c = (int)(e - r * cols);
        out[e] = uniform_at<T>(seed, offset + (uint64_t)r, c);
    }
}

// Mean of user values f[N, S]: the kernels of tq_values.hpp with unit weights.
template <typename T>
struct MeanScale {
    const T* domain;
    int d;
    long long N;
    __device__ double operator()() const {
        double vol = 1.0;
        for (int k = 0; k < d; ++k) vol *= (double)domain[2 * k + 1] - (double)domain[2 * k];
        return vol / (double)N;
    }
};

static long long mc_spt(const tq_mc_desc* m) {
    if (m->samples_per_thread > 0) return m->samples_per_thread;
    // aim for ~512K threads (8 waves per SIMD), at least 16 samples each
    long long spt = (m->N + (1LL << 19) - 1) >> 19;
    if (spt < 16) spt = 16;
    return spt;
}

static long long mc_blocks(const tq_mc_desc* m) {
    const long long spt = mc_spt(m);
    const long long threads = (m->N + spt - 1) / spt;
    long long b = (threads + kBlock - 1) / kBlock;
    return b < 1 ? 1 : b;
}

static int check_mc(const tq_mc_desc* m) {
    if (!m) return fail(TQ_E_NULL, "mc descriptor is NULL");
    if (m->dtype != TQ_F32 && m->dtype != TQ_F64) return fail(TQ_E_ARG, "dtype must be TQ_F32 or TQ_F64");
    if (m->dim < 1 || m->dim > TQ_MAX_DIM) return fail(TQ_E_ARG, "dim out of range (1..16)");
    if (m->N < 1) return fail(TQ_E_ARG, "N must be >= 1");
    if (mc_blocks(m) > 0x7fffffffLL) return fail(TQ_E_ARG, "N too large for one launch; raise samples_per_thread");
    return TQ_OK;
}

template <typename T, int FAM, int D = TQ_MAX_DIM>
static void launch_mc_dim(const McArgs<T>& A, long long nb, hipStream_t st) {
    if constexpr (D > 1) {
        if (A.d < D) return launch_mc_dim<T, FAM, D - 1>(A, nb, st);
    }
    hipLaunchKernelGGL((k_mc<T, FAM, D>), dim3((unsigned)nb), dim3(kBlock), 0, st, A);
}

template <typename T>
static int launch_mc(const tq_mc_desc* m, const tq_integrand* f, const void* domain, void* ws, size_t wsb,
                     void* out, double* stats, hipStream_t st, const uint64_t* offset_dev = nullptr) {
    const long long nb = mc_blocks(m);
    if (!ws || wsb < (size_t)nb * 2 * sizeof(double)) return fail(TQ_E_WORKSPACE, "mc workspace too small");
    McArgs<T> A;
    A.d = m->dim;
    A.N = m->N;
    A.spt = mc_spt(m);
    A.seed = m->seed;
    A.offset = m->offset;
    A.offset_dev = offset_dev;
    A.domain = (const T*)domain;
    A.partials = (double*)ws;
    A.p = make_params<T>(*f);
    TQ_DISPATCH_FAMILY(f->family, (launch_mc_dim<T, FAM>(A, nb, st)););
    int rc = check_launch("k_mc");
    if (rc) return rc;
    hipLaunchKernelGGL((k_mc_finalize<T>), dim3(1), dim3(1024), 0, st, (const double*)ws, nb, (const T*)domain,
                       m->dim, m->N, f->c0, (T*)out, stats);
    return check_launch("k_mc_finalize");
}

template <typename T>
static int launch_mean(const void* fv, long long N, long long S, const void* domain, int d, void* ws, size_t wsb,
                       void* out, hipStream_t st) {
    ValuePlan V;
    const int rc = plan_values(0, 1, 0, nullptr, N, S, (int)sizeof(T), V);
    if (rc) return rc;
    if (!ws || wsb < values_workspace(V)) return fail(TQ_E_WORKSPACE, "reduce workspace too small");
    return launch_values<T>(V, (const T*)fv, (double*)ws, MeanScale<T>{(const T*)domain, d, N}, (T*)out, st);
}

}  // namespace tq

using namespace tq;

extern "C" {

size_t tq_mc_workspace_size(const tq_mc_desc* m) {
    if (check_mc(m)) return 0;
    return (size_t)mc_blocks(m) * 2 * sizeof(double);
}

int tq_mc_integrate(const tq_mc_desc* m, const tq_integrand* f, const void* domain, void* workspace,
                    size_t workspace_bytes, void* out, double* stats, void* stream) {
    int rc = check_mc(m);
    if (rc) return rc;
    rc = check_integrand(f, m->dim);
    if (rc) return rc;
    if (!domain) return fail(TQ_E_NULL, "domain is NULL");
    if (!out && !stats) return fail(TQ_E_NULL, "no output pointer");
    if (m->dtype == TQ_F32)
        return launch_mc<float>(m, f, domain, workspace, workspace_bytes, out, stats, as_stream(stream));
    return launch_mc<double>(m, f, domain, workspace, workspace_bytes, out, stats, as_stream(stream));
}

int tq_mc_integrate_dev_offset(const tq_mc_desc* m, const tq_integrand* f, const void* domain,
                               const uint64_t* offset_dev, void* workspace, size_t workspace_bytes, void* out,
                               double* stats, void* stream) {
    int rc = check_mc(m);
    if (rc) return rc;
    rc = check_integrand(f, m->dim);
    if (rc) return rc;
    if (!domain || !offset_dev) return fail(TQ_E_NULL, "domain/offset_dev is NULL");
    if (!out && !stats) return fail(TQ_E_NULL, "no output pointer");
    if (m->dtype == TQ_F32)
        return launch_mc<float>(m, f, domain, workspace, workspace_bytes, out, stats, as_stream(stream), offset_dev);
    return launch_mc<double>(m, f, domain, workspace, workspace_bytes, out, stats, as_stream(stream), offset_dev);
}

int tq_mc_points(const tq_mc_desc* m, const void* domain, void* points, void* stream) {
    int rc = check_mc(m);
    if (rc) return rc;
    if (!domain || !points) return fail(TQ_E_NULL, "domain/points is NULL");
    if (m->dtype == TQ_F32) return launch_mc_points<float>(m, domain, points, as_stream(stream));
    return launch_mc_points<double>(m, domain, points, as_stream(stream));
}

size_t tq_mc_reduce_workspace_size(int64_t N, int64_t S) {
    if (N < 1 || S < 1) return 0;
    size_t most = 0;  // the data type sets the span's rounding: room for either
    for (int tsize = 4; tsize <= 8; tsize += 4) {
        ValuePlan V;
        if (plan_values(0, 1, 0, nullptr, N, S, tsize, V)) return 0;
        if (values_workspace(V) > most) most = values_workspace(V);
    }
    return most;
}

int tq_mc_reduce(int32_t dtype, const void* fvals, int64_t N, int64_t S, const void* domain, int32_t dim,
                 void* workspace, size_t workspace_bytes, void* out, void* stream) {
    if (dtype != TQ_F32 && dtype != TQ_F64) return fail(TQ_E_ARG, "dtype must be TQ_F32 or TQ_F64");
    if (N < 1 || S < 1 || S > 65535) return fail(TQ_E_ARG, "N/S out of range");
    if (dim < 1) return fail(TQ_E_ARG, "dim must be >= 1");
    if (!fvals || !domain || !out) return fail(TQ_E_NULL, "fvals/domain/out is NULL");
    if (dtype == TQ_F32)
        return launch_mean<float>(fvals, N, S, domain, dim, workspace, workspace_bytes, out, as_stream(stream));
    return launch_mean<double>(fvals, N, S, domain, dim, workspace, workspace_bytes, out, as_stream(stream));
}

int tq_uniform(uint64_t seed, uint64_t offset, int32_t dtype, int64_t rows, int32_t cols, void* out,
               void* stream) {
    if (dtype != TQ_F32 && dtype != TQ_F64) return fail(TQ_E_ARG, "dtype must be TQ_F32 or TQ_F64");
    if (rows < 0 || cols < 1) return fail(TQ_E_ARG, "rows/cols out of range");
    if (rows == 0) return TQ_OK;
    if (!out) return fail(TQ_E_NULL, "out is NULL");
    long long blocks = (rows * cols + kBlock - 1) / kBlock;
    if (blocks > 65536) blocks = 65536;
    if (dtype == TQ_F32)
        hipLaunchKernelGGL((k_uniform<float>), dim3((unsigned)blocks), dim3(kBlock), 0, as_stream(stream), seed,
                           offset, (long long)rows, (int)cols, (float*)out);
    else
        hipLaunchKernelGGL((k_uniform<double>), dim3((unsigned)blocks), dim3(kBlock), 0, as_stream(stream), seed,
                           offset, (long long)rows, (int)cols, (double*)out);
    return check_launch("k_uniform");
}

}  // extern "C"
