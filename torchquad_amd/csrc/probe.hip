// Measurement hooks: the attainable rate, on the device at hand, of the
// fused grid kernel's inner point loop and of the instructions it is made
// of.  bench.py states the grid kernel's rate against these.
#include "tq_host.hpp"

namespace tq {

constexpr int kProbeTable = 256;  // loop-table entries of the point-loop probe

// KIND 0: eight independent v_fma_f32 chains per lane; 1: eight v_exp_f32
// chains; 2, 3: the product grid loop's body -- a loop factor from LDS at a
// wave-uniform address and one multiply-add per point with each of the lane's
// own factors, four (2) or eight (3) of them.  Each trip is 32 instructions
// (0, 1), 1024 points (2) or 2048 (3).
template <int KIND>
__global__ __launch_bounds__(kBlock) void k_probe(float* out, int iters) {
    __shared__ float tab[kProbeTable];
    for (int j = threadIdx.x; j < kProbeTable; j += kBlock) tab[j] = 0.001f * (float)(j + 1);
    __syncthreads();
    float a[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) a[k] = 0.1f + 0.01f * (float)((threadIdx.x + k) & 31);
    float acc = 0.0f, sum[8] = {};
    for (int i = 0; i < iters; ++i) {
        if (KIND >= 2) {
#pragma unroll 8
            for (int j = 0; j < kProbeTable; ++j) {
                const float e = tab[j];
#pragma unroll
                for (int k = 0; k < 4 * (KIND - 1); ++k) sum[k & 7] = fmaf(a[k & 7], e, sum[k & 7]);
            }
            asm volatile("" ::: "memory");  // the table is read again on every trip
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
#pragma unroll
                for (int k = 0; k < 8; ++k)
                    a[k] = KIND == 0 ? fmaf(a[k], 0.999f, 0.0005f) : __builtin_amdgcn_exp2f(a[k]);
            }
        }
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) acc += a[k] + sum[k];
    out[(long long)blockIdx.x * kBlock + threadIdx.x] = acc;
}

}  // namespace tq

using namespace tq;

extern "C" int tq_probe_rates(int32_t kind, int64_t blocks, int32_t iters, float* out, void* stream) {
    if (!out) return fail(TQ_E_NULL, "out is NULL");
    if (kind < 0 || kind > 3) return fail(TQ_E_ARG, "kind must be 0, 1, 2 or 3");
    if (blocks < 1 || blocks > (1 << 20) || iters < 1 || iters > (1 << 20))
        return fail(TQ_E_ARG, "blocks and iters must be in 1..2^20");
    const hipStream_t s = as_stream(stream);
    if (kind == 0) hipLaunchKernelGGL(k_probe<0>, dim3((unsigned)blocks), dim3(kBlock), 0, s, out, iters);
    else if (kind == 1) hipLaunchKernelGGL(k_probe<1>, dim3((unsigned)blocks), dim3(kBlock), 0, s, out, iters);
    else if (kind == 2) hipLaunchKernelGGL(k_probe<2>, dim3((unsigned)blocks), dim3(kBlock), 0, s, out, iters);
    else hipLaunchKernelGGL(k_probe<3>, dim3((unsigned)blocks), dim3(kBlock), 0, s, out, iters);
    return check_launch("k_probe");
}
