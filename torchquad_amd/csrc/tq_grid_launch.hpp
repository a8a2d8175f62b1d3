// What the fused grid kernels share: the workspace with its completion
// counters, the one-launch sum over workgroups and the device's CU count.
#pragma once
#include "tq_host.hpp"

namespace tq {

// Workspace of the fused kernels: completion counters in the first
// kWsHeader bytes (zero before the first launch, and every launch leaves
// them zero), then one FP64 partial per workgroup.  Workgroup b counts into
// group counter b % kDoneGroups; the last workgroup of each group counts
// into the top counter, whose last arrival sums the partials.  One counter
// for all workgroups serialised their atomics at about 15 ns each (10112
// workgroups: 148 us for 3.9e7 evaluations).
constexpr int kDoneGroups = 16;
constexpr int kDoneStride = 64;  // words between counters (256 bytes; 4 KB measured the same)
constexpr int kDoneTop = kDoneGroups * kDoneStride;
constexpr size_t kWsHeader = ((size_t)(kDoneTop + 1) * sizeof(unsigned int) + 255) & ~(size_t)255;

struct BlockSums {
    unsigned int* done;  // completion counters; zero between launches
    double* partials;
};

inline BlockSums block_sums(void* ws) {
    return BlockSums{(unsigned int*)ws, (double*)((unsigned char*)ws + kWsHeader)};
}

// x of the lane that DPP control CTRL selects; 0 where it selects none.
template <int CTRL, int ROW_MASK>
__device__ inline double dpp_from(double x) {
    union {
        double d;
        int i[2];
    } v, r;
    v.d = x;
    r.i[0] = __builtin_amdgcn_update_dpp(0, v.i[0], CTRL, ROW_MASK, 0xF, false);
    r.i[1] = __builtin_amdgcn_update_dpp(0, v.i[1], CTRL, ROW_MASK, 0xF, false);
    return r.d;
}

// Sum of the wave's lanes, valid in lane 63 only: DPP moves instead of the
// butterfly's twelve LDS permutes, whose latency a small launch waits for.
__device__ inline double wave_sum_last(double v) {
    v += dpp_from<0x111, 0xF>(v);  // row_shr 1, 2, 4, 8
    v += dpp_from<0x112, 0xF>(v);
    v += dpp_from<0x114, 0xF>(v);
    v += dpp_from<0x118, 0xF>(v);
    v += dpp_from<0x142, 0xA>(v);  // row_bcast15 into rows 1 and 3
    v += dpp_from<0x143, 0xC>(v);  // row_bcast31 into rows 2 and 3
    return v;
}

// Block sum in a fixed order (the waves' sums in wave order), valid in thread 0.
__device__ inline double block_sum_dpp(double v, double* s_red) {
    v = wave_sum_last(v);
    if ((threadIdx.x & (kWave - 1)) == kWave - 1) s_red[threadIdx.x >> 6] = v;
    __syncthreads();
    double r = 0.0;
    if (threadIdx.x == 0)
        for (int w = 0; w < (int)(blockDim.x >> 6); ++w) r += s_red[w];
    __syncthreads();
    return r;
}

// Sum of `acc` over every thread of the launch, in an order that does not
// depend on which workgroup is last.  Returns true in the workgroup that
// finishes last, whose thread 0 gets the sum; the counters are zero again
// when it returns.  Each workgroup stores its partial, releases it to device
// scope (an L2 write-back without the invalidate that a full fence would
// add) and counts; the last arrival of a group acquires its group's partials
// and releases them on to the top counter, so the final workgroup sees all.
__device__ inline bool sum_over_blocks(double acc, const BlockSums& S, double* s_red, double* sum) {
    __shared__ bool s_last;
    const int tid = threadIdx.x;
    const double bs = block_sum_dpp(acc, s_red);
    if (tid == 0) {
        S.partials[blockIdx.x] = bs;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        const unsigned nb = gridDim.x, grp = blockIdx.x % kDoneGroups;
        const unsigned members = (nb - 1 - grp) / kDoneGroups + 1;  // blocks b < nb with b % kDoneGroups == grp
        unsigned int* gc = S.done + grp * kDoneStride;
        bool last = false;
        if (__hip_atomic_fetch_add(gc, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == members - 1) {
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
            __hip_atomic_store(gc, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
            const unsigned groups = nb < (unsigned)kDoneGroups ? nb : (unsigned)kDoneGroups;
            last = __hip_atomic_fetch_add(S.done + kDoneTop, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
                   groups - 1;
        }
        s_last = last;
    }
    __syncthreads();
    if (!s_last) return false;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    double v = 0.0;
    for (unsigned i = tid; i < gridDim.x; i += blockDim.x) v += S.partials[i];
    v = block_sum_dpp(v, s_red);
    if (tid == 0) {
        *sum = v;
        __hip_atomic_store(S.done + kDoneTop, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    return true;
}

// CU count of the current device (0 if unknown), remembered per device.
inline int device_cus() {
    constexpr int kMax = 64;
    static int known[kMax] = {};  // a racing second writer stores the same value
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    if (dev >= 0 && dev < kMax && __atomic_load_n(&known[dev], __ATOMIC_RELAXED) > 0)
        return __atomic_load_n(&known[dev], __ATOMIC_RELAXED);
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    if (dev >= 0 && dev < kMax) __atomic_store_n(&known[dev], cus, __ATOMIC_RELAXED);
    return cus;
}

// grid_product.hip: the product kernel where it applies (`taken`).
template <typename T>
int launch_grid_product(const tq_grid_desc* gd, const tq_integrand* f, const void* domain, void* ws,
                        size_t ws_bytes, void* out, double* out64, hipStream_t st, bool* taken);

}  // namespace tq
