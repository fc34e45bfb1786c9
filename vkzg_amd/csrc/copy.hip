// Small copies between pinned host memory and device memory, by a kernel.
#include "kernels.h"

namespace vkzg_amd {

namespace {
constexpr uint32_t kThreads = 256;

__device__ __forceinline__ void copy_part(const CopyPart &p, uint32_t t, uint32_t n) {
    if (((reinterpret_cast<uintptr_t>(p.src) | reinterpret_cast<uintptr_t>(p.dst) | p.bytes) & 15u) == 0) {
        const uint4 *src = static_cast<const uint4 *>(p.src);
        uint4 *dst = static_cast<uint4 *>(p.dst);
        for (uint32_t i = t; i < p.bytes / 16; i += n) dst[i] = src[i];
    } else {
        const uint32_t *src = static_cast<const uint32_t *>(p.src);
        uint32_t *dst = static_cast<uint32_t *>(p.dst);
        for (uint32_t i = t; i < p.bytes / 4; i += n) dst[i] = src[i];
    }
}

// One load in flight per thread, 16 bytes each: the link's latency is the time.
__global__ void __launch_bounds__(kThreads) k_copy(CopyPart a, CopyPart b) {
    const uint32_t t = blockIdx.x * kThreads + threadIdx.x, n = gridDim.x * kThreads;
    copy_part(a, t, n);
    copy_part(b, t, n);
}
}  // namespace

hipError_t launch_copy(const CopyPart &a, const CopyPart &b, hipStream_t s) {
    if ((a.bytes | b.bytes) & 3u) return hipErrorInvalidValue;
    const size_t most = a.bytes > b.bytes ? a.bytes : b.bytes;
    if (most == 0) return hipSuccess;
    if (most >= kKernelCopyMax) return hipErrorInvalidValue;
    const uint32_t grid = (uint32_t)((most / 16 + kThreads - 1) / kThreads);
    hipLaunchKernelGGL(k_copy, dim3(grid ? grid : 1), dim3(kThreads), 0, s, a, b);
    return hipGetLastError();
}

}  // namespace vkzg_amd
