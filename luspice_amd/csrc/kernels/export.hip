// export.hip -- results to pinned host memory, with a word that says they are
// there (gfx950).
//
// The host waits for a handful of status words, or a small solution, at the end
// of every solve.  A copy through the runtime and hipStreamSynchronize take 15
// us (22 us more when the target is pageable); one kernel that stores the words
// to pinned memory and then a sequence number the host polls takes 11 us, and
// the wait alone 9 us instead of 12 (4 KB, measured behind a kernel of 3 us).
// The kernel runs after everything queued before it on the stream; the last
// workgroup to finish its part, by a counter that wraps, stores the number.
#include "common.hpp"
#include "launch.hpp"

namespace lsp {

constexpr int kExportWords = 1024;      // 4-byte words per workgroup

__global__ void __launch_bounds__(256) export_kernel(const unsigned *src, unsigned *dst, int words, unsigned *ctr,
                                                     unsigned long long *done, unsigned long long seq)
{
    const int w0 = blockIdx.x * kExportWords + threadIdx.x;
#pragma unroll
    for (int u = 0; u < kExportWords / 256; u++) {
        const int w = w0 + 256 * u;
        if (w < words) dst[w] = src[w];
    }
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0 && atomicInc(ctr, gridDim.x - 1) == gridDim.x - 1) {
        __threadfence_system();
        __hip_atomic_store(done, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

hipError_t launch_export(const void *src, void *dst, size_t bytes, unsigned *ctr, unsigned long long *done,
                         unsigned long long seq, hipStream_t st)
{
    const int words = (int)(bytes / 4);
    const int blocks = words > kExportWords ? (words + kExportWords - 1) / kExportWords : 1;
    hipLaunchKernelGGL(export_kernel, dim3(blocks), dim3(256), 0, st, (const unsigned *)src, (unsigned *)dst, words, ctr,
                       done, seq);
    return hipGetLastError();
}

}  // namespace lsp
