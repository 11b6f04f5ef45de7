// Transfers of the synchronous host-array calls. Each call's inputs sit in one pinned block that a
// kernel on the call's stream copies to the device, and its outputs come back the same way with the
// error word: one launch each instead of a blit per array, which from pageable memory also waits for
// the stream (eight rows of 4096 through the routed layer in mode B, host call: 629 -> 334 us with the
// bindings' conversion). Bound by the launches and, past a few hundred KB, by PCIe.
#include "pw_launch.h"

namespace pw {

// n 16-byte units; flags (optional) cleared
__global__ __launch_bounds__(256) void upload_kernel(const uint4 *__restrict__ host, uint4 *__restrict__ dev, uint32_t n,
                                                     uint32_t *flags)
{
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256)
        dev[i] = host[i];
    if (flags && blockIdx.x == 0 && threadIdx.x == 0)
        *flags = 0u;
}

// n 16-byte units; the error word to host_flags, then cleared
__global__ __launch_bounds__(256) void download_kernel(const uint4 *__restrict__ dev, uint4 *__restrict__ host, uint32_t n,
                                                       uint32_t *flags, uint32_t *host_flags)
{
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256)
        host[i] = dev[i];
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        *host_flags = *flags;
        *flags = 0u;
    }
}

static dim3 copy_grid(uint32_t n)
{
    const uint32_t wgs = (n + 255) / 256;
    return dim3(wgs < 1 ? 1 : wgs > 1024 ? 1024 : wgs);
}

void launch_upload(const void *host, void *dev, size_t bytes, uint32_t *flags, hipStream_t stream)
{
    const uint32_t n = (uint32_t)((bytes + 15) / 16);
    hipLaunchKernelGGL(upload_kernel, copy_grid(n), dim3(256), 0, stream, (const uint4 *)host, (uint4 *)dev, n, flags);
}

void launch_download(const void *dev, void *host, size_t bytes, uint32_t *flags, uint32_t *host_flags, hipStream_t stream)
{
    const uint32_t n = (uint32_t)((bytes + 15) / 16);
    hipLaunchKernelGGL(download_kernel, copy_grid(n), dim3(256), 0, stream, (const uint4 *)dev, (uint4 *)host, n, flags,
                       host_flags);
}

}  // namespace pw
