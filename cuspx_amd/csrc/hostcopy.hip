// hostcopy.hip -- copies between a lane's pinned host buffer and its device
// buffer on the lane's stream.
//
// Up to kKernelCopy bytes a kernel copies, 16 bytes a lane, reading or writing
// the host memory over the link itself: a copy engine's transfer adds a
// hand-over between queues on each side, which a small call waits for longer
// than for its bytes.  Host calls with the engine -> with the kernel, us:
// signing SHA2-128f 1 request 174 -> 133, 14 (234 KB out) 207 -> 168, 32 (534
// KB) 281 -> 242, 110 (1836 KB) 641 -> 602; SHAKE256-256f 1 314 -> 271;
// verifying SHA2-128f 1 558 -> 549, 64 and more no different.  Larger outputs
// are copied in pieces that overlap the host's own copies.
#include "engine.hpp"

namespace spx {

__global__ void __launch_bounds__(256) k_copy16(uint4* dst, const uint4* src, uint32_t n) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) dst[i] = src[i];
}

// bytes: a multiple of 16, as are both addresses; dst or src is host memory
// that the device can address
int host_copy(void* dst, const void* src, uint64_t bytes, hipMemcpyKind kind, hipStream_t s) {
    if (bytes == 0) return 0;
    if (bytes > kKernelCopy)
        return hipMemcpyAsync(dst, src, bytes, kind, s) == hipSuccess ? 0 : kErrHip;
    const uint32_t n = (uint32_t)(bytes / 16);
    (void)hipGetLastError();
    hipLaunchKernelGGL(k_copy16, dim3((n + 255) / 256), dim3(256), 0, s, (uint4*)dst,
                       (const uint4*)src, n);
    return hipGetLastError() == hipSuccess ? 0 : kErrHip;
}

}  // namespace spx
