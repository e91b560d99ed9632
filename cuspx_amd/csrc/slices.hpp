// slices.hpp -- a launch cut so that none of its parts reaches the runtime's
// limit: HIP refuses gridDim.x * blockDim.x >= 2^32.
//
// A lane per WOTS chain reaches that within the device's memory: SHA2-128s
// signing at 34240 requests (71 GB of workspace), SHA2-192s at 23498, SHA2-128s
// key generation at 239675 keys, SHA2-128f signing at 697235 requests (206 GB).
// The cut is by requests, with the arguments' base addresses moved to the
// slice's first one (BatchArgs rows), so that the kernels know nothing of it:
// a first-workgroup argument changed k_chains' register assignment and cost it
// 1.4% (SHA2-128s, 200 requests).
#pragma once
#include <cstdint>

namespace spx {

constexpr uint64_t kSliceLanes = 1ull << 31;  // half: slices are equal to within a request

// f(first request, requests) for the slices of n requests whose launch has
// `lanes` lanes in all; no call for n = 0
template <class F>
inline void for_slices(uint32_t n, uint64_t lanes, const F& f) {
    const uint64_t c = n ? lanes / kSliceLanes + 1 : 0;
    for (uint64_t s = 0; s < c; s++) {
        const uint32_t a = (uint32_t)(n * s / c), b = (uint32_t)(n * (s + 1) / c);
        if (a < b) f(a, b - a);
    }
}

}  // namespace spx
