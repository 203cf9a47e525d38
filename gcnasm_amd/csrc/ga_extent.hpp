// ga_extent.hpp -- the bytes that a buffer descriptor of a strided operand covers
// (plain C++, host and device).
#pragma once

#include <stdint.h>

#if defined(__HIP__) || defined(__HIPCC__)
#define GA_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define GA_HOST_DEVICE inline
#endif

namespace ga {

// `rows` rows (at least one) of `used` bytes, `ld` bytes apart: up to the last
// row's last used byte, not to the end of its stride, which a strided view's
// storage need not hold. The pipelined kernels copy a few K steps past K and
// read rows and columns past the last: whatever of that lies behind this extent
// comes back as zeros instead of from outside the operand. At most what a
// descriptor addresses, a multiple of 16 below 4 GiB.
constexpr GA_HOST_DEVICE uint32_t rows_bytes(long long rows, long long ld, long long used)
{
    const long long n = (rows - 1) * ld + used;
    return (uint32_t)(n > 0xFFFFFFF0ll ? 0xFFFFFFF0ll : n);
}

// The same for fp32 scale matrices, ld and used in floats, in 32 bits: the host
// has checked that they lie within 4 GiB.
constexpr GA_HOST_DEVICE uint32_t rows_bytes_f32(uint32_t rows, uint32_t ld, uint32_t used)
{
    return ((rows - 1) * ld + used) * 4u;
}

} // namespace ga
