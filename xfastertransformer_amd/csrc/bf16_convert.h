// fp32 -> bf16 narrowing as the reference's bfloat16_t assignment does it (include/bfloat16.h:40-65):
// round to nearest even on normals, subnormals flushed to signed zero, infinities kept, NaN quieted.
// Pure integer arithmetic on the bit pattern: what the host converts with, what the oracle's conversion is compared with over all 2^32 inputs, and what the
// device's own conversion (common.h) is compared with there.
#pragma once
#include <stdint.h>

#if defined(__HIPCC__)
#define XFT_HOST_DEVICE __host__ __device__
#else
#define XFT_HOST_DEVICE
#endif

namespace xfthip {

XFT_HOST_DEVICE inline uint16_t f32_bits_to_bf16_ref(uint32_t u) {
    const uint32_t a = u & 0x7FFFFFFFu;
    if (a > 0x7F800000u) return (uint16_t)((u >> 16) | 0x40u);
    if (a == 0x7F800000u) return (uint16_t)(u >> 16);
    if (a < 0x00800000u) return (uint16_t)((u >> 16) & 0x8000u);
    return (uint16_t)((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
}

} // namespace xfthip
