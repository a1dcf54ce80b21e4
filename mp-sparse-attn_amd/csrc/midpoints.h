// Where a product of a 16-bit value and the pre-scale may lie next to a midpoint between two E2M1 values (quantize_kernel.h says what
// for).  No HIP in here: the host compiler builds it for its test.
#pragma once
#include <stdint.h>
#include <string.h>

// a value's bits, without sign, exponent and the first two mantissa bits, within 128 units of zeros
constexpr uint32_t MIDPOINT_NEAR = 128u << 11;

inline bool midpoint_pattern(float x) {
    uint32_t u;
    memcpy(&u, &x, 4);
    return (u << 11) + MIDPOINT_NEAR < 2 * MIDPOINT_NEAR;
}

// Whether no product of pre and a value of `digits` significant bits (bfloat16 8, float16 11) has the pattern: a product's mantissa
// depends on the two mantissas alone, and there are 128 or 1024 of the value's.  (Not looked at: products below float32's normal
// range, which are none of a block's whose scale is a normal float32.)
inline bool never_near_midpoint(float pre, int digits) {
    uint32_t u;
    memcpy(&u, &pre, 4);
    const uint32_t exponent = u >> 23 & 255u;
    if (exponent == 0u || exponent == 255u) return false;
    u = (u & 0x007FFFFFu) | 0x3F800000u;
    float p;
    memcpy(&p, &u, 4);
    bool near = false;
    for (int m = 1 << (digits - 1); m < 1 << digits; ++m) near |= midpoint_pattern((float)m * p);
    return !near;
}
