// fp32 numbers as exact sums of three bf16 parts (gptq_parts.hip)
#pragma once
#include "amct_common.h"

namespace amct {

constexpr int kPartsSum = 128;                      // steps of a sum before it is subtracted from W

// x = h + m + l; two values side by side in each word
AMCT_DEV void split_parts(float x0, float x1, uint32_t& h, uint32_t& m, uint32_t& l) {
    typedef float v2f __attribute__((ext_vector_type(2)));
    typedef __bf16 v2b __attribute__((ext_vector_type(2)));
    h = __builtin_bit_cast(uint32_t, __builtin_convertvector((v2f{x0, x1}), v2b));
    x0 = x0 - __uint_as_float(h << 16);
    x1 = x1 - __uint_as_float(h & 0xFFFF0000u);
    m = __builtin_bit_cast(uint32_t, __builtin_convertvector((v2f{x0, x1}), v2b));
    x0 = x0 - __uint_as_float(m << 16);
    x1 = x1 - __uint_as_float(m & 0xFFFF0000u);
    l = __builtin_bit_cast(uint32_t, __builtin_convertvector((v2f{x0, x1}), v2b));
}

// 0 or in [2^-100, 2^60): no part underflows, and no product or sum of the parts overflows
AMCT_DEV bool parts_hold(float x) {
    const uint32_t t = __float_as_uint(x) & 0x7FFFFFFFu;
    return t == 0 || (t >= (27u << 23) && t < (187u << 23));
}

}  // namespace amct
