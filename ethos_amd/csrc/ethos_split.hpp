// A float32 value as three bf16 values, for exact products on the bf16 matrix cores.
#pragma once

#include "ethos_common.hpp"

namespace ethos {

// Two float32 values -> their three bf16 planes, one packed word each (a low, b high): the upper
// half (truncated, so that no finite value becomes an infinity), then the remainder and what is
// left of it, both to nearest; their sum is the value.  An infinity has zeros below it (against another
// operand's lower planes it still gives a NaN: such sums are taken again, gemm.hip); a NaN leaves
// one in the second plane.
__device__ __forceinline__ void split3(float a, float b, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
    const uint32_t ua = __float_as_uint(a), ub = __float_as_uint(b);
    hi = __builtin_amdgcn_perm(ub, ua, 0x07060302u);
    float ra = a - __uint_as_float(ua & 0xffff0000u), rb = b - __uint_as_float(ub & 0xffff0000u);
    ra = __builtin_isinf(a) ? 0.0f : ra;
    rb = __builtin_isinf(b) ? 0.0f : rb;
    mid = pack_bf16x2(ra, rb);
    lo = pack_bf16x2(ra - __uint_as_float(mid << 16), rb - __uint_as_float(mid & 0xffff0000u));
}

}  // namespace ethos
