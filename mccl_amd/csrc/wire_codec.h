// wire_codec.h -- the rounding of the wire codec, for every kernel that encodes: fp32 -> bf16, round to nearest
// even, NaN -> 0x7FC0 (torch/headeronly/util/BFloat16.h:100-114).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mcclx {
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// The result as the fp32 whose low half is zero.
__device__ __forceinline__ uint32_t bf16_round_bits(float x) {
    const uint32_t r = (uint32_t)__builtin_bit_cast(uint16_t, (__bf16)x) << 16;  // v_cvt_pk_bf16_f32
    return (x != x) ? 0x7FC00000u : r;
}
// Two values with one v_cvt_pk_bf16_f32, the first in the low half.  A NaN whose quiet bit is set (every NaN an
// add, a multiply or a decoded bf16 operand can hand over) converts to a NaN, which one is left open.
__device__ __forceinline__ uint32_t bf16_pair(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
}
// The same with every NaN made 0x7FC0.
__device__ __forceinline__ uint32_t bf16_encode_pair(float a, float b) {
    uint32_t r = bf16_pair(a, b);
    r = (a != a) ? (r & 0xFFFF0000u) | 0x7FC0u : r;
    return (b != b) ? (r & 0x0000FFFFu) | 0x7FC00000u : r;
}
}  // namespace mcclx
