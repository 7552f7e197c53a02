// fp32 activations as bf16 MFMA operands: three bf16 terms per value.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace sa {

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

constexpr int kTerms = 3;   // |x - sum of the terms| <= 2^-27 |x|

// t_0 = rne(x), t_i = rne(x - t_0 - ... - t_{i-1}) of 8 values (each
// difference is exact in fp32).
__device__ __forceinline__ void split_terms(f32x4_t a, f32x4_t b, bf16x8_t (&t)[kTerms]) {
    f32x2_t v[4] = {{a[0], a[1]}, {a[2], a[3]}, {b[0], b[1]}, {b[2], b[3]}};
#pragma unroll
    for (int i = 0; i < kTerms; ++i) {
        u32x4_t packed;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const uint32_t bits = __builtin_bit_cast(uint32_t, __builtin_convertvector(v[e], bf16x2_t));
            packed[e] = bits;
            v[e] -= f32x2_t{__uint_as_float(bits << 16), __uint_as_float(bits & 0xffff0000u)};
        }
        t[i] = __builtin_bit_cast(bf16x8_t, packed);
    }
}

}  // namespace sa
