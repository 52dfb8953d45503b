// Device-side pieces of the kernels that run fp32 operands as three bf16 parts each: the split, and what to mistrust.
#pragma once
#include "conv_device.hpp"

namespace tdc {

typedef __bf16 bf8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf4_t __attribute__((ext_vector_type(4)));

// neither zero nor of a magnitude in [2^-90, infinity)
static __device__ __forceinline__ bool suspect(float sum) {
    const unsigned twice = __float_as_uint(sum) << 1;   // (without the sign)
    return twice - 2u * 0x12800000u >= 2u * (0x7f800000u - 0x12800000u) && twice != 0;
}
// Whether any of several sums is: two and a half vector instructions each.  (The total may overflow without any of them being
// infinite; then each is looked at in vain.)
struct Range {
    unsigned low = ~0u;
    float total = 0.0f;
    __device__ __forceinline__ void add(float sum) {
        low = min(low, (__float_as_uint(sum) << 1) - 1u);   // (zero: the largest)
        total += fabsf(sum);
    }
    __device__ __forceinline__ bool suspect() const { return low < 2u * 0x12800000u - 1u || !(total < __builtin_inff()); }
};

// What a thread has met among the values it split: whether any is below 2^-110 but not zero, and whether any reaches 2^20.  Two
// vector instructions a value (beside five for the split).
struct Extremes {
    unsigned low = ~0u;
    float high = 0.0f;
    template <int N>
    __device__ __forceinline__ void add(const float (&x)[N]) {
#pragma unroll
        for (int i = 0; i < N; i += 2) {
            low = min(min(low, (__float_as_uint(x[i]) << 1) - 1u), (__float_as_uint(x[i + 1]) << 1) - 1u);   // (zero: the largest)
            asm("v_max3_f32 %0, %1, |%2|, |%3|" : "=v"(high) : "v"(high), "v"(x[i]), "v"(x[i + 1]));   // (fmaxf would quiet each value first)
        }
    }
    __device__ __forceinline__ bool tiny() const { return low < 2u * 0x08800000u - 1u; }
    __device__ __forceinline__ bool large() const { return high >= 0x1p20f; }
};
constexpr int EXTREMES_FLOATS = 8;   // of LDS, in front of everything else: one word per wave

// x = h[0] + h[1] + h[2] exactly for finite x (8 bits of the mantissa each), as long as the lowest part stays representable.
// (Two values at a time: v_cvt_pk_bf16_f32 rounds both and leaves them where the operand registers want them; value by value the
// compiler converts each of them twice, seven vector instructions a value instead of five.)
template <int N, typename V>
static __device__ __forceinline__ void split3(const float (&x)[N], V (&h)[3]) {
    typedef __bf16 bf2_t __attribute__((ext_vector_type(2)));
    typedef unsigned words_t __attribute__((ext_vector_type(N / 2)));
    words_t w[3];
#pragma unroll
    for (int i = 0; i < N; i += 2) {
        f2_t r = {x[i], x[i + 1]};
#pragma unroll
        for (int s = 0; s < 3; ++s) {
            const unsigned both = __builtin_bit_cast(unsigned, __builtin_convertvector(r, bf2_t));
            w[s][i / 2] = both;
            r[0] -= __uint_as_float(both << 16);
            r[1] -= __uint_as_float(both & 0xffff0000u);
        }
    }
#pragma unroll
    for (int s = 0; s < 3; ++s) h[s] = __builtin_bit_cast(V, w[s]);
}

// Whether the split may have lost what counts in a sum of a channel with factor `scale` (below 0: it has tiny weights).
static __device__ __forceinline__ bool in_question(float sum, float scale, bool tiny_input, bool large_input) {
    const bool tiny_weights = scale < 0.0f;
    return suspect(sum) || (sum == 0.0f && (tiny_input || tiny_weights)) || (tiny_input && fabsf(scale) > 1.0f) || (large_input && tiny_weights);
}

}  // namespace tdc
