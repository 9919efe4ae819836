// fp32 operands for the bf16 matrix cores: the exact three-way split and the six-term product step, shared by the dense
// products (om_gemm_s.hpp) and the 3x3 convolutions (om_conv3_s.hpp).
#pragma once

#include "om_internal.hpp"

namespace oms {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
// Global accesses of operands whose rows need not be 16-byte aligned (the hardware takes 4-byte alignment).
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float f2u __attribute__((ext_vector_type(2), aligned(4)));

// Operands are scaled by 2^24 before they are split and finished sums scaled back by 2^-48, both exactly: the lowest part of
// the smallest subnormal is then 2^-125, a normal bf16 value, so nothing of any operand below 2^104 is lost to bf16's range,
// whatever it is multiplied with. Larger ones become infinite, as sums of 2^80 do, and are recomputed (beyond()). The price is
// one multiplication beside the five and a half operations a value's split takes.
constexpr float kScale = 0x1p24f, kUnscale = 0x1p-48f;

// Two fp32 values, scaled, split into packed bf16 pairs, each part rounded to nearest. (v_dot2_f32_bf16 would give a residual
// in one instruction, but it shares the matrix pipe: beside an MFMA it costs 16 cycles, the unpack and subtraction 8.)
__device__ __forceinline__ uint32_t pack2(float x0, float x1) {
    const bf16x2 v = {(__bf16)x0, (__bf16)x1};
    return __builtin_bit_cast(uint32_t, v);
}
__device__ __forceinline__ void split2(float x0, float x1, uint32_t &h, uint32_t &m, uint32_t &l) {
    x0 *= kScale;
    x1 *= kScale;
    h = pack2(x0, x1);
    asm("" : "+v"(h));  // else the compiler converts x0 a second time instead of shifting h
    const float r0 = x0 - __uint_as_float(h << 16), r1 = x1 - __uint_as_float(h & 0xFFFF0000u);
    m = pack2(r0, r1);
    asm("" : "+v"(m));
    l = pack2(r0 - __uint_as_float(m << 16), r1 - __uint_as_float(m & 0xFFFF0000u));
}

// One lane's eight values of a fragment (16 k), as three MFMA operands.
struct Frag {
    u32x4 p[3];
    // Values 4 q .. 4 q + 3.
    __device__ __forceinline__ void set4(int q, const float *x) {
        uint32_t h, m, l;
        split2(x[0], x[1], h, m, l);
        p[0][2 * q] = h;
        p[1][2 * q] = m;
        p[2][2 * q] = l;
        split2(x[2], x[3], h, m, l);
        p[0][2 * q + 1] = h;
        p[1][2 * q + 1] = m;
        p[2][2 * q + 1] = l;
    }
};
__device__ __forceinline__ floatx16 mma(u32x4 a, u32x4 b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// One 16-k step of a 32 x 32 block: a's rows are the result's registers, b's its lanes. The five small terms go to `low`,
// hh to `acc`.
__device__ __forceinline__ void mma6(const u32x4 (&a)[3], const u32x4 (&b)[3], floatx16 &acc, floatx16 &low) {
    low = mma(a[1], b[1], low);
    low = mma(a[2], b[0], low);
    low = mma(a[0], b[2], low);
    low = mma(a[1], b[0], low);
    low = mma(a[0], b[1], low);
    acc = mma(a[0], b[0], acc);
}

// A finished block of sums, scaled back.
__device__ __forceinline__ void finish_sums(floatx16 &acc, const floatx16 &low) {
#pragma unroll
    for (int e = 0; e < 16; e++) acc[e] = (acc[e] + low[e]) * kUnscale;
}
// Whether a wavefront's finished sums hold one that the split could not carry: an operand or a sum past the scaled range
// leaves an infinity or a NaN. `big` collects over the sums of a lane (start at 0).
__device__ __forceinline__ void note(float v, unsigned &big) {
    const unsigned u = __float_as_uint(v) & 0x7FFFFFFFu;
    big = u > big ? u : big;
}
__device__ __forceinline__ bool beyond(unsigned big) { return __any(big >= 0x7F800000u); }
// Takes those sums, and only those, from `fp32`: a result depends on its own operands, not on what shares its wavefront.
__device__ __forceinline__ void take_beyond(floatx16 &acc, const floatx16 &fp32) {
#pragma unroll
    for (int e = 0; e < 16; e++) acc[e] = (__float_as_uint(acc[e]) & 0x7FFFFFFFu) >= 0x7F800000u ? fp32[e] : acc[e];
}

}  // namespace oms
