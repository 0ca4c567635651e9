// Arithmetic of the 8-bit asymmetric layer that its kernels share (duq_int8.hip, duq_quant_gemm8.hip).
#pragma once
#include "duq_device.h"

namespace duq {

typedef float v4f32 __attribute__((ext_vector_type(4)));

constexpr int kQmaxAsym8 = 126;  // src/kernels/quant.cu:242

// clamp(rint(h(x / s)) + zi, 0, 126); the add wraps like the 32-bit add of the reference
__device__ __forceinline__ uint32_t asym8_code(float x, float s, int zi)
{
    const f16 hq = (f16)(x / s);  // IEEE float32 quotient, then one rounding to binary16
    const int qi = rint_i32((float)hq);
    const int sum = (int)((uint32_t)qi + (uint32_t)zi);
    return (uint32_t)clampi(sum, 0, kQmaxAsym8);
}
__device__ __forceinline__ int asym8_zero_int(float z) { return rint_i32((float)(f16)z); }

// Scale, zero point and code arithmetic of one row from its smallest and largest element (NaN if the row holds one).
//
// x / s has to be the float32 quotient, rounded once, and then rounded to binary16.  The division the compiler makes of it
// is a dozen instructions per element and was the longest of the quantizer's three phases (load, arithmetic, store).  A row
// has one divisor: y = 1 / s is computed once, q0 = x y is within 1.5 units in the last place, and q = q0 + (x - q0 s) y
// (Markstein, "Computation of elementary functions on the IBM RISC System/6000 processor", 1990) misses the correctly
// rounded quotient only where x / s is closer than 2^-21 such units to the middle between two float32 numbers.  After the
// rounding to binary16 that could show only beside the middle of two binary16 numbers; the pairs (x, s) with a quotient
// that close to such a place are few enough to try them all (tests/test_int8_quotient.py), and none is rounded otherwise.
// (No operand near the ends of the exponent range: `fast`.  Quotients so small that a remainder underflows give the code of
// zero either way.)
// From there two elements go together: both roundings to binary16 in one conversion, and in rows whose quotients stay
// below 500 (all but rows far off zero for their spread) the rounding to an integer is the addition of 1536, which leaves
// the integer in the low bits.  2048 x 4096 11.1 -> 8.4 us (5.0 TB/s), 512 x 11008 8.9 -> 7.3, 8 x 4096 3.2 -> 2.3.
struct RowCode8 {
    float s, z, y;
    int zi;
    bool fast;
    __device__ __forceinline__ RowCode8(float lo, float hi)
    {
        // scale = (max - min) / 127, zeros = round(-min / scale)  (quantizer.py:50-51), float32.  torch evaluates
        // tensor / scalar on a GPU as tensor * float32(1 / scalar), which is what the reference's scale is
        const float d = hi - lo;
        s = d * (1.0f / 127.0f);
        z = __builtin_rintf((-lo) / s);
        zi = asym8_zero_int(z);
        y = 1.0f / s;
        // (a NaN fails every comparison, an infinity the second)
        fast = s >= 0x1p-100f && s <= 0x1p100f && fmaxf(__builtin_fabsf(lo), __builtin_fabsf(hi)) <= 500.0f * s;
    }
    __device__ __forceinline__ float quotient(float x) const
    {
        const float q0 = x * y;
        float q = __builtin_fmaf(__builtin_fmaf(-q0, s, x), y, q0);
        asm("" : "+v"(q));  // round to float32 here, then to binary16 (no mixed multiply-add with a single rounding)
        return q;
    }
    __device__ __forceinline__ uint32_t quick4(const v4f32 g) const
    {
        const uint16_t off = (uint16_t)(0x6600 - zi);  // 0x6600: the bits of 1536
        v2us c[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const v2h h = v2h{(f16)quotient(g[2 * i]), (f16)quotient(g[2 * i + 1])} + v2h{(f16)1536.0f, (f16)1536.0f};
            c[i] = __builtin_elementwise_min(__builtin_elementwise_sub_sat(__builtin_bit_cast(v2us, h), v2us{off, off}),
                                             v2us{kQmaxAsym8, kQmaxAsym8});
        }
        return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, c[1]), __builtin_bit_cast(uint32_t, c[0]), 0x06040200u);
    }
    __device__ __forceinline__ uint32_t slow4(const v4f32 g) const
    {
        uint32_t w = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) w |= asym8_code(g[e], s, zi) << (8 * e);
        return w;
    }
};

// float32 dequant: x = (s_r * s_c) * (float(acc) - (z_r + z_c))
__device__ __forceinline__ float dequant_hprec_one(int acc, float sr, float zr, float sc, float zc)
{
    const float scales = sr * sc;
    const float zeros = zr + zc;
    const float t = (float)acc - zeros;
    return scales * t;  // built with -ffp-contract=off: no fused multiply-add
}

}  // namespace duq
