// Weight preparation: a row of a layer's weight -> its scale, zero point and packed codes in one pass (conversion of a
// torch.nn.Linear on the GPU; the arithmetic is that of the torch statements of the reference's from_linear / from_float,
// qlinear4bit/nn/linear.py:58-78, 123-145, 185-206, 262-297, 338-368, operator by operator).
//
// Bound by memory: 2 bytes read and half a byte written per element (4096 x 4096: 42 MB).  As torch operators the same
// work is a dozen passes and two host synchronizations, 0.38 ms; this kernel takes 22 us.  One workgroup per row, units of
// 8 elements (one 128-bit load, one 32-bit store), the row kept in registers between statistics and codes.  The
// dual-uniform layers quantize input columns below `split` with one pair of parameters and the others with a second.
#include "duq_launch.h"
#include "duq_rowquant.h"

namespace duq {

enum WeightKind { kAbs = 0, kShifted = 1, kGiven = 2 };
// kAbs     : asymmetric, statistics over |w| (scale = (max - min) / 15, zero = round(-min / scale)), codes 0..15 formed in
//            binary16: clamp(h(rint(h(w / scale)) + zero))
// kShifted : the activation quantizer's signed-shifted form (duq_quant.hip), statistics over w
// kGiven   : symmetric codes rint(w / scale) with the caller's scales, no clamp; `bad` is set where one is outside [-8, 7]

struct WeightParams {
    const uint16_t *w;  // [rows, cols] binary16
    uint8_t *q;         // [rows, cols / 2]
    uint16_t *s[2], *z[2];  // [rows] per column range (kGiven: s is read)
    int32_t *rowsum[2];     // kShifted: sum of the shifted codes of a range
    uint32_t rows, cols, split;
    int32_t *bad;
};

constexpr int kUnits = 8;  // units of a lane that stay in registers: rows of up to 16384 elements

template <int KIND>
__global__ __launch_bounds__(256) void weight_rows_kernel(WeightParams p)
{
    __shared__ float red[4][2][3];
    __shared__ int red_sum[4][2];
    const uint32_t tid = threadIdx.x, row = blockIdx.x, nunits = p.cols >> 3;
    const v4u *src = reinterpret_cast<const v4u *>(p.w + (uint64_t)row * p.cols);
    uint32_t *dst = reinterpret_cast<uint32_t *>(p.q + (uint64_t)row * (p.cols >> 1));
    const bool cached = nunits <= 256 * kUnits;
    auto elem = [](const v4u &g, int e) { return bits_to_f16((uint16_t)((e & 1) ? g[e >> 1] >> 16 : g[e >> 1] & 0xFFFFu)); };
    auto range_of = [&](uint32_t u, int e) { return u * 8 + e >= p.split ? 1 : 0; };

    v4u regs[kUnits];
    float mn[2] = {__builtin_inff(), __builtin_inff()}, mx[2] = {-__builtin_inff(), -__builtin_inff()};
    uint32_t am[2] = {0, 0};  // largest |w| bit pattern: above 0x7C00 there is a NaN, which fminf / fmaxf drop
    f16 s[2], z[2];
    float rcp[2];
    if (KIND != kGiven) {
        auto stat = [&](uint32_t u, const v4u &g) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const f16 v = elem(g, e);
                const uint32_t a = f16_to_bits(v) & 0x7FFFu;
                const float f = KIND == kAbs ? (float)bits_to_f16((uint16_t)a) : (float)v;
                const bool r = range_of(u, e);
                (r ? mn[1] : mn[0]) = fminf(r ? mn[1] : mn[0], f);
                (r ? mx[1] : mx[0]) = fmaxf(r ? mx[1] : mx[0], f);
                (r ? am[1] : am[0]) = max(r ? am[1] : am[0], a);
            }
        };
        if (cached) {
#pragma unroll
            for (int i = 0; i < kUnits; ++i) {
                const uint32_t u = tid + i * 256;
                if (u < nunits) regs[i] = __builtin_nontemporal_load(&src[u]);
            }
#pragma unroll
            for (int i = 0; i < kUnits; ++i)
                if (tid + i * 256 < nunits) stat(tid + i * 256, regs[i]);
        } else {
            for (uint32_t u = tid; u < nunits; u += 256) stat(u, src[u]);
        }
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const float a = wave_min_f32(mn[r]), b = wave_max_f32(mx[r]);
            const uint32_t m = wave_max_u32(am[r]);
            if ((tid & 63u) == 0) {
                red[tid >> 6][r][0] = a;
                red[tid >> 6][r][1] = b;
                red[tid >> 6][r][2] = __builtin_bit_cast(float, m);
            }
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            float a = red[0][r][0], b = red[0][r][1];
            uint32_t m = __builtin_bit_cast(uint32_t, red[0][r][2]);
#pragma unroll
            for (int w = 1; w < 4; ++w) {
                a = fminf(a, red[w][r][0]);
                b = fmaxf(b, red[w][r][1]);
                m = max(m, __builtin_bit_cast(uint32_t, red[w][r][2]));
            }
            if (m > 0x7C00u) a = b = __builtin_nanf("");
            const f16 lo = (f16)a, d = (f16)b - lo;  // (both exact binary16 values)
            float q15 = (float)d * (1.0f / 15.0f);
            asm volatile("" : "+v"(q15));
            s[r] = (f16)q15;
            rcp[r] = row_rcp(s[r]);
            float qz = (float)-lo * rcp[r];
            asm volatile("" : "+v"(qz));
            z[r] = (f16)__builtin_rintf((float)(f16)qz);
        }
        if (tid < 2 && (tid == 1 || p.split)) {
            const int o = p.split ? (int)tid : 0;  // (no split: the only range is the second, its parameters the first set)
            p.s[o][row] = f16_to_bits(tid ? s[1] : s[0]);
            p.z[o][row] = f16_to_bits(KIND == kShifted ? (tid ? z[1] : z[0]) - (f16)8.0f : (tid ? z[1] : z[0]));
        }
    } else {
        s[0] = bits_to_f16(p.s[0][row]);
        s[1] = p.split ? bits_to_f16(p.s[1][row]) : s[0];
        rcp[0] = row_rcp(s[0]);
        rcp[1] = row_rcp(s[1]);
    }
    const int zi[2] = {KIND == kShifted ? rint_i32((float)z[0]) : 0, KIND == kShifted ? rint_i32((float)z[1]) : 0};
    int sum[2] = {0, 0};
    bool bad = false;
    auto codes = [&](uint32_t u, const v4u &g) -> uint32_t {
        uint32_t word = 0;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const f16 v = elem(g, e);
            const bool r = range_of(u, e);
            uint32_t c;
            if (KIND == kShifted) {
                c = asym_code(v, r ? rcp[1] : rcp[0], r ? zi[1] : zi[0]) ^ 8u;
                (r ? sum[1] : sum[0]) += (int)(c << 28) >> 28;
            } else {
                float qf = (float)v * (r ? rcp[1] : rcp[0]);
                asm volatile("" : "+v"(qf));
                const f16 t = (f16)__builtin_rintf((float)(f16)qf);
                if (KIND == kAbs) {
                    c = (uint32_t)clampi(rint_i32((float)(f16)(t + (r ? z[1] : z[0]))), 0, 15);
                } else {
                    const int i = (int)(int8_t)cvt_i32_sat((float)t);  // (torch's conversion to int8)
                    bad = bad || i < -8 || i > 7;
                    c = (uint32_t)i & 15u;
                }
            }
            word |= c << (4 * e);
        }
        return word;
    };
    if (cached && KIND != kGiven) {
#pragma unroll
        for (int i = 0; i < kUnits; ++i) {
            const uint32_t u = tid + i * 256;
            if (u < nunits) dst[u] = codes(u, regs[i]);
        }
    } else {
        for (uint32_t u = tid; u < nunits; u += 256) dst[u] = codes(u, src[u]);
    }
    if (KIND == kGiven && bad) *p.bad = 1;  // (same value from every writer)
    if (KIND == kShifted) {
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const int t = wave_sum_i32(sum[r]);
            if ((tid & 63u) == 0) red_sum[tid >> 6][r] = t;
        }
        __syncthreads();
        if (tid < 2 && (tid == 1 || p.split)) p.rowsum[p.split ? tid : 0][row] = red_sum[0][tid] + red_sum[1][tid] + red_sum[2][tid] + red_sum[3][tid];
    }
}

// float32 weights -> int8 codes 0..127 over |w| (LinearQuant8bitASQ): units of 4 elements
__global__ __launch_bounds__(256) void weight_rows8_kernel(const float *w, uint32_t cols, int8_t *q, float *scale, float *zero)
{
    typedef float v4f_t __attribute__((ext_vector_type(4)));
    __shared__ float red[4][3];
    const uint32_t tid = threadIdx.x, row = blockIdx.x, nunits = cols >> 2;
    const v4f_t *src = reinterpret_cast<const v4f_t *>(w + (uint64_t)row * cols);
    uint32_t *dst = reinterpret_cast<uint32_t *>(q + (uint64_t)row * cols);
    v4f_t regs[kUnits];
    const bool cached = nunits <= 256 * kUnits;
    float mn = __builtin_inff(), mx = 0.f;
    uint32_t am = 0;
    auto stat = [&](const v4f_t &g) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float a = fabsf(g[e]);
            mn = fminf(mn, a);
            mx = fmaxf(mx, a);
            am = max(am, __builtin_bit_cast(uint32_t, a));
        }
    };
    if (cached) {
#pragma unroll
        for (int i = 0; i < kUnits; ++i)
            if (tid + i * 256 < nunits) regs[i] = __builtin_nontemporal_load(&src[tid + i * 256]);
#pragma unroll
        for (int i = 0; i < kUnits; ++i)
            if (tid + i * 256 < nunits) stat(regs[i]);
    } else {
        for (uint32_t u = tid; u < nunits; u += 256) stat(src[u]);
    }
    mn = wave_min_f32(mn);
    mx = wave_max_f32(mx);
    am = wave_max_u32(am);
    if ((tid & 63u) == 0) {
        red[tid >> 6][0] = mn;
        red[tid >> 6][1] = mx;
        red[tid >> 6][2] = __builtin_bit_cast(float, am);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        mn = fminf(mn, red[k][0]);
        mx = fmaxf(mx, red[k][1]);
        am = max(am, __builtin_bit_cast(uint32_t, red[k][2]));
    }
    if (am > 0x7F800000u) mn = mx = __builtin_nanf("");
    const float s = (mx - mn) * (float)(1.0 / 127.0);  // (torch multiplies by the reciprocal of a scalar divisor)
    const float z = __builtin_rintf(-mn / s);
    if (tid == 0) {
        scale[row] = s;
        zero[row] = z;
    }
    auto codes = [&](const v4f_t &g) {
        uint32_t word = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float t = __builtin_rintf(g[e] / s) + z;
            t = t != t ? t : fminf(fmaxf(t, 0.f), 127.f);
            word |= ((uint32_t)cvt_i32_sat(t) & 0xFFu) << (8 * e);
        }
        return word;
    };
    if (cached) {
#pragma unroll
        for (int i = 0; i < kUnits; ++i)
            if (tid + i * 256 < nunits) dst[tid + i * 256] = codes(regs[i]);
    } else {
        for (uint32_t u = tid; u < nunits; u += 256) dst[u] = codes(src[u]);
    }
}

int launch_weight_rows(int kind, const uint16_t *w, uint32_t rows, uint32_t cols, uint32_t split, uint8_t *q, uint16_t *s1,
                       uint16_t *z1, int32_t *r1, uint16_t *s2, uint16_t *z2, int32_t *r2, int32_t *bad, hipStream_t stream)
{
    const WeightParams p{w, q, {s1, s2}, {z1, z2}, {r1, r2}, rows, cols, split, bad};
    if (kind == kAbs)
        hipLaunchKernelGGL(weight_rows_kernel<kAbs>, dim3(rows), dim3(256), 0, stream, p);
    else if (kind == kShifted)
        hipLaunchKernelGGL(weight_rows_kernel<kShifted>, dim3(rows), dim3(256), 0, stream, p);
    else
        hipLaunchKernelGGL(weight_rows_kernel<kGiven>, dim3(rows), dim3(256), 0, stream, p);
    return (int)hipGetLastError();
}

int launch_weight_rows8(const float *w, uint32_t rows, uint32_t cols, int8_t *q, float *scale, float *zero, hipStream_t stream)
{
    hipLaunchKernelGGL(weight_rows8_kernel, dim3(rows), dim3(256), 0, stream, w, cols, q, scale, zero);
    return (int)hipGetLastError();
}

}  // namespace duq
