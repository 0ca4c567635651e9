// Products of activations with long rows and few columns (attention probabilities against V: K is the context, N the head dimension),
// both operands in binary16: a launch that quantizes B, and one that quantizes A, multiplies and dequantizes.
//
// The rows of A are nearly all of the bytes.  As a quantizer launch and a batched GEMM they were read, written as codes and read again.
// Here a workgroup of eight wavefronts quantizes the 32 rows of its tile into LDS, as nibbles, and takes the codes of B, all columns of
// them, from the L2 in fragment order.  Two or three workgroups share a CU, so that one reads while another multiplies.
//
// What bounds it: the rows of A (32 x 2048 x 64 x 2048, 268 MB, in 54 us: 4.9 TB/s), and what the multiplications do not hide behind them
// (128 columns 69, 256 of half as many problems 47).  Against the two launches, asymmetric, us: those three 83.5 -> 54.3, 88.7 -> 69.6, 52.0
// -> 47.1; 32 x 1021 x 128 x 1024 29.5 -> 24.1, 8 x 1021 x 64 x 1024 13.2 -> 10.3, 8 x 4090 x 64 x 4096 77.5 -> 52.5, 8 x 4090 x 128 x 4096 79.1 -> 61.7.
// Tiles of 64 rows, two workgroups a CU: the first three 57.7, 72.3, 46.1, 8 x 1021 x 64 x 1024 13.1 (half the workgroups).  Two groups of
// rows requested ahead at two workgroups a CU: 58.2, 75.4, 51.4.  Workgroups that stay for several tiles and request the next tile's rows
// behind the last codes of B: 103, 114, 73, since loads return in their order and the multiplications come to wait for those rows.
#include <algorithm>

#include "duq_epilogue.h"
#include "duq_launch.h"
#include "duq_rowquant.h"
#include "duq_tiles.h"

namespace duq {

namespace {

typedef int v16i __attribute__((ext_vector_type(16)));

constexpr int kRows = 32;  // of A in a tile

// ---- B: LANES lanes a row, UNITS units of eight elements each.  Fragment order: per problem, tile of 32 rows and step of 64 elements a
// kilobyte, in which lane (r, h) of the product has bytes [16 * h, +16) of row r's 32.  Rows past N up to a whole tile hold anything.
struct TileQuantParams {
    const uint16_t *b;        // [batch, N, K]
    uint8_t *q;
    uint16_t *s, *z;          // [batch, N]
    uint32_t rows, N, K;
    float clip;
    int qmax;
};

template <int LANES, int UNITS, bool ASYM>
__global__ __launch_bounds__(256) void quantize_tiles_kernel(TileQuantParams p)
{
    const uint32_t row = blockIdx.x * (256 / LANES) + threadIdx.x / LANES, u0 = threadIdx.x % LANES, nunits = p.K / 8;
    const uint32_t from = min(row, p.rows - 1);
    const v4u *const x = reinterpret_cast<const v4u *>(p.b) + (uint64_t)from * nunits;
    v4u raw[UNITS];
#pragma unroll
    for (int j = 0; j < UNITS; ++j) raw[j] = x[min(u0 + j * LANES, nunits - 1)];
    RowQuant<ASYM, LANES == 64> rq;
    uint32_t w[UNITS];
    quantize_in_group<LANES>(raw, u0, nunits, p.clip, p.qmax, rq, w);
    if (row >= p.rows) return;
    const uint32_t problem = row / p.N, n = row % p.N, steps = p.K / 64;
    uint8_t *const to = p.q + ((uint64_t)problem * ((p.N + 31) / 32) + n / 32) * steps * 1024 + n % 32 * 16;
#pragma unroll
    for (int j = 0; j < UNITS; ++j) {
        const uint32_t c = u0 + j * LANES;
        if (c < nunits) *reinterpret_cast<uint32_t *>(to + c / 8 * 1024 + c / 4 % 2 * 512 + c % 4 * 4) = w[j];
    }
    if (u0 == 0) {
        p.s[row] = f16_to_bits(rq.s);
        if (ASYM) p.z[row] = f16_to_bits(rq.z);
    }
}

// Tiles of 32 columns that a workgroup has wavefronts for.
constexpr uint32_t long_column_tiles(uint32_t N) { return N <= 32 ? 1 : N <= 64 ? 2 : N <= 128 ? 4 : 8; }

// What a wavefront with column tile ct may read of its problem's codes: for tiles past the last (of four or eight, 65 to 96 and 129 to
// 224 columns have fewer) nothing, and every load gives zeros.
__host__ __device__ __forceinline__ uint32_t long_codes(uint32_t ct, uint32_t tiles, uint32_t steps) { return ct < tiles ? tiles * steps * 1024 : 0; }

// Where a lane finds its 16 bytes of step i.  Only the lane's offset is sure to be compared with the end of the codes, so it is what sends
// steps past the last out of range.
struct LongPiece {
    uint32_t lane_offset, offset;
};
__host__ __device__ __forceinline__ LongPiece long_piece(uint32_t lane, uint32_t ct, uint32_t i, uint32_t steps)
{
    return {i < steps ? lane * 16 : kOobOffset, i < steps ? (ct * steps + i) * 1024 : 0};
}

// The first 56 bytes (through reserved) reach the kernel in registers (DUQ_HEAD_DECL / with_head).
struct ProductLongParams {
    const uint16_t *a;        // [batch, M, K]
    const uint8_t *q;         // codes of B, in fragment order
    const uint16_t *s, *z;    // [batch, N]
    uint32_t M, N, K, tiles_m;
    uint32_t units;           // workgroups
    uint32_t reserved;
    uint16_t *y;              // [batch, M, N]
    float clip;
    int qmax;
};
static_assert(offsetof(ProductLongParams, y) == kHeadBytes, "the fields delivered in registers");

// LANES lanes a row of A, UNITS units each; CT tiles of 32 columns: the wavefronts split the columns, and what is left of eight the
// steps of K.
template <int LANES, int UNITS, int CT, bool ASYM>
__global__ __launch_bounds__(512, LANES * UNITS > 384 ? 4 : 6) void product_long_kernel(DUQ_HEAD_DECL, ProductLongParams tail)
{
    ProductLongParams p = with_head(tail, DUQ_HEAD_USE);
    to_global(p.a);
    to_global(p.q);
    to_global(p.s);
    to_global(p.z);
    to_global(p.y);
    constexpr int R = kRows, PASS = 512 / LANES, PASSES = R / PASS, KS = 8 / CT, MODE = ASYM ? 1 : 0;
    constexpr uint32_t kStride = LANES * UNITS * 4 + 16, kSum = (32 * CT + 4) * 4;  // bytes per row of codes and of sums: 4 dwords off a multiple of 8
    __shared__ __attribute__((aligned(16))) uint8_t lds[R * (kStride > kSum ? kStride : kSum)];
    __shared__ __attribute__((aligned(16))) uint16_t col_s[32 * CT], col_z[32 * CT], row_s[R], row_z[R];

    // every XCD a contiguous range of workgroups: one problem's codes of B in one L2
    const uint32_t each = p.units / 8, rem = p.units % 8, xcd = blockIdx.x % 8, local = blockIdx.x / 8;
    const uint32_t id = xcd < rem ? xcd * (each + 1) + local : rem * (each + 1) + (xcd - rem) * each + local;
    const uint32_t problem = id / p.tiles_m, m0 = id % p.tiles_m * R, rows = min(p.M - m0, (uint32_t)R);
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t l32 = lane & 31u, h = lane >> 5, nunits = p.K / 8, steps = p.K / 64;

    // ---- rows of A, PASS at a time (rows past the end of A: its last one again, stored by nobody; units past a row's: not counted)
    const v4u *const a = reinterpret_cast<const v4u *>(p.a) + ((uint64_t)problem * p.M + m0) * nunits;
    const uint32_t u0 = tid % LANES, r0 = tid / LANES;
    v4u raw[UNITS];
    auto fetch_a = [&](int pass) {
        const v4u *const row = a + (uint64_t)min(pass * PASS + r0, rows - 1) * nunits;
#pragma unroll
        for (int j = 0; j < UNITS; ++j) raw[j] = __builtin_nontemporal_load(row + min(u0 + j * LANES, nunits - 1));
    };
    fetch_a(0);
    if (tid < 32 * CT) {
        const uint32_t n = problem * p.N + min(tid, p.N - 1);
        col_s[tid] = p.s[n];
        if (ASYM) col_z[tid] = p.z[n];
    }

    // ---- codes of B: this wavefront's columns, steps ks, ks + KS, ..., four at a time (steps and whole tiles of columns past the end: zeros)
    const uint32_t ct = wave % CT, ks = wave / CT, tiles = (p.N + 31) / 32;
    const __amdgpu_buffer_rsrc_t rB = make_rsrc(p.q + (uint64_t)problem * tiles * steps * 1024, long_codes(ct, tiles, steps));
    v4u w[2][4];
    auto fetch_b = [&](v4u(&to)[4], uint32_t at) {
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            const LongPiece piece = long_piece(lane, ct, ks + (at + k) * KS, steps);
            to[k] = buf_load16(rB, piece.lane_offset, piece.offset);
        }
    };
#pragma unroll
    for (int pass = 0; pass < PASSES; ++pass) {
        RowQuant<ASYM, LANES == 64> rq;
        uint32_t codes[UNITS];
        quantize_in_group<LANES>(raw, u0, nunits, p.clip, p.qmax, rq, codes);
        if (pass + 1 < PASSES) fetch_a(pass + 1);
        if (pass == PASSES - 1) fetch_b(w[0], 0);
        const uint32_t r = pass * PASS + r0;
#pragma unroll
        for (int j = 0; j < UNITS; ++j)
            if (u0 + j * LANES < nunits) *reinterpret_cast<uint32_t *>(lds + r * kStride + (u0 + j * LANES) * 4) = codes[j];
        if (u0 == 0) {
            row_s[r] = f16_to_bits(rq.s);
            if (ASYM) row_z[r] = f16_to_bits(rq.z);
        }
    }
    lds_barrier();

    v16i acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0;
    constexpr uint32_t kNibbles = 0xF0F0F0F0u;
    auto multiply = [&](const v4u(&from)[4], uint32_t at) {
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            const uint32_t i = min(ks + (at + k) * KS, steps - 1);  // (past the end: B's codes are zeros)
            const v4i we = __builtin_bit_cast(v4i, (from[k] << 4) & kNibbles), wo = __builtin_bit_cast(v4i, from[k] & kNibbles);
            const v4u x = *reinterpret_cast<const v4u *>(lds + l32 * kStride + i * 32 + h * 16);
            acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(we, __builtin_bit_cast(v4i, (x << 4) & kNibbles), acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(wo, __builtin_bit_cast(v4i, x & kNibbles), acc, 0, 0, 0);
        }
    };
    const uint32_t mine = (steps + KS - 1) / KS;
#pragma unroll 1
    for (uint32_t at = 0; at < mine; at += 8) {
        fetch_b(w[1], at + 4);
        multiply(w[0], at);
        fetch_b(w[0], at + 8);
        multiply(w[1], at + 4);
    }
    lds_barrier();  // the codes are read: their place takes the sums

    // ---- a lane holds row l32, columns 8 * q + 4 * h + (0..3) of its 32
#pragma unroll
    for (int turn = 0; turn < (KS > 1 ? 2 : 1); ++turn) {
        if ((ks == 0) == (turn == 0)) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                int *const to = reinterpret_cast<int *>(lds + l32 * kSum) + ct * 32 + q * 8 + h * 4;
                if (turn == 0)
                    *reinterpret_cast<v4i *>(to) = v4i{acc[q * 4], acc[q * 4 + 1], acc[q * 4 + 2], acc[q * 4 + 3]};
                else
#pragma unroll
                    for (int r = 0; r < 4; ++r) __hip_atomic_fetch_add(to + r, acc[q * 4 + r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
        }
        lds_barrier();
    }
#pragma unroll
    for (int it = 0; it < (R * 4 * CT + 511) / 512; ++it) {
        const uint32_t i = it * 512 + tid, row = i / (4 * CT), n = i % (4 * CT) * 8;
        if (row >= rows || n >= p.N) continue;
        const RowEpi rp{bits_to_f16(row_s[row]), ASYM ? bits_to_f16(row_z[row]) : (f16)0, 0};
        const int *const sums = reinterpret_cast<const int *>(lds + row * kSum) + n;
        v4u out;
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            const v4i c = *reinterpret_cast<const v4i *>(sums + half * 4);
            const v2u s = *reinterpret_cast<const v2u *>(col_s + n + half * 4), z = ASYM ? *reinterpret_cast<const v2u *>(col_z + n + half * 4) : v2u{0u, 0u};
#pragma unroll
            for (int k = 0; k < 2; ++k)
                out[half * 2 + k] = dequant_pair_x256<MODE, false>(c[2 * k], c[2 * k + 1], rp, pair_cols_from_raw<MODE, false>(s, z, s, z, v2u{0u, 0u}, n, k));
        }
        store_row_piece(p.y + ((uint64_t)problem * p.M + m0 + row) * p.N + n, out, p.N - n);
    }
}

}  // namespace

// Both launches last as long as their longest chain, the quantizer of B and one tile, which grows with the rows' length and the columns,
// so the fewer the tiles the shorter the rows have to be; and the rows of B are quantized by fewer lanes than by the other quantizer, so those of
// A have to outnumber them.  Two launches / these, us: one problem 1 x 1021 x 64 x 1024 6.9 / 9.0, 1 x 4093 x 256 x 4096 20.7 / 23.5; 64 tiles of 1024
// elements 10.5 / 9.2, of 2048 on 128 columns 13.9 / 12.8, of 3072 16.3 / 17.1, of 2048 on 256 15.1 / 16.8; 128 of 3072 on 128 columns 20.5 / 19.2, of
// 2048 on 256 20.7 / 19.6, of 3072 on 256 24.0 / 25.2; 544 of 2176 on 256 36.5 / 39.1, 1024 of 4096 on 256 88.7 / 81.5; 32 x 64 x 128 x 2048 15.7 / 16.6.
bool product_long_takes(uint32_t batch, uint32_t M, uint32_t N, uint32_t K)
{
    if (K <= 256 || K > 4096 || K % 64 != 0 || N == 0 || N > 256 || M < 32 || batch < 2) return false;
    const uint64_t tiles = (uint64_t)batch * ((M + kRows - 1) / kRows);
    if (tiles >= (1u << 30) || M < (K <= 1536 ? N : 2 * N)) return false;
    return tiles >= (N <= 128 ? (K <= 2048 ? 64u : 128u) : K <= 1536 ? 64u : K <= 2048 ? 256u : 1024u);
}

// The end of what a workgroup reads of its problem's codes of B.
uint32_t product_long_reads(uint32_t N, uint32_t K)
{
    uint32_t end = 0;
    const uint32_t tiles = (N + 31) / 32, steps = K / 64, ct = long_column_tiles(N), ks = 8 / ct;
    for (uint32_t wave = 0; wave < 8; ++wave)
        for (uint32_t at = 0; at < (steps + ks - 1) / ks + 16; ++at) {  // (the ring requests up to sixteen steps past the last)
            const LongPiece piece = long_piece(63, wave % ct, wave / ct + at * ks, steps);
            if (piece.lane_offset < long_codes(wave % ct, tiles, steps)) end = std::max(end, piece.offset + piece.lane_offset + 16);
        }
    return end;
}

// q: codes of B, batch * ((N + 31) / 32 * 32) * (K / 2) bytes; s, z [batch, N].
int launch_product_long(bool asym, const uint16_t *a, const uint16_t *b, uint32_t batch, uint32_t M, uint32_t N, uint32_t K, float clip_a,
                        int qmax_a, float clip_b, int qmax_b, uint16_t *y, uint8_t *q, uint16_t *s, uint16_t *z, hipStream_t stream)
{
    if (!product_long_takes(batch, M, N, K)) return (int)hipErrorInvalidValue;
    const uint32_t lanes = K > 2048 ? 64 : K > 1024 ? 32 : 16;
    const TileQuantParams t{b, q, s, z, batch * N, N, K, clip_b, qmax_b};
    ProductLongParams p{a, q, s, z, M, N, K, (M + kRows - 1) / kRows, 0, 0, y, clip_a, qmax_a};
    p.units = batch * p.tiles_m;
    const dim3 quantizers((t.rows + 256 / lanes - 1) / (256 / lanes));
#define DUQ_LONG_CT(C) DUQ_LAUNCH_HEAD((product_long_kernel<decltype(l)::value, decltype(u)::value, C, decltype(zero_points)::value>), dim3(p.units), dim3(512), 0, stream, p)
    auto launch = [&](auto l, auto u, auto zero_points) {
        hipLaunchKernelGGL((quantize_tiles_kernel<decltype(l)::value, decltype(u)::value, decltype(zero_points)::value>), quantizers, dim3(256), 0, stream, t);
        if (const int e = (int)hipGetLastError()) return e;
        const uint32_t ct = long_column_tiles(N);
        if (ct == 1) DUQ_LONG_CT(1);
        else if (ct == 2) DUQ_LONG_CT(2);
        else if (ct == 4) DUQ_LONG_CT(4);
        else DUQ_LONG_CT(8);
        return (int)hipGetLastError();
    };
#undef DUQ_LONG_CT
#define DUQ_LONG(L, U) (asym ? launch(std::integral_constant<int, L>{}, std::integral_constant<int, U>{}, std::true_type{}) \
                             : launch(std::integral_constant<int, L>{}, std::integral_constant<int, U>{}, std::false_type{}))
    if (K <= 512) return DUQ_LONG(16, 4);
    if (K <= 1024) return DUQ_LONG(16, 8);
    if (K <= 1536) return DUQ_LONG(32, 6);
    if (K <= 2048) return DUQ_LONG(32, 8);
    if (K <= 3072) return DUQ_LONG(64, 6);
    return DUQ_LONG(64, 8);
#undef DUQ_LONG
}

}  // namespace duq
