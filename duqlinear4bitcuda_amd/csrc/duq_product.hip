// Products of activations with short rows (attention scores: K is the head dimension, 64 to 256), both operands in binary16:
// quantizers, int4 product and dequant in one launch (duq_quantize_product).
//
// A workgroup of eight wavefronts owns 256 rows of B (output columns) and a run of row tiles of A, 64 rows each.  Every wavefront
// quantizes the rows of B of its own 32 columns once and keeps their codes as MFMA fragments in registers; then the workgroup takes tile
// after tile of A: the rows of the tiles to come (two at a time, four lanes to a row, where a row's registers allow it) are requested before
// the MFMAs of this one, and quantized after its outputs were staged and before they are stored.  The codes are bytes from the
// beginning: nibbles would be packed and expanded again.
//
// What bounds it is the outputs' stores, 32 KB a tile (32 products of 2048 x 2048 x 128: 268 MB in 55 us; with the stores left out some 40,
// without the quantizer 57, in the form of four wavefronts); the vector work beside them is the dequant, 3.5 instructions per output,
// and the quantizer, four per element of A once per 256 columns.  A launch of one workgroup per tile (gemm_s4_shortk_kernel) that
// a quantizer launch precedes waits for its operands at the head of every tile, and its stores do not begin before the quantizer has
// ended.  Against that, asymmetric and symmetric, us: 32 x 2048 x 2048 x 128 71.4 -> 55.2 and 70.2 -> 54.0, x 64 61.9 -> 52.3, x 256 98.0 -> 79.8;
// 32 x 1152 x 1152 x 128 31.6 -> 22.7, 8 x 512 x 512 x 128 7.8 -> 6.5, 32 x 32 x 2048 x 128 10.2 -> 6.6, 32 x 2000 x 1992 x 128 74.3 -> 63.4.  Four
// wavefronts with 64 columns each: 58.7 for the first, 75 for the third, but a tile takes them 2.35 us against 1.5 where nothing else
// runs on a CU (1 x 4096 x 4096 x 128 13.3 against 11.8); a tile quantized at a time, eight lanes to a row: 60.2.
#include "duq_epilogue.h"
#include "duq_launch.h"
#include "duq_rowquant.h"
#include "duq_tiles.h"

namespace duq {

// The first 56 bytes (through streamed) reach the kernel in registers (DUQ_HEAD_DECL / with_head).
struct ProductTilesParams {
    const uint16_t *a, *b;  // [batch, M, K], [batch, N, K]
    uint16_t *y;            // [batch, M, N]
    uint32_t M, N, tiles_n;
    uint32_t splits, per;   // workgroups that share the row tiles of 256 columns, and the tiles of each
    uint32_t units;         // workgroups
    uint32_t streamed;      // outputs go past the L2
    uint32_t reserved;
    float clip_a;
    int qmax_a;
    float clip_b;
    int qmax_b;
};
static_assert(offsetof(ProductTilesParams, clip_a) == kHeadBytes, "the fields delivered in registers");

typedef int v16i __attribute__((ext_vector_type(16)));

// NP: pieces of 32 elements in a row, 2, 4, 6 or 8.
template <int NP, bool ASYM>
__global__ __launch_bounds__(512, 4) void product_tiles_kernel(DUQ_HEAD_DECL, ProductTilesParams tail)
{
    ProductTilesParams p = with_head(tail, DUQ_HEAD_USE);
    to_global(p.a);
    to_global(p.b);
    to_global(p.y);
    constexpr int BM = 64, BN = 256, MODE = ASYM ? 1 : 0;
    constexpr int LA = NP <= 4 ? 4 : 8, NU = 4 * NP / LA, TP = 512 / LA / BM;  // lanes per row of A, units of each, tiles quantized together
    constexpr uint32_t kStride = NP * 32 + 16, kYStride = 2 * BN + 16;  // bytes per row of codes and of outputs: 4 dwords off a multiple of 8
    constexpr uint32_t kOwn = 32 * kStride;                             // at first: B's rows of a wavefront
    __shared__ __attribute__((aligned(16))) uint8_t lds[TP * BM * kStride + BM * kYStride > 8 * kOwn ? TP * BM * kStride + BM * kYStride : 8 * kOwn];
    __shared__ __attribute__((aligned(16))) uint16_t col_s[BN], col_z[ASYM ? BN : 4], row_s[TP * BM], row_z[ASYM ? TP * BM : 4];
    uint8_t *const codes = lds, *const stage = lds + TP * BM * kStride;

    // every XCD a contiguous range of workgroups, column blocks fastest: whole output rows leave from one XCD
    const uint32_t each = p.units / 8, rem = p.units % 8, xcd = blockIdx.x % 8, local = blockIdx.x / 8;
    const uint32_t id = xcd < rem ? xcd * (each + 1) + local : rem * (each + 1) + (xcd - rem) * each + local;
    const uint32_t n0 = id % p.tiles_n * BN, problem = id / p.tiles_n / p.splits;
    const uint32_t t0 = id / p.tiles_n % p.splits * p.per, t1 = min(t0 + p.per, (p.M + BM - 1) / BM);
    if (t0 >= t1) return;
    const v4u *const a = reinterpret_cast<const v4u *>(p.a) + (uint64_t)problem * p.M * (4 * NP);
    const v4u *const b = reinterpret_cast<const v4u *>(p.b) + (uint64_t)problem * p.N * (4 * NP);
    uint16_t *const y = p.y + (uint64_t)problem * p.M * p.N;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t l32 = lane & 31u, h = lane >> 5;

    // rows of A: LA lanes each, lane ua its units ua, ua + LA, ... (rows past the end of an operand: its last one again, stored by nobody)
    const uint32_t ua = tid % LA, ra = tid / LA;
    v4u raw[NU];
    auto fetch_a = [&](uint32_t t) {
        const v4u *const row = a + (uint64_t)min(t * BM + ra, p.M - 1) * (4 * NP) + ua;
#pragma unroll
        for (int j = 0; j < NU; ++j) raw[j] = row[LA * j];
    };
    auto quantize_a = [&]() {
        RowQuant<ASYM, false> rq;
        v2u w[NU];
        row_in_group<LA>(raw, ua, 4 * NP, p.clip_a, p.qmax_a, rq);
        rq.quant_units_bytes(raw, w);
#pragma unroll
        for (int j = 0; j < NU; ++j) *reinterpret_cast<v2u *>(codes + ra * kStride + ua * 8 + j * (8 * LA)) = w[j];
        if (ua == 0) {
            row_s[ra] = f16_to_bits(rq.s);
            if (ASYM) row_z[ra] = f16_to_bits(rq.z);
        }
    };

    // ---- B: each wavefront the rows of its own 32 columns, four lanes to a row and two rows to a lane, through LDS of its own into its
    // fragments
    v4i fw[NP];
    {
        const uint32_t rb = lane >> 2, ub = lane & 3u;
        uint8_t *const own = lds + wave * kOwn;
        v4u x[2][NP];
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const v4u *const row = b + (uint64_t)min(n0 + wave * 32 + r * 16 + rb, p.N - 1) * (4 * NP) + ub;
#pragma unroll
            for (int j = 0; j < NP; ++j) x[r][j] = row[4 * j];
        }
        fetch_a(t0);
        RowQuant<ASYM, false> rq[2];
#pragma unroll
        for (int r = 0; r < 2; ++r) row_in_group<4>(x[r], ub, 4 * NP, p.clip_b, p.qmax_b, rq[r]);
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            v2u w[NP];
            rq[r].quant_units_bytes(x[r], w);
#pragma unroll
            for (int j = 0; j < NP; ++j) *reinterpret_cast<v2u *>(own + (r * 16 + rb) * kStride + ub * 8 + j * 32) = w[j];
            if (ub == 0) {
                col_s[wave * 32 + r * 16 + rb] = f16_to_bits(rq[r].s);
                if (ASYM) col_z[wave * 32 + r * 16 + rb] = f16_to_bits(rq[r].z);
            }
        }
        __builtin_amdgcn_wave_barrier();  // (a wavefront's LDS operations run in order)
#pragma unroll
        for (int i = 0; i < NP; ++i) fw[i] = *reinterpret_cast<const v4i *>(own + l32 * kStride + h * 16 + i * 32);
    }
    lds_barrier();  // every wavefront has its fragments
    quantize_a();

    // The accumulators start at the bits of a float whose last place is one unit of theirs, and are that float plus the sum all along
    // (asymmetric codes are carried x 16: kF32Base, as in gemm_s4_shortk_kernel).
    constexpr float kBase = ASYM ? kF32Base : 12582912.0f;  // 1.5 * 2^23
    uint32_t start = __builtin_bit_cast(uint32_t, kBase);
    asm volatile("" : "+v"(start));
    const uint8_t *const frag = codes + l32 * kStride + h * 16;  // + 32 * step + 32 * kStride * tile
#pragma unroll 1
    for (uint32_t t = t0; t < t1; ++t) {
        lds_barrier();  // this tile's codes and row parameters are there, the last one's outputs are read
        const uint32_t half = TP == 1 ? 0u : (t - t0) & 1u;
        if (half == 0 && t + TP < t1) fetch_a(t + TP);
        v16i acc[2];
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[c][r] = (int)start;
#pragma unroll
        for (int i = 0; i < NP; ++i)
#pragma unroll
            for (int c = 0; c < 2; ++c)
                acc[c] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fw[i], *reinterpret_cast<const v4i *>(frag + (half * BM + c * 32) * kStride + i * 32), acc[c], 0, 0, 0);
        // lane: row c * 32 + l32, columns 8 * q + 4 * h + (0..3) of the wavefront's 32
        auto sum = [](int v) { return __builtin_bit_cast(float, v) - kBase; };
        RowEpi rowp[2];
#pragma unroll
        for (int c = 0; c < 2; ++c) rowp[c] = RowEpi{bits_to_f16(row_s[half * BM + c * 32 + l32]), ASYM ? bits_to_f16(row_z[half * BM + c * 32 + l32]) : (f16)0, 0};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (NP == 8) __builtin_amdgcn_sched_barrier(0);  // (two columns' parameters at a time: registers)
            const uint32_t n = wave * 32 + q * 8 + h * 4;
            const v2u s = *reinterpret_cast<const v2u *>(col_s + n), z = ASYM ? *reinterpret_cast<const v2u *>(col_z + n) : v2u{0u, 0u};
            PairCols<MODE, false> cols[2];
#pragma unroll
            for (int k = 0; k < 2; ++k) cols[k] = pair_cols_from_raw<MODE, false>(s, z, s, z, v2u{0u, 0u}, n, k);
#pragma unroll
            for (int c = 0; c < 2; ++c)
                *reinterpret_cast<v2u *>(stage + (c * 32 + l32) * kYStride + n * 2) =
                    v2u{dequant_pair<MODE, false>(sum(acc[c][q * 4]), sum(acc[c][q * 4 + 1]), rowp[c], cols[0]),
                        dequant_pair<MODE, false>(sum(acc[c][q * 4 + 2]), sum(acc[c][q * 4 + 3]), rowp[c], cols[1])};
        }
        lds_barrier();  // the whole tile is staged, the codes and row parameters are read
        if (half == TP - 1 && t + 1 < t1) quantize_a();
        // an instruction stores 512 bytes of two rows
        const uint32_t m0 = t * BM, rows_here = min(p.M - m0, (uint32_t)BM);
        const uint32_t piece = lane & 31u, ncol0 = n0 + piece * 8, row0 = wave * 8 + h;
        const uint8_t *const mine = stage + row0 * kYStride + piece * 16;
        if (p.N % 8 == 0 && reinterpret_cast<uintptr_t>(p.y) % 16 == 0) {
            const __amdgpu_buffer_rsrc_t rY = make_rsrc(y + (uint64_t)m0 * p.N, rows_here * p.N * 2);
            auto store_rows = [&](auto past) {
#pragma unroll
                for (int it = 0; it < 4; ++it) {
                    const uint32_t row = row0 + it * 2;
                    const v4u v = *reinterpret_cast<const v4u *>(mine + it * 2 * kYStride);
                    const uint32_t off = (row < rows_here && ncol0 < p.N) ? (row * p.N + ncol0) * 2 : kOobOffset;
                    __builtin_amdgcn_raw_buffer_store_b128(v, rY, (int)off, 0, decltype(past)::value ? 2 : 0);
                }
            };
            if (p.streamed) store_rows(std::true_type{});
            else store_rows(std::false_type{});
        } else {
            for (int it = 0; it < 4; ++it) {
                const uint32_t row = row0 + it * 2;
                const v4u v = *reinterpret_cast<const v4u *>(mine + it * 2 * kYStride);
                if (row < rows_here) store_row_piece(y + (uint64_t)(m0 + row) * p.N + ncol0, v, p.N - min(ncol0, p.N));
            }
        }
    }
}

// The rows of B cost a workgroup about as much as a tile: the run of tiles that makes the least of rounds of 256 workgroups, the longest
// of those that are level; a tenth more where a CU has one workgroup alone.  32 x 2048 x 2048 x 128 in one to eight runs 58.8, 55.3, 56.0,
// 55.3, 60.7 (six), 62.3 us, 8 x 4000 x 4000 x 128 102, 59.7, 59.3, 58.0, 59.1, 56.6.
struct TileRuns {
    uint32_t per, splits;  // tiles of a run, runs of 256 columns
    uint64_t runs, rounds;
};
static TileRuns tile_runs(uint32_t batch, uint32_t M, uint32_t N)
{
    TileRuns r{};
    const uint32_t tiles_m = (M + 63) / 64;
    const uint64_t blocks = (uint64_t)batch * ((N + 255) / 256);
    uint64_t least = ~0ull;
    for (uint32_t s = 1; s <= tiles_m && blocks * (s - 1) < 1024; ++s) {
        const uint32_t per = (tiles_m + s - 1) / s;
        const uint64_t rounds = (blocks * ((tiles_m + per - 1) / per) + 255) / 256, cost = rounds * (per + 1) * (rounds == 1 ? 11 : 10);
        if (cost < least) least = cost, r.per = per, r.rounds = rounds;
    }
    r.splits = (tiles_m + r.per - 1) / r.per;
    r.runs = blocks * r.splits;
    return r;
}

// All rows of up to 256 elements but for a few where the quantizer launch and the kernel behind it (for a single problem the GEMM of the
// layers) are ahead, asymmetric, us, two launches / this one:
//  rows of 256 on few blocks of columns, where many workgroups quantize the same rows of B, and with wide problems, where as many do those
//   of A: 1 x 4090 x 4096 15.7 / 16.9, 8 x 1215 x 1216 15.4 / 15.8, 1 x 2048 x 12288 22.2 / 24.6, 2 x 3000 x 11520 44.9 / 52.5, but 12 x 2046 x 2048
//   42.1 / 39.0; and with up to eight problems whose tiles leave more than a quarter of one round of long runs empty (the part of the last tile of
//   columns past N, and CUs without a run), up to twelve that leave more than 5/16: 6 x 1597 x 1600 17.1 / 18.6, 8 x 1317 x 1328 17.4 / 19.0, 4 x 1934 x
//   3168 24.0 / 25.7, 12 x 1085 x 1088 17.1 / 18.4, but 6 x 1725 x 1728 19.2 / 18.7, 12 x 1126 x 1144 20.7 / 19.3, 7 x 1533 x 1568 19.5 / 18.6;
//  large outputs whose rows do not begin at half lines: 32 x 2000 x 1992 x 256 94.5 / 97.7; single problems of many rows past 150 Mi outputs: 1 x 8192 x 20480 x
//   128 69.3 / 73.0;
//  single problems near square whose runs of three tiles (rows of 192: to five) are too few for the CUs, or just too many for one round: 1 x
//   3067 x 3072 x 128 10.0 / 10.5, 1 x 2493 x 3328 x 128 9.5 / 10.2, 1 x 3581 x 3584 x 192 12.8 / 13.5, 1 x 4221 x 4224 x 192 15.2 / 15.8, symmetric
//   1 x 3709 x 3712 x 256 14.0 / 14.5, but 1 x 3453 x 3456 x 128 11.2 / 10.4, 1 x 2813 x 2816 x 128 9.5 / 8.5, 1 x 1021 x 9216 x 128 10.7 / 10.0, 1 x 4093 x
//   4096 x 192 14.5 / 13.7;
//  in a recording, where a launch costs the host nothing, a few tiles: 1 x 64 x 64 x 256 4.9 / 7.0, 8 x 60 x 64 x 256 6.8 / 7.2, 16 x 60 x 64 x 256 7.2 /
//   7.4, 1 x 64 x 64 x 128 4.9 / 5.6, 1 x 2 x 4096 x 128 5.1 / 5.8, 1 x 16 x 4096 x 128 5.4 / 5.8; eager the first two and the fourth 7.5 / 6.8,
//   7.5 / 7.0, 7.4 / 5.4.
bool product_tiles_takes(bool asym, uint32_t batch, uint32_t M, uint32_t N, uint32_t K)
{
    if (K == 0 || K > 256 || K % 64 != 0 || M < 2 || N > (1u << 24)) return false;  // (a tile of outputs: 32-bit offsets)
    const uint64_t blocks = (uint64_t)batch * ((N + 255) / 256);
    if (blocks * ((M + 63) / 64) >= (1u << 30)) return false;
    if (K > 192 && N % 32 != 0 && (uint64_t)M * N * batch > (16u << 20)) return false;
    if (asym && K > 192 && M > 1024 && (blocks <= 40 || batch == 1 || N > 6144)) return false;
    if (asym && K > 192 && M > 1024 && batch <= 12) {
        const TileRuns r = tile_runs(batch, M, N);
        const uint64_t outputs = 256ull * r.per * (64 * 256);   // of a round whose CUs all have a run of whole tiles
        if (r.rounds == 1 && r.per >= 5 && (uint64_t)M * N * batch < outputs / 16 * (batch <= 8 ? 12 : 11)) return false;
    }
    if (batch != 1) return true;
    if (M > 1024 && (uint64_t)M * N > (150u << 20)) return false;
    if (K <= 64 || M < 2048 || N < 2048 || !(asym || K > 192)) return true;
    const TileRuns r = tile_runs(batch, M, N);
    if (r.rounds == 1) return !(r.per >= 3 && r.per <= (K <= 128 ? 3u : 5u) && r.runs <= (r.per == 3 ? 224u : 228u));
    return !(asym && r.rounds == 2 && r.per == 1);
}

bool product_tiles_eager_only(uint32_t batch, uint32_t M, uint32_t N, uint32_t K)
{
    return K > 64 && (uint64_t)batch * ((N + 255) / 256) * ((M + 63) / 64) < (M <= 16 || K > 128 ? 32u : 2u);
}

int launch_product_tiles(bool asym, const uint16_t *a, const uint16_t *b, uint32_t batch, uint32_t M, uint32_t N, uint32_t K, float clip_a,
                         int qmax_a, float clip_b, int qmax_b, uint16_t *y, hipStream_t stream)
{
    if (!product_tiles_takes(asym, batch, M, N, K)) return (int)hipErrorInvalidValue;
    ProductTilesParams p{};
    p.a = a;
    p.b = b;
    p.y = y;
    p.M = M;
    p.N = N;
    p.tiles_n = (N + 255) / 256;
    p.clip_a = clip_a;
    p.qmax_a = qmax_a;
    p.clip_b = clip_b;
    p.qmax_b = qmax_b;
    p.streamed = streams_short_rows(M, N, K, batch);
    const TileRuns r = tile_runs(batch, M, N);
    p.per = r.per;
    p.splits = r.splits;
    p.units = (uint32_t)r.runs;
#define DUQ_TILES(NP)                                                                                                     \
    do {                                                                                                                  \
        if (asym) DUQ_LAUNCH_HEAD((product_tiles_kernel<NP, true>), dim3(p.units), dim3(512), 0, stream, p);              \
        else DUQ_LAUNCH_HEAD((product_tiles_kernel<NP, false>), dim3(p.units), dim3(512), 0, stream, p);                  \
    } while (0)
    if (K <= 64) DUQ_TILES(2);
    else if (K <= 128) DUQ_TILES(4);
    else if (K <= 192) DUQ_TILES(6);
    else DUQ_TILES(8);
#undef DUQ_TILES
    return (int)hipGetLastError();
}

}  // namespace duq
