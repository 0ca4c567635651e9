// Quantizer, GEMM and dequant of the 8-bit layer for a few dozen rows in one launch: float32 activations in.
//
// duq_quant_gemm.hip's kernel for int8: a workgroup quantizes the rows of its tile itself, with the arithmetic of the row quantizer
// (src/kernels/quant.cu:241-279, qlinear4bit/nn/quantizer.py:38-55), while its whole share of the weights comes to LDS, from the
// weight as stored or its tiled copy.  Rows are twice as many bytes as in the 4-bit kernel and their codes 42 instructions per eight
// elements, so a workgroup has half as many elements, 32768 (128 KB; 1.2 us of fetching, 1.5 of vector work beside the weights').  8 tokens
// 4096 x 4096 6.2 -> 5.65 us called eagerly, 73 x 4359 x 896 9.4 -> 6.0, where two launches take 8.2 us of host time at least.
#include "duq_int8_common.h"
#include "duq_launch.h"
#include "duq_tiles.h"

namespace duq {

namespace {

// The first 56 bytes (through y) reach the kernel in registers (DUQ_HEAD_DECL / with_head).
struct QuantGemm8Params {
    const float *X;    // [M, K]
    const int8_t *B;   // [N, K], or its tiled copy
    uint32_t M, N, K;
    uint32_t groups;   // of rows, and 2^16 over them from bit 9 on
    uint32_t chunks;   // of columns, in a workgroup
    uint32_t tiled;
    const float *s_col;
    float *y;
    const float *z_col, *bias;
};
static_assert(offsetof(QuantGemm8Params, y) + sizeof(float *) == kHeadBytes, "the fields delivered in registers");

// ROWS rows of eight wavefronts, each row held by 512 / ROWS lanes, UPL pieces of four elements a lane.
template <int ROWS, int UPL, int NT, int BUFS, bool SPLIT>
struct QuantTile8 {
    static constexpr int LPR = 512 / ROWS, RPI = 64 / LPR, MT = (ROWS + 15) / 16;  // lanes of a row, rows of a wavefront, row tiles
    static constexpr int KB = LPR * UPL * 4;                      // the longest row
    // SPLIT: the wavefronts split K, a wavefront multiplies SLICE bytes of every row of the tile at a time.  Otherwise each has one of
    // the eight 16 x 16 tiles, and all of K.
    static constexpr int SLICE = SPLIT && KB / 8 < 128 ? KB / 8 : 128;
    static constexpr int V = SPLIT ? 8 : 1, S = KB / V / SLICE, U = SLICE / 64;  // wavefronts and slices of one along K, 64-byte fragments in a slice
    static constexpr int XSTRIDE = KB + 16;                       // (the rows of a fragment read fall on different banks)
    static constexpr int kX = ROWS * XSTRIDE, kW = NT * 16 * KB /* of one buffer */, kPart = SPLIT ? NT * MT * 8 * 1024 : 0;
    static_assert(U >= 1 && (SPLIT || MT * NT == 8), "work for every wavefront");
    static_assert(kX + BUFS * kW + kPart <= 159 * 1024, "LDS");
};

// The plan of quant_gemm_s4_kernel: eight wavefronts quantize and then multiply, four others only fetch weights.
template <int ROWS, int UPL, int NT, int BUFS, bool SPLIT>
__global__ __launch_bounds__(768) void quant_gemm_s8_kernel(DUQ_HEAD_DECL, QuantGemm8Params tail)
{
    QuantGemm8Params p = with_head(tail, DUQ_HEAD_USE);
    to_global(p.y);
    using Tile = QuantTile8<ROWS, UPL, NT, BUFS, SPLIT>;
    constexpr int LPR = Tile::LPR, RPI = Tile::RPI, MT = Tile::MT, V = Tile::V, S = Tile::S, U = Tile::U;
    constexpr uint32_t SLICE = Tile::SLICE, XSTRIDE = Tile::XSTRIDE;
    __shared__ __attribute__((aligned(256))) uint8_t lds_w[BUFS * Tile::kW];
    __shared__ __attribute__((aligned(16))) uint8_t xs[Tile::kX];
    __shared__ v4i part[SPLIT ? NT : 1][SPLIT ? MT : 1][8][SPLIT ? 64 : 1];
    __shared__ float srow[MT * 16], zrow[MT * 16];

    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t l16 = lane & 15u, g = lane >> 4;
    // groups of ROWS rows share the weights of a column range: consecutive in `at`, an eighth of which runs on one XCD
    const uint32_t width = 16 * NT * (BUFS == 1 ? 1 : p.chunks);
    const uint32_t groups = p.groups & 0x1FFu, per_xcd = ((p.N + width - 1) / width * groups + 7) / 8;
    const uint32_t at = blockIdx.x % 8 * per_xcd + blockIdx.x / 8, tile = at * (p.groups >> 9) >> 16;  // (tile = at / groups)
    const uint32_t col0 = tile * width, m0 = (at - tile * groups) * ROWS;
    if (col0 >= p.N) return;
    const uint32_t chunks = BUFS == 1 ? 1 : min(p.chunks, (p.N - col0 + 16 * NT - 1) / (16 * NT));
    auto sync = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

    // ---- the wavefronts that fetch: instruction i takes kilobyte i of [column tile][slice][wavefront], rows of SLICE bytes whose
    // 16-byte pieces lie at piece ^ (row / Q), so that the sixteen rows of a fragment read sixteen places.  The tiled copy has the
    // same piece of 32 rows side by side, in [32 rows][step of 32 k][half of the step]: eight rows of it are a line.
    constexpr uint32_t PR = SLICE / 16, RPW = 64 / PR, Q = 256 / SLICE;   // pieces a row, rows an instruction
    if (wave >= 8) {
        const uint32_t first = p.tiled ? col0 & ~31u : col0, last = p.tiled ? (p.N + 31u) & ~31u : p.N;  // (rows past N: zeros, or read as zero)
        const uint64_t a = reinterpret_cast<uint64_t>(p.B + (uint64_t)first * p.K);
        const v4u dW = {(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a), (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)(a >> 32) & 0xFFFFu)),
                        (uint32_t)__builtin_amdgcn_readfirstlane((int)(min(last - first, width + 32) * p.K)), 0x00020000u};
        const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds_w;
        constexpr uint32_t kInstr = Tile::kW / 1024;
        static_assert(kInstr % 4 == 0 && BUFS * (kInstr / 4) <= 63, "vmcnt");
        auto fetch = [&](uint32_t chunk) {
#pragma unroll
            for (uint32_t j = 0; j < kInstr / 4; ++j) {
                const uint32_t i = j * 4 + (wave - 8);
                const uint32_t r = i % (16 / RPW) * RPW + lane / PR, v = i / (16 / RPW) % V, s = i / (16 / RPW) / V % S, n = i / (16 / RPW) / V / S;
                const uint32_t piece = (s * V + v) * PR + ((lane % PR) ^ (r / Q)), row = col0 - first + (chunk * NT + n) * 16 + r;
                const uint32_t from = p.tiled ? (row >> 5) * 32 * p.K + (piece >> 1) * 1024 + ((piece & 1u) * 32 + (row & 31u)) * 16 : row * p.K + piece * 16;
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(lds0 + (chunk % BUFS) * Tile::kW + i * 1024),
                             "v"(piece * 16 < p.K ? from : kOobOffset), "s"(dW)
                             : "memory", "m0");
            }
        };
        if (ROWS == 8) __builtin_amdgcn_s_barrier();  // (behind the requests for the activations, which are needed first)
        fetch(0);
        if (BUFS == 1) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            sync();  // the weights are here, and everybody's codes
            if (SPLIT) sync();  // the partial sums are written
        } else {
            fetch(1);  // (rows past the tensor read as zero)
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kInstr / 4) : "memory");
            for (uint32_t c = 0; c < chunks; ++c) {
                sync();  // (first the codes;) the weights of chunk c are here
                sync();  // ... and read
                fetch(c + 2);
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kInstr / 4) : "memory");
            }
        }
        return;
    }
    static_assert(BUFS == 1 || !SPLIT, "the barriers above");

    // ---- the wavefronts that quantize: lane l holds pieces l % LPR, + LPR, ... of row l / LPR of this wavefront's.  Pieces past the row
    // end are copies of its last one, which change no statistic, and their codes meet no weight.
    const uint32_t nvec = p.K >> 2, u0 = lane % LPR, qrow = wave * RPI + lane / LPR;
    const __amdgpu_buffer_rsrc_t rX = make_rsrc(p.X + (uint64_t)m0 * p.K, min(p.M - m0, (uint32_t)ROWS) * p.K * 4);  // rows past M read as zero
    v4f32 raw[UPL];
#pragma unroll
    for (int j = 0; j < UPL; ++j) raw[j] = __builtin_bit_cast(v4f32, buf_load16(rX, (qrow * nvec + min(u0 + j * LPR, nvec - 1)) * 16, 0));
    if (ROWS == 8) __builtin_amdgcn_s_barrier();
    // the parameters of the outputs this thread finishes, behind them.  SPLIT: 256 threads take half of the column tiles (one row
    // tile), or half of the row tiles; otherwise a lane holds four columns of a row of its wavefront's tile
    constexpr int FN = !SPLIT ? 4 : MT == 1 ? (NT + 1) / 2 : NT, FM = !SPLIT || MT == 1 ? 1 : MT / 2;
    const uint32_t src_lane = (tid >> 2) & 63u, er = tid & 3u, fg = tid >> 8;
    const uint32_t my_m = SPLIT ? src_lane & 15u : l16, my_c = (src_lane >> 4) * 4 + er;
    const bool bias = p.bias != nullptr;
    struct Columns {
        float s[FN], z[FN], b[FN];
    } cp, cpn;
    auto column = [&](uint32_t chunk, int f) {
        return col0 + (SPLIT ? (chunk * NT + (MT == 1 ? f * 2 + fg : f)) * 16 + my_c : (chunk * NT + wave / MT) * 16 + g * 4 + f);
    };
    auto fetch_columns = [&](uint32_t chunk, Columns &c) {
#pragma unroll
        for (int f = 0; f < FN; ++f) {
            const uint32_t n = min(column(chunk, f), p.N - 1);
            c.s[f] = p.s_col[n];
            c.z[f] = p.z_col[n];
            c.b[f] = bias ? p.bias[n] : 0.f;
        }
    };
    fetch_columns(0, cp);

    const bool live = m0 + qrow < p.M;
    if (RPI > 1 || live) {
        // (v_minimum3_f32 / v_maximum3_f32 return a NaN when an operand is one, as torch's min and max do)
        float lo = INFINITY, hi = -INFINITY;
#pragma unroll
        for (int j = 0; j < UPL; ++j)
#pragma unroll
            for (int e = 0; e < 4; e += 2) {
                asm("v_minimum3_f32 %0, %0, %1, %2" : "+v"(lo) : "v"(raw[j][e]), "v"(raw[j][e + 1]));
                asm("v_maximum3_f32 %0, %0, %1, %2" : "+v"(hi) : "v"(raw[j][e]), "v"(raw[j][e + 1]));
            }
        lo = __builtin_bit_cast(float, lanes_reduce<LPR>(__builtin_bit_cast(uint32_t, lo), [](uint32_t x, uint32_t y) {
            asm("v_minimum3_f32 %0, %0, %1, %1" : "+v"(x) : "v"(y));
            return x;
        }));
        hi = __builtin_bit_cast(float, lanes_reduce<LPR>(__builtin_bit_cast(uint32_t, hi), [](uint32_t x, uint32_t y) {
            asm("v_maximum3_f32 %0, %0, %1, %1" : "+v"(x) : "v"(y));
            return x;
        }));
        if (lo != lo || hi != hi) lo = hi = __builtin_nanf("");
        if (RPI > 1 && !live) hi = 127.f;  // (zeros alone would send the rows beside them down the element-wise path)
        const RowCode8 rc(lo, hi);
        uint8_t *const to = xs + qrow * XSTRIDE + u0 * 4;
        if (__builtin_amdgcn_ballot_w64(!rc.fast) == 0) {
#pragma unroll
            for (int j0 = 0; j0 < UPL; j0 += 4) {
                if ((uint32_t)(j0 * LPR) >= nvec) break;
                uint32_t c[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) c[j] = rc.quick4(raw[j0 + j]);
#pragma unroll
                for (int j = 0; j < 4; ++j) *reinterpret_cast<uint32_t *>(to + (j0 + j) * (LPR * 4)) = c[j];
            }
        } else {  // element by element, in a loop that fetches them again
#pragma unroll 1
            for (uint32_t u = u0; u < nvec; u += 4 * LPR) {
                v4f32 in[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) in[j] = __builtin_bit_cast(v4f32, buf_load16(rX, (qrow * nvec + min(u + j * LPR, nvec - 1)) * 16, 0));
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (u + j * LPR < nvec) *reinterpret_cast<uint32_t *>(to + (u - u0 + j * LPR) * 4) = rc.slow4(in[j]);
            }
        }
        if (u0 == 0) {
            srow[qrow] = rc.s;
            zrow[qrow] = rc.z;
        }
    }
    if (SPLIT || BUFS == 1) sync();

    // ---- products
    // (one tile to a wavefront, several chunks: its rows' fragments stay in registers)
    constexpr bool kHold = !SPLIT && BUFS > 1;
    v4i held[kHold ? S * U : 1];
    if constexpr (kHold) {
        sync();  // the codes are here, and the first chunk's weights
#pragma unroll
        for (int f = 0; f < S * U; ++f) held[f] = *reinterpret_cast<const v4i *>(xs + (wave % MT * 16 + l16) * XSTRIDE + f * 64 + g * 16);
    }
    for (uint32_t chunk = 0; chunk < chunks; ++chunk) {
        if (BUFS > 1) fetch_columns(chunk + 1, cpn);  // (before this chunk's stores: what waits for it would wait for them too)
        if (!SPLIT && BUFS > 1 && chunk > 0) sync();  // this chunk's weights are here
        constexpr int AN = SPLIT ? NT : 1, AM = SPLIT ? MT : 1;  // the wavefront's tiles
        const uint32_t v = SPLIT ? wave : 0, am = SPLIT ? 0 : wave % MT, an = SPLIT ? 0 : wave / MT;
        const uint8_t *const ws = lds_w + chunk % BUFS * Tile::kW + (an * S * V + v) * (16 * SLICE) + l16 * SLICE;
        const uint8_t *const xr = xs + (am * 16 + l16 % (ROWS < 16 ? ROWS : 16)) * XSTRIDE + v * SLICE + g * 16;
        v4i acc[AN][AM];
#pragma unroll
        for (int n = 0; n < AN; ++n)
#pragma unroll
            for (int m = 0; m < AM; ++m) acc[n][m] = v4i{0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < S; ++s) {
            if ((s * V + v) * SLICE >= p.K) break;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                v4i x[AM];
#pragma unroll
                for (int m = 0; m < AM; ++m)
                    x[m] = kHold ? held[s * U + u] : *reinterpret_cast<const v4i *>(xr + m * (16 * XSTRIDE) + s * (V * SLICE) + u * 64);
#pragma unroll
                for (int n = 0; n < AN; ++n) {
                    const v4i w = *reinterpret_cast<const v4i *>(ws + (n * S + s) * (V * 16 * SLICE) + ((u * 4 + g) ^ (l16 / Q)) * 16);
#pragma unroll
                    for (int m = 0; m < AM; ++m) acc[n][m] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w, x[m], acc[n][m], 0, 0, 0);
                }
            }
        }
        if constexpr (SPLIT) {
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int m = 0; m < MT; ++m) part[n][m][wave][lane] = acc[n][m];
            sync();
        } else if (BUFS > 1) {
            sync();  // everybody has read them
        }

#pragma unroll
        for (int fm = 0; fm < FM; ++fm) {
            const uint32_t mt = !SPLIT ? am : MT == 1 ? 0 : fm * 2 + fg, row = mt * 16 + my_m;
            const bool mine = ROWS >= 16 || row < ROWS;
            const float sr = mine ? srow[row] : 0.f, zr = mine ? zrow[row] : 0.f;
            const uint32_t m = m0 + row;
            v4f32 out;
#pragma unroll
            for (int f = 0; f < FN; ++f) {
                const uint32_t nt = MT == 1 ? f * 2 + fg : f;
                if (SPLIT && nt >= (uint32_t)NT) continue;
                int sum = 0;
                if constexpr (SPLIT) {
                    const int *const sums = reinterpret_cast<const int *>(part[nt][mt]) + src_lane * 4 + er;
#pragma unroll
                    for (int i = 0; i < 8; ++i) sum += sums[i * 256];
                } else {
                    sum = acc[0][0][f];
                }
                float o = dequant_hprec_one(sum, sr, zr, cp.s[f], cp.z[f]);
                if (bias) o = o + cp.b[f];
                const uint32_t n = column(chunk, f);
                if (SPLIT) {
                    if (mine && m < p.M && n < p.N) p.y[(uint64_t)m * p.N + n] = o;
                } else {
                    out[f % 4] = o;
                }
            }
            if constexpr (!SPLIT) {
                typedef v4f32 v4f32_any __attribute__((aligned(4)));
                const uint32_t n = column(chunk, 0);
                if (m < p.M && n < p.N) {
                    float *const to = p.y + (uint64_t)m * p.N + n;
                    if (n + 3 < p.N) {
                        *reinterpret_cast<v4f32_any *>(to) = out;
                    } else {
#pragma unroll
                        for (int f = 0; f < 4; ++f)
                            if (n + f < p.N) to[f] = out[f];
                    }
                }
            }
        }
        if (BUFS > 1) cp = cpn;
    }
}

template <int ROWS, int UPL, int NT, int BUFS>
bool launch_shape8(QuantGemm8Params &p, uint32_t chunks, hipStream_t stream)
{
    constexpr bool SPLIT = (ROWS + 15) / 16 * NT < 8;
    using Tile = QuantTile8<ROWS, UPL, NT, BUFS, SPLIT>;
    // groups of rows, and 2^16 over them: (at * m) >> 16 == at / groups while at * (groups - 1) < 2^16
    const uint32_t width = 16 * NT * chunks;
    const uint64_t groups = (p.M + ROWS - 1) / ROWS, tiles = (p.N + width - 1) / width;
    if (groups > 64 || (groups > 1 && (groups * tiles + 8) * (groups - 1) >= 65536) || p.K > Tile::KB || ((uint64_t)width + 64) * p.K >= kOobOffset) return false;
    p.groups = (uint32_t)groups | (uint32_t)((65535 + groups) / groups) << 9;
    p.chunks = chunks;
    DUQ_LAUNCH_HEAD((quant_gemm_s8_kernel<ROWS, UPL, NT, BUFS, SPLIT>), dim3((uint32_t)((tiles * groups + 7) / 8 * 8)), dim3(768), 0, stream, p);
    return true;
}

}  // namespace

int launch_quant_gemm8(QuantGemmShape s, const float *x, const int8_t *B, bool b_tiled, uint32_t M, uint32_t N, uint32_t K, const float *s_col,
                       const float *z_col, const float *bias, float *y, hipStream_t stream)
{
    QuantGemm8Params p{x, B, M, N, K, 0, 0, b_tiled, s_col, y, z_col, bias};
    bool launched = false;
    const bool half = (uint64_t)s.rows * K <= 16384;  // eight pieces for every lane
#define DUQ_Q8(R, U, C, B)                                                                   \
    if (s.rows == R && half == (U == 8) && s.cols == C && (s.chunks > 1) == (B > 1)) \
        launched = launch_shape8<R, U, C, B>(p, s.chunks, stream);
    DUQ_Q8(8, 8, 1, 1)
    DUQ_Q8(8, 8, 2, 1)
    DUQ_Q8(8, 8, 3, 1)
    DUQ_Q8(8, 16, 1, 1)
    DUQ_Q8(16, 8, 1, 1)
    DUQ_Q8(16, 8, 2, 1)
    DUQ_Q8(16, 8, 3, 1)
    DUQ_Q8(16, 8, 8, 1)
    DUQ_Q8(16, 16, 1, 1)
    DUQ_Q8(16, 16, 2, 1)
    DUQ_Q8(16, 16, 3, 1)
    DUQ_Q8(32, 8, 4, 1)
    DUQ_Q8(32, 8, 4, 2)
    DUQ_Q8(32, 16, 4, 1)
#undef DUQ_Q8
    return launched ? (int)hipGetLastError() : (int)hipErrorInvalidValue;
}

}  // namespace duq
