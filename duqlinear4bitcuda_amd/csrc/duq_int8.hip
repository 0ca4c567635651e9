// The 8-bit asymmetric layer of the reference (LinearQuant8bitASQ) for gfx950: per-token int8
// quantizer (float32 in), int8 x int8 -> int32 GEMM on v_mfma_i32_32x32x32_i8, float32
// dequant ("hprec") stand-alone or fused into the GEMM.
//   quantize : src/kernels/quant.cu:241-279      scale/zero : qlinear4bit/nn/quantizer.py:38-55
//   GEMM     : src/kernels/gemm.cu:46-81         dequant    : src/kernels/quant.cu:281-323
// Arithmetic is float32 with one rounding per operator, as in the reference; the quantizer's
// value goes through binary16 on its way to the integer (the reference passes a float to
// __half2int_rn).
#include "duq_int8_common.h"
#include "duq_launch.h"
#include "duq_tiles.h"

// Cache policy of the decode-size kernels' weight loads: 2 = non-temporal (the weights are read once, in whole cache
// lines; measured 1-6 % faster: 16 x 11008 x 4096 10.3 against 10.85 us, 16 x 4096 x 8192 9.5 against 10.1)
#ifndef DUQ_S8_ROWS_WLOAD_AUX
#define DUQ_S8_ROWS_WLOAD_AUX 2
#endif
#ifndef DUQ_S8_DEC_WLOAD_AUX
#define DUQ_S8_DEC_WLOAD_AUX 2
#endif
#ifndef DUQ_S8_SKINNY_WLOAD_AUX
#define DUQ_S8_SKINNY_WLOAD_AUX 2
#endif

namespace duq {

typedef int v16i32 __attribute__((ext_vector_type(16)));

// smallest and largest element so far, and whether a NaN was met (fminf / fmaxf pass one over)
__device__ __forceinline__ void row_stats8(const v4f32 &g, float &lo, float &hi, bool &nan_seen)
{
#pragma unroll
    for (int e = 0; e < 4; e += 2) {
        lo = fminf(fminf(lo, g[e]), g[e + 1]);
        hi = fmaxf(fmaxf(hi, g[e]), g[e + 1]);
        nan_seen |= __builtin_isunordered(g[e], g[e + 1]);
    }
}

// ---------------------------------------------------------------------------------
// given-scale quantizer (asym_quant_host_8bit): 4 elements per lane step when the row
// length allows, else one
// ---------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void asym_quant8_kernel(const float *x, const float *scale, const float *zeros,
                                                          uint32_t rows, uint32_t cols, int8_t *q, bool vec)
{
    if (vec) {
        const uint32_t per_row = cols >> 2;
        const uint64_t total = (uint64_t)rows * per_row;
        for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (uint64_t)gridDim.x * blockDim.x) {
            const uint32_t row = (uint32_t)(i / per_row);
            const v4f32 v = __builtin_nontemporal_load(reinterpret_cast<const v4f32 *>(x) + i);
            const float s = scale[row];
            const int zi = asym8_zero_int(zeros[row]);
            uint32_t w = 0;
#pragma unroll
            for (int e = 0; e < 4; ++e) w |= asym8_code(v[e], s, zi) << (8 * e);
            reinterpret_cast<uint32_t *>(q)[i] = w;
        }
    } else {
        const uint64_t total = (uint64_t)rows * cols;
        for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (uint64_t)gridDim.x * blockDim.x) {
            const uint32_t row = (uint32_t)(i / cols);
            q[i] = (int8_t)asym8_code(x[i], scale[row], asym8_zero_int(zeros[row]));
        }
    }
}

int launch_asym_quant8(const float *x, const float *scale, const float *zeros, uint32_t rows, uint32_t cols, int8_t *q,
                       hipStream_t stream)
{
    if (rows == 0 || cols == 0) return 0;
    const bool vec = cols % 4 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(q) % 4 == 0;
    const uint64_t total = (uint64_t)rows * (vec ? cols / 4 : cols);
    const uint32_t blocks = (uint32_t)std::min<uint64_t>((total + 255) / 256, 1u << 20);
    hipLaunchKernelGGL(asym_quant8_kernel, dim3(blocks), dim3(256), 0, stream, x, scale, zeros, rows, cols, q, vec);
    return (int)hipGetLastError();
}

// ---------------------------------------------------------------------------------
// fused row quantizer (AsymQuantizer8bit.forward in one pass): one workgroup per row, the row
// held in registers between the min / max reduction and the quantization (up to 8 x 4
// elements per lane; longer rows are read a second time, from L2)
// ---------------------------------------------------------------------------------

// NV: 16-byte pieces of a row that a lane holds (0: none, the row is read twice).  Pieces past the row end are copies of
// its last one, which change no statistic, and their codes are stored nowhere (beyond the descriptor): no piece hangs on a
// branch of its own, so the chains of the quotients run side by side.
template <int WAVES, int NV>
__global__ __launch_bounds__(WAVES * 64) void quantize_rows_asym8_kernel(const float *x, uint32_t rows, uint32_t cols,
                                                                         int8_t *q, float *scale, float *zeros)
{
    constexpr int T = WAVES * 64;
    constexpr bool CACHED = NV > 0;
    __shared__ float red[2][WAVES];
    const uint32_t row = blockIdx.x, tid = threadIdx.x;
    const uint32_t nvec = cols >> 2;
    const v4f32 *xrow = reinterpret_cast<const v4f32 *>(x + (uint64_t)row * cols);
    uint32_t *qrow = reinterpret_cast<uint32_t *>(q + (uint64_t)row * cols);
    v4f32 regs[CACHED ? NV : 1];
    float lo = INFINITY, hi = -INFINITY;
    bool nan_seen = false;
    auto reduce = [&](const v4f32 &g) { row_stats8(g, lo, hi, nan_seen); };
    if (CACHED) {
#pragma unroll
        for (int i = 0; i < NV; ++i) regs[i] = __builtin_nontemporal_load(&xrow[min(tid + i * T, nvec - 1)]);
#pragma unroll
        for (int i = 0; i < NV; ++i) reduce(regs[i]);
    } else {
        for (uint32_t u = tid; u < nvec; u += T) reduce(xrow[u]);
    }
    lo = wave_min_f32(lo);
    hi = wave_max_f32(hi);
    nan_seen = __builtin_amdgcn_ballot_w64(nan_seen) != 0;
    if (WAVES > 1) {
        if ((tid & 63u) == 0) {
            red[0][tid >> 6] = nan_seen ? __builtin_nanf("") : lo;
            red[1][tid >> 6] = hi;
        }
        __syncthreads();
        lo = red[0][0];
        hi = red[1][0];
        nan_seen = lo != lo;
#pragma unroll
        for (int w = 1; w < WAVES; ++w) {
            nan_seen |= red[0][w] != red[0][w];
            lo = fminf(lo, red[0][w]);
            hi = fmaxf(hi, red[1][w]);
        }
    }
    if (nan_seen) lo = hi = __builtin_nanf("");  // torch's min / max return NaN for a row that holds one
    const RowCode8 rc(lo, hi);
    if (tid == 0) {
        scale[row] = rc.s;
        zeros[row] = rc.z;
    }
    auto quantize = [&](auto code4) {
        if (CACHED) {
            const __amdgpu_buffer_rsrc_t rQ = make_rsrc(qrow, cols);
            uint32_t c[CACHED ? NV : 1];
#pragma unroll
            for (int i = 0; i < NV; ++i) c[i] = code4(regs[i]);
#pragma unroll
            for (int i = 0; i < NV; ++i) __builtin_amdgcn_raw_buffer_store_b32(c[i], rQ, (int)((tid + i * T) * 4), 0, 0);
        } else {
            for (uint32_t u = tid; u < nvec; u += T) qrow[u] = code4(xrow[u]);
        }
    };
    if (__builtin_amdgcn_readfirstlane(rc.fast))  // (one row, one answer)
        quantize([&](const v4f32 &g) { return rc.quick4(g); });
    else
        quantize([&](const v4f32 &g) { return rc.slow4(g); });
}

int launch_quantize_rows_asym8(const float *x, uint32_t rows, uint32_t cols, int8_t *q, float *scale, float *zeros,
                               hipStream_t stream)
{
    if (rows == 0 || cols == 0) return 0;
    const uint32_t nvec = cols / 4;
    uint32_t waves = 1;
    while (waves < 16 && waves * 64 * 4 < nvec) waves *= 2;  // four 128-bit loads per lane when the row allows
    const dim3 grid(rows);
#define DUQ_ROWS8(W, V) \
    hipLaunchKernelGGL((quantize_rows_asym8_kernel<W, V>), grid, dim3(W * 64), 0, stream, x, rows, cols, q, scale, zeros)
    switch (waves) {
    case 1: DUQ_ROWS8(1, 4); break;
    case 2: DUQ_ROWS8(2, 4); break;
    case 4: DUQ_ROWS8(4, 4); break;
    case 8: DUQ_ROWS8(8, 4); break;
    default:
        if (nvec <= 16 * 64 * 4) DUQ_ROWS8(16, 4);
        else if (nvec <= 16 * 64 * 8) DUQ_ROWS8(16, 8);
        else DUQ_ROWS8(16, 0);
    }
#undef DUQ_ROWS8
    return (int)hipGetLastError();
}

// ---------------------------------------------------------------------------------
// float32 dequant: x = (s_r * s_c) * (float(acc) - (z_r + z_c)) [+ bias]
// ---------------------------------------------------------------------------------
struct Epi8 {
    const float *s_row, *z_row, *s_col, *z_col, *bias;
};

__global__ __launch_bounds__(256) void dequant_hprec_kernel(const int32_t *acc, Epi8 e, uint32_t rows, uint32_t cols, float *x)
{
    const uint64_t total = (uint64_t)rows * cols;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t row = (uint32_t)(i / cols), col = (uint32_t)(i % cols);
        float v = dequant_hprec_one(acc[i], e.s_row[row], e.z_row[row], e.s_col[col], e.z_col[col]);
        if (e.bias) v = v + e.bias[col];
        x[i] = v;
    }
}

int launch_dequant_hprec(const int32_t *acc, const float *s_row, const float *z_row, const float *s_col,
                         const float *z_col, const float *bias, uint32_t rows, uint32_t cols, float *x, hipStream_t stream)
{
    if (rows == 0 || cols == 0) return 0;
    const uint64_t total = (uint64_t)rows * cols;
    const uint32_t blocks = (uint32_t)std::min<uint64_t>((total + 255) / 256, 1u << 20);
    hipLaunchKernelGGL(dequant_hprec_kernel, dim3(blocks), dim3(256), 0, stream, acc, Epi8{s_row, z_row, s_col, z_col, bias},
                       rows, cols, x);
    return (int)hipGetLastError();
}

// ---------------------------------------------------------------------------------
// GEMM  C[m,n] = sum_k A[m,k] * B[n,k]   (int8, int32 accumulation)
// ---------------------------------------------------------------------------------
// Tile 32*TM (M) x 256 (N), 4 wavefronts side by side along N (32*TM x 64 each, TM x 2 MFMA tiles of 32 x 32),
// 256-k chunks of 8 steps.  A wavefront's 64 weight rows are needed by no other wavefront, so weights go
// global -> registers: lane (r = lane % 32, h = lane / 32) holds bytes [32*s + 16*h, +16) of row r for step s, which
// is the operand layout of v_mfma_i32_32x32x32_i8; the register of step s is refetched for the next chunk as soon
// as the step's last MFMA has been issued, so every weight load has a whole chunk (64 MFMAs,
// 2048 cycles) to arrive.  Activations are shared by the four wavefronts: global -> registers -> LDS (three buffers, rows padded
// to 272 bytes, one barrier per chunk) -> fragments read one step ahead; the register of piece j is stored at step
// j (for the chunk after next) and refetched at once (for the chunk after that), again a whole chunk ahead.
// The weight operand is the MFMA "A" side, so a lane ends up with four consecutive output columns of one row.
// The first 56 bytes (through tiles_n) reach the kernels in registers (DUQ_HEAD_DECL / with_head).
struct Gemm8Params {
    const int8_t *A;  // [M, K]
    const int8_t *B;  // [N, K]
    uint32_t M, N, K;
    uint32_t tiles_m;
    int32_t *C;       // int32 out (not fused)
    float *y;         // float32 out (fused)
    uint32_t tiles_n;
    Epi8 epi;
};
static_assert(offsetof(Gemm8Params, epi) == kHeadBytes, "the fields delivered in registers");

// Outputs of prefill-sized tiles.  Descriptor of `rows` rows (at most 64: 32-bit offsets) from row m on: those past M are
// beyond it.
template <bool FUSED>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t out_rows(const Gemm8Params &p, uint32_t m, uint32_t rows)
{
    const uint32_t here = m < p.M ? min(p.M - m, rows) : 0u;
    return make_rsrc(FUSED ? (const void *)(p.y + (uint64_t)m * p.N) : (const void *)(p.C + (uint64_t)m * p.N), here * p.N * 4);
}
// Four neighbouring outputs, columns n .. n + 3 (`whole`: all inside the row) of the descriptor's row `row`.  One store
// without a branch, at whatever alignment the row has (the hardware splits it); the last columns of an N that is no multiple
// of four one by one, on a branch that other widths do not take.  With four stores per lane for such N, and
// a branch around every store that the conversion sank into: 2048 x 11007 x 4096 109.6 us, now 99.1; 700 x 8191 x 4096 34.8 / 28.6;
// 2048 x 3001 x 512 18.2 / 13.7; and 2048 x 11008 x 4096 93.6 / 91.6, 4096 x 11008 x 4096 169 / 164.6, but 1500 x 5000 x 4096 34.6 /
// 35.4 (2048 x 5000 x 2048 39.5 / 38.7).
__device__ __forceinline__ void store_quad8(const Gemm8Params &p, __amdgpu_buffer_rsrc_t r, uint32_t row, uint32_t n, bool whole, v4i v)
{
    const uint32_t off = (row * p.N + n) * 4;
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, v), r, (int)(whole ? off : kOobOffset), 0, 2);
    if (p.N % 4 != 0) {
#pragma unroll
        for (int e = 0; e < 3; ++e)
            __builtin_amdgcn_raw_buffer_store_b32((uint32_t)v[e], r, (int)(!whole && n + e < p.N ? off + e * 4 : kOobOffset), 0, 0);
    }
}

__device__ __forceinline__ void lds_barrier8() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

template <int TM, int TN>
struct Tile8 {
    static constexpr int BM = 32 * TM, BN = 128 * TN;
    // steps (of 32 k) per chunk: 8, or 4 with 256-row tiles (TM = 8: all 256 accumulation registers hold accumulators
    // and three activation buffers of 256-k chunks would not fit in LDS)
    static constexpr int NS = TM == 8 ? 4 : 8;
    static constexpr uint32_t kStride = 32 * NS + 16, kEStride = 32 * TN * 4 + 16;  // epilogue staging: 32 rows of 32*TN int32 per wavefront
    static constexpr uint32_t kLds = 3 * BM * kStride > 4 * 32 * kEStride ? 3 * BM * kStride : 4 * 32 * kEStride;
};

// The tile of rows m0 .. and columns n0 ...  lds: Tile8::kLds bytes; row_par: [2][BM], its per-row scale and zero point.
template <int TM, int TN, bool FUSED, bool BIAS, bool TILED>
__device__ __forceinline__ void gemm8_tile(const Gemm8Params &p, uint8_t *lds, float *row_par, const uint32_t m0, const uint32_t n0)
{
    static_assert(TM == 8 || TM == 4 || TM == 3 || TM == 2 || TM == 1, "32-row MFMA tiles per wavefront along M");
    // TN = 32-column MFMA tiles per wavefront: tiles of 256 columns (TN = 2), or of 128 (TN = 1, with 64-row tiles:
    // twice the workgroups for problems that leave CUs without a 64 x 256 tile)
    static_assert(TN == 2 || (TN == 1 && TM == 2), "column tiles per wavefront");
    constexpr int BM = Tile8<TM, TN>::BM, BN = Tile8<TM, TN>::BN, NS = Tile8<TM, TN>::NS;
    constexpr uint32_t kChunk = 32 * NS;  // 256 (128)
    constexpr uint32_t kStride = Tile8<TM, TN>::kStride;
    constexpr uint32_t kBuf = BM * kStride;
    constexpr int PPR = kChunk / 16;      // 16-byte pieces per row of a chunk
    constexpr int NXP = BM * PPR / 256;   // 16-byte activation pieces per thread and chunk: 8, 4, 2 (TM = 8: 8)

    constexpr uint32_t kEStride = Tile8<TM, TN>::kEStride;

    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63u, wave = tid >> 6;
    const uint32_t l32 = lane & 31u, h = lane >> 5;
    const uint32_t nchunks = (p.K + kChunk - 1) / kChunk;

    // tiled weights: whole 32-row tiles (the last one zero-padded), K * 32 bytes each
    const uint32_t wrows = TILED ? min((p.N + 31u) / 32u * 32u - n0, (uint32_t)BN) : min(p.N - n0, (uint32_t)BN);
    const __amdgpu_buffer_rsrc_t rW = make_rsrc(p.B + (uint64_t)n0 * p.K, wrows * p.K);
    const __amdgpu_buffer_rsrc_t rX = make_rsrc(p.A + (uint64_t)m0 * p.K, min(p.M - m0, (uint32_t)BM) * p.K);

    // K % 32 == 0, so a 16-byte piece is all inside a row or all past its end; pieces past K (in the last chunk, or of
    // chunks past the last) are redirected out of the descriptor's range and read as zero
    uint32_t wrow[TN];
#pragma unroll
    for (int t = 0; t < TN; ++t)
        wrow[t] = TILED ? (wave * (32 * TN) + t * 32) * p.K + lane * 16 : (wave * (32 * TN) + t * 32 + l32) * p.K + h * 16;
    auto load_w = [&](int t, int s, uint32_t c) -> v4i {
        const uint32_t k = c * kChunk + s * 32;  // + h*16 < K  <=>  k < K
        // tiled: the fragment of (tile, step) is 1 KB in lane order, steps one after the other
        return __builtin_bit_cast(v4i, buf_load16(rW, k < p.K ? wrow[t] + (TILED ? k * 32 : k) : kOobOffset, 0));
    };
    uint32_t xrow[NXP], xlds[NXP];
    const uint32_t xpiece = tid % PPR;
#pragma unroll
    for (int j = 0; j < NXP; ++j) {
        const uint32_t row = tid / PPR + j * (256 / PPR);
        xrow[j] = row * p.K + xpiece * 16;
        xlds[j] = row * kStride + xpiece * 16;
    }
    auto load_x = [&](int j, uint32_t c) -> v4u {
        const uint32_t k = c * kChunk;
        return buf_load16(rX, k + xpiece * 16 < p.K ? xrow[j] + k : kOobOffset, 0);
    };
    // fragment of rows b*32 + l32, step s: bytes [32*s + 16*h, +16) of the row's chunk
    const uint32_t frag = l32 * kStride + h * 16;
    auto read_x = [&](uint32_t buf, int b, int s) -> v4i {
        return *reinterpret_cast<const v4i *>(lds + buf + frag + b * 32 * kStride + s * 32);
    };

    constexpr int WR = 1;  // chunks of weights in flight (2 measured no faster: the loop is bound by bytes per cycle, not by latency)
    v4i wreg[WR][TN][NS];
    v4u xreg[NXP];
    v4i fx[2][TM];
    v16i32 acc[TN][TM];
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
        for (int b = 0; b < TM; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[t][b][r] = 0;

    // ---- epilogue parameters first: their latency disappears behind the loop
    constexpr uint32_t kLanesPerRow = 8 * TN, kRowsPerStore = 64 / kLanesPerRow;  // a staged row is 128 * TN bytes
    const uint32_t c16 = lane % kLanesPerRow, r4 = lane / kLanesPerRow;
    const uint32_t n_out = n0 + wave * (32 * TN) + c16 * 4;  // first of the four output columns this lane stores
    float sc[4], zc[4], bs[4];
    if (FUSED) {
        if (tid < BM) {
            const uint32_t m = min(m0 + tid, p.M - 1);
            row_par[tid] = p.epi.s_row[m];
            row_par[BM + tid] = p.epi.z_row[m];
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t nn = min(n_out + r, p.N - 1);
            sc[r] = p.epi.s_col[nn];
            zc[r] = p.epi.z_col[nn];
            bs[r] = BIAS ? p.epi.bias[nn] : 0.f;
        }
    }

    // ---- prologue: activations of chunks 0 and 1 -> LDS, chunk 2 -> registers; weights of chunk 0
#pragma unroll
    for (int q = 0; q < 2; ++q) {
#pragma unroll
        for (int j = 0; j < NXP; ++j) xreg[j] = load_x(j, q);
#pragma unroll
        for (int j = 0; j < NXP; ++j) *reinterpret_cast<v4u *>(lds + q * kBuf + xlds[j]) = xreg[j];
    }
    // issued in the order of the main loop's chunks, so that the loop's wait counts are the same on entry and on
    // the back edge (the compiler takes the stricter of the two)
#pragma unroll
    for (int w = 0; w < WR; ++w) {
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            if (TM == 1) {
#pragma unroll
                for (int t = 0; t < TN; ++t) wreg[w][t][s] = load_w(t, s, w);
            }
            if (w == WR - 1) {
#pragma unroll
                for (int j = 0; j < NXP; ++j)
                    if (j * NS / NXP == s) xreg[j] = load_x(j, 2);
            }
            if (TM != 1) {
#pragma unroll
                for (int t = 0; t < TN; ++t) wreg[w][t][s] = load_w(t, s, w);
            }
        }
    }
    lds_barrier8();
#pragma unroll
    for (int b = 0; b < TM; ++b) fx[0][b] = read_x(0, b, 0);

    uint32_t cur = 0, nxt = kBuf, nx2 = 2 * kBuf;
    auto chunk = [&](auto par, uint32_t c) {
        constexpr int W = decltype(par)::value % WR;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
#pragma unroll
            for (int b = 0; b < TM; ++b) {
#pragma unroll
                for (int t = 0; t < TN; ++t) {
                    asm volatile("v_mfma_i32_32x32x32_i8 %0, %1, %2, %0"
                                 : "+a"(acc[t][b])
                                 : "v"(wreg[W][t][s]), "v"(fx[s & 1][b]));
                    __builtin_amdgcn_sched_barrier(0);
                    // ---- side work in the shadow of this MFMA
                    if (t == 0)  // next step's fragment of this row tile (the next chunk's first step comes from `nxt`)
                        fx[(s + 1) & 1][b] = s + 1 < NS ? read_x(cur, b, s + 1) : read_x(nxt, b, 0);
                    if (b == TM - 1)  // last use of this step's weight register: refetch it for the next chunk
                        wreg[W][t][s] = load_w(t, s, c + WR);
                    // activation pieces: chunk c+2 -> its LDS buffer, then fetch chunk c+3; the pieces of a step in
                    // one slot, or (TM = 8: two pieces per step) in slots of their own
                    if (t == TN - 1 && (TM == 8 || b == 0)) {
#pragma unroll
                        for (int j = 0; j < NXP; ++j)
                            if (j * NS / NXP == s && (TM != 8 || b == 2 + 4 * (j % 2))) {
                                *reinterpret_cast<v4u *>(lds + nx2 + xlds[j]) = xreg[j];
                                xreg[j] = load_x(j, c + 3);
                            }
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
        // the MFMAs are opaque to the compiler's hazard tracking: accumulator copies at a join must find them retired
        asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
        lds_barrier8();
        const uint32_t t = cur;
        cur = nxt;
        nxt = nx2;
        nx2 = t;
    };
    using Even = std::integral_constant<int, 0>;
    using Odd = std::integral_constant<int, 1>;
    uint32_t c = 0;
    for (; c + 1 < nchunks; c += 2) {  // no branch inside the loop (the compiler's load counting stays exact)
        chunk(Even{}, c);
        chunk(Odd{}, c + 1);
    }
    if (c < nchunks) chunk(Even{}, c);
    asm volatile("s_nop 15\n\ts_nop 15\n\ts_nop 15" ::: "memory");

    // ---- epilogue.  In the accumulators a lane holds row l32 and, for column tile t and q = 0..3, the four
    // consecutive columns 32*t + 8*q + 4*h + (0..3): stored from there, one instruction would touch 32 rows with 32
    // bytes each.  Each wavefront turns its 32 x 64 block around in its own piece of LDS (the loop's buffers are free
    // after the last barrier) so that a store instruction writes whole rows of 256 (128) contiguous bytes.
    uint8_t *stage = lds + wave * (32 * kEStride);
    const bool whole = n_out + 3 < p.N;
#pragma unroll
    for (int b = 0; b < TM; ++b) {
#pragma unroll
        for (int t = 0; t < TN; ++t)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                *reinterpret_cast<v4i *>(stage + l32 * kEStride + (t * 32 + q * 8 + h * 4) * 4) =
                    v4i{acc[t][b][q * 4], acc[t][b][q * 4 + 1], acc[t][b][q * 4 + 2], acc[t][b][q * 4 + 3]};
        const uint32_t mb = m0 + b * 32;
        const __amdgpu_buffer_rsrc_t rY = out_rows<FUSED>(p, mb, 32);
#pragma unroll
        for (int it = 0; it < 32 / (int)kRowsPerStore; ++it) {
            const uint32_t row = it * kRowsPerStore + r4;
            v4i a = *reinterpret_cast<const v4i *>(stage + row * kEStride + c16 * 16);
            if (FUSED) {
                const float sr = row_par[b * 32 + row], zr = row_par[BM + b * 32 + row];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float o = dequant_hprec_one(a[r], sr, zr, sc[r], zc[r]);
                    if (BIAS) o = o + bs[r];
                    a[r] = __builtin_bit_cast(int, o);
                }
            }
            store_quad8(p, rY, row, n_out, whole, a);
        }
    }
}

template <int TM, int TN, bool FUSED, bool BIAS, bool TILED>
__global__ __launch_bounds__(256) void gemm_s8_kernel(DUQ_HEAD_DECL, Gemm8Params tail)
{
    Gemm8Params p = with_head(tail, DUQ_HEAD_USE);
    to_global(p.A);
    to_global(p.B);
    to_global(p.C);
    to_global(p.y);
    __shared__ __attribute__((aligned(16))) uint8_t lds[Tile8<TM, TN>::kLds];
    __shared__ float row_par[2 * Tile8<TM, TN>::BM];
    uint32_t tile_m, tile_n;
    tile_of_block(blockIdx.x, p.tiles_m, p.tiles_n, tile_m, tile_n);
    gemm8_tile<TM, TN, FUSED, BIAS, TILED>(p, lds, row_par, tile_m * Tile8<TM, TN>::BM, tile_n * Tile8<TM, TN>::BN);
}

// Rounds that do not come out even: p.tiles_m x p.tiles_n tiles of 128 x 256, as many as fill whole rounds of 256 workgroups,
// and behind them the columns that are left in tiles of 32 * TM x 128 * TN.
template <int TM, int TN, bool BIAS, bool TILED>
__global__ __launch_bounds__(256) void gemm_s8_mixed_kernel(DUQ_HEAD_DECL, Gemm8Params tail)
{
    Gemm8Params p = with_head(tail, DUQ_HEAD_USE);
    to_global(p.A);
    to_global(p.B);
    to_global(p.C);
    to_global(p.y);
    using Rest = Tile8<TM, TN>;
    static_assert(TM < 4, "fits beside nothing larger than the 128 x 256 tile's share of LDS");
    __shared__ __attribute__((aligned(16))) uint8_t lds[Tile8<4, 2>::kLds];
    __shared__ float row_par[2 * 128];
    const uint32_t whole = p.tiles_m * p.tiles_n;
    uint32_t tile_m, tile_n;
    if (blockIdx.x < whole) {
        tile_of_block(blockIdx.x, p.tiles_m, p.tiles_n, tile_m, tile_n);
        gemm8_tile<4, 2, true, BIAS, TILED>(p, lds, row_par, tile_m * 128, tile_n * 256);
    } else {
        const uint32_t n1 = p.tiles_n * 256;
        tile_of_block(blockIdx.x - whole, (p.M + Rest::BM - 1) / Rest::BM, (p.N - n1 + Rest::BN - 1) / Rest::BN, tile_m, tile_n);
        gemm8_tile<TM, TN, true, BIAS, TILED>(p, lds, row_par, tile_m * Rest::BM, n1 + tile_n * Rest::BN);
    }
}

// ---------------------------------------------------------------------------------
// split kernel (17 to some hundred rows, one round of its tiles): a 64 x 64 tile per workgroup
// ---------------------------------------------------------------------------------
// Such launches have fewer 64 x 128 tiles than CUs and last as long as one workgroup's walk over K.  Here eight
// wavefronts each take one of the eight 32-k steps of every 256-k chunk for the whole tile (2 x 2 MFMA tiles), which is
// twice the workgroups and an eighth of the walk.  Both operands go to LDS without registers, four chunks in flight; a
// row's sixteen 16-byte pieces lie at piece ^ (row % 16) (the load instruction puts lane l's bytes 16 * l behind its base,
// so the lane's source swizzles), tiled weights in their own fragment order.  The sums meet in LDS with integer adds, laid
// out so that neither the adds nor the reads that turn them to rows share a bank.
template <bool FUSED, bool BIAS, bool TILED>
__global__ __launch_bounds__(512) void gemm_s8_split_kernel(DUQ_HEAD_DECL, Gemm8Params tail)
{
    Gemm8Params p = with_head(tail, DUQ_HEAD_USE);
    to_global(p.A);
    to_global(p.B);
    to_global(p.C);
    to_global(p.y);
    constexpr uint32_t kStage = 32768, kW = 16384;  // bytes of a chunk; offset of its weights
    constexpr int NST = 4;
    __shared__ __attribute__((aligned(256))) uint8_t lds[NST * kStage];
    uint32_t tile_m, tile_n;
    tile_of_block(blockIdx.x, p.tiles_m, p.tiles_n, tile_m, tile_n);
    const uint32_t m0 = tile_m * 64, n0 = tile_n * 64;
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t l32 = lane & 31u, h = lane >> 5;
    const uint32_t nchunks = (p.K + 255) / 256;

    // ---- global -> LDS: two instructions per operand, wavefront and chunk.  Row-major: rows 4 * (8 * j + wave) .. + 3 of
    // the tile; tiled: this wavefront's own fragments, step `wave` of both 32-row tiles.  K % 32 == 0: a piece is all
    // inside its row or past it, and then reads as zero (as do rows past the descriptor and chunks past the end).
    auto desc = [](const void *base, uint32_t bytes) {
        const uint64_t a = reinterpret_cast<uint64_t>(base);
        return v4u{(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a), (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)(a >> 32) & 0xFFFFu)),
                   (uint32_t)__builtin_amdgcn_readfirstlane((int)bytes), 0x00020000u};
    };
    const uint32_t wrows = TILED ? min((p.N + 31u) / 32u * 32u - n0, 64u) : min(p.N - n0, 64u);
    const v4u dX = desc(p.A + (uint64_t)m0 * p.K, min(p.M - m0, 64u) * p.K);
    const v4u dW = desc(p.B + (uint64_t)n0 * p.K, wrows * p.K);
    const uint32_t lr = wave * 4 + (lane >> 4), piece = (lane & 15u) ^ (lr & 15u);  // (32 * j rows further on: the same)
    const uint32_t row0 = lr * p.K + piece * 16;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds;
    auto to_lds = [&](const v4u d, uint32_t dst, uint32_t off) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(dst), "v"(off), "s"(d) : "memory", "m0");
    };
    auto load = [&](uint32_t c, uint32_t stage) {
        const uint32_t k = c * 256;
        [[maybe_unused]] const bool in_row = k + piece * 16 < p.K, in_step = k + wave * 32 < p.K;
#pragma unroll
        for (uint32_t j = 0; j < 2; ++j) to_lds(dX, lds0 + stage + (j * 8 + wave) * 1024, in_row ? row0 + j * 32 * p.K + k : kOobOffset);
#pragma unroll
        for (uint32_t j = 0; j < 2; ++j)
            if (TILED)
                to_lds(dW, lds0 + stage + kW + (j * 8 + wave) * 1024, in_step ? j * 32 * p.K + k * 32 + wave * 1024 + lane * 16 : kOobOffset);
            else
                to_lds(dW, lds0 + stage + kW + (j * 8 + wave) * 1024, in_row ? row0 + j * 32 * p.K + k : kOobOffset);
    };
    // ---- LDS -> registers: this wavefront's step of the chunk
    const uint32_t pos = ((2 * wave + h) ^ (l32 & 15u)) * 16;
    auto frag = [&](uint32_t base, uint32_t j) { return *reinterpret_cast<const v4i *>(lds + base + (j * 32 + l32) * 256 + pos); };
    v4i fx[2][2], fw[2][2];
    auto read = [&](int set, uint32_t stage) {
#pragma unroll
        for (uint32_t j = 0; j < 2; ++j) {
            fx[set][j] = frag(stage, j);
            fw[set][j] = TILED ? *reinterpret_cast<const v4i *>(lds + stage + kW + (j * 8 + wave) * 1024 + lane * 16) : frag(stage + kW, j);
        }
    };
    v16i32 acc[2][2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[t][b][r] = 0;

    static_assert(NST == 4, "the waits below: two later chunks (eight loads) may be in flight");
#pragma unroll
    for (uint32_t c = 0; c < NST; ++c) load(c, c * kStage);
    // parameters of the outputs this thread stores: four columns, rows tid / 16 and 32 further on
    const uint32_t cg = tid & 15u, n = n0 + cg * 4;
    float sc[4], zc[4], bs[4], sr[2], zr[2];
    if (FUSED) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t nn = min(n + r, p.N - 1);
            sc[r] = p.epi.s_col[nn];
            zc[r] = p.epi.z_col[nn];
            bs[r] = BIAS ? p.epi.bias[nn] : 0.f;
        }
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const uint32_t m = min(m0 + b * 32 + (tid >> 4), p.M - 1);
            sr[b] = p.epi.s_row[m];
            zr[b] = p.epi.z_row[m];
        }
    }
    asm volatile("s_waitcnt vmcnt(12)\n\ts_barrier" ::: "memory");  // chunk 0 is here
    read(0, 0);
    uint32_t cur = 0;
    for (uint32_t c = 0; c < nchunks; c += 2) {  // two chunks per turn for the two register sets; one past the end is zeros
#pragma unroll
        for (int set = 0; set < 2; ++set) {
            // the next chunk is here, and every wavefront has read this one: its place takes the chunk NST further on
            asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)\n\ts_barrier" ::: "memory");
            const uint32_t nxt = cur + kStage == NST * kStage ? 0 : cur + kStage;
            read(set ^ 1, nxt);
            load(c + set + NST, cur);
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int t = 0; t < 2; ++t) acc[t][b] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fw[set][t], fx[set][b], acc[t][b], 0, 0, 0);
            cur = nxt;
        }
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");

    // ---- the eight partial tiles meet: register r of tile (t, b) of all lanes at 64 consecutive integers, lane l at
    // l ^ (4 * (q + 4 * t)) (r = 4 * q + ..), so that the sixteen threads of an output row read sixteen banks apart
    int32_t *const red = reinterpret_cast<int32_t *>(lds);
    auto at = [&](uint32_t t, uint32_t b, uint32_t q, uint32_t r, uint32_t l) { return red + ((b * 2 + t) * 16 + q * 4 + r) * 64 + (l ^ ((q + 4 * t) * 4)); };
#pragma unroll
    for (int pass = 0; pass < 2; ++pass) {
#pragma unroll
        for (int g = 0; g < 4; ++g)
            if (((uint32_t)g == wave) == (pass == 0))
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    int32_t *const d = at(g & 1, g >> 1, r >> 2, r & 3, lane);
                    if (pass == 0)
                        *d = acc[g & 1][g >> 1][r];
                    else
                        __hip_atomic_fetch_add(d, acc[g & 1][g >> 1][r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                }
        __syncthreads();
    }
    const bool whole = n + 3 < p.N;
    const __amdgpu_buffer_rsrc_t rY = out_rows<FUSED>(p, m0, 64);
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        v4i a;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            a[r] = *at(cg >> 3, b, (cg >> 1) & 3u, r, (cg & 1u) * 32 + (tid >> 4));
            if (FUSED) {
                float o = dequant_hprec_one(a[r], sr[b], zr[b], sc[r], zc[r]);
                if (BIAS) o = o + bs[r];
                a[r] = __builtin_bit_cast(int, o);
            }
        }
        store_quad8(p, rY, b * 32 + (tid >> 4), n, whole, a);
    }
}

// ---------------------------------------------------------------------------------
// LDS kernel: few rows, and more on narrow problems (what lds8_takes gives it)
// ---------------------------------------------------------------------------------
// The kernels below take their activations (and row-major weights) in the layout of the matrix instruction, sixteen bytes of
// each of sixteen rows from neighbouring lanes, a cache line per lane, which a CU serves at a quarter of its rate; and long
// rows on few columns leave most compute units without a workgroup.  Here both operands come through LDS without registers, in
// whole pieces of a row (tiled weights: in runs of 256 bytes), as in the 4-bit LDS kernel, whose tiles, stages and groups of rows
// these are.  Measured (N x K, tiled weights out of the caches, us): 16 rows 4096 x 4096 6.0 -> 5.4, 4096 x 11008 13.4 -> 11.0 (45 MB: 4.1
// TB/s), 250 x 8192 8.3 -> 6.8; 32 rows 7.2 -> 6.5, 19.6 -> 13.6, 12.6 -> 6.6.
template <int MT, int NT, bool FUSED, bool BIAS, bool TILED>
__global__ __launch_bounds__(512) void gemm_s8_lds_kernel(DUQ_HEAD_DECL, Gemm8Params tail)
{
    Gemm8Params p = with_head(tail, DUQ_HEAD_USE);
    to_global(p.A);
    to_global(p.B);
    to_global(p.C);
    to_global(p.y);
    using Tile = LdsTile<MT, NT>;
    constexpr int G = Tile::G, U = Tile::U, L = Tile::L, DEPTH = Tile::DEPTH;
    constexpr uint32_t RB = Tile::RB, kStage = Tile::kStage;
    constexpr int FT = (MT * NT + 1) / 2;  // output tiles a group of 256 threads finishes
    static_assert(DEPTH >= 2 && DEPTH * L <= 63, "vmcnt");
    __shared__ __attribute__((aligned(256))) uint8_t lds[Tile::kLds];

    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t l16 = lane & 15u, g = lane >> 4;
    // groups of 16 * MT rows share the weights of a column tile: consecutive in `at`, an eighth of which runs on one XCD
    const uint32_t groups = p.tiles_m & 0x1FFu, per_xcd = ((p.N + 16 * NT - 1) / (16 * NT) * groups + 7) / 8;
    const uint32_t at = blockIdx.x % 8 * per_xcd + blockIdx.x / 8, tile = at * (p.tiles_m >> 9) >> 16;  // (tile = at / groups)
    const uint32_t n0 = tile * (16 * NT), m0 = (at - tile * groups) * (16 * MT);
    if (n0 >= p.N) return;
    const auto desc = [](const int8_t *base, uint32_t bytes) {
        const uint64_t a = reinterpret_cast<uint64_t>(base);
        return v4u{(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a), (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)(a >> 32) & 0xFFFFu)),
                   (uint32_t)__builtin_amdgcn_readfirstlane((int)bytes), 0x00020000u};
    };
    const v4u dX = desc(p.A + (uint64_t)m0 * p.K, min(p.M - m0, 16u * MT) * p.K);  // rows past M and N read as zero
    // (tiled: the whole 32-row tile, zero-padded past N, of which NT = 1 takes the lower or the upper half)
    const v4u dW = TILED ? desc(p.B + (uint64_t)(n0 / 32) * 32 * p.K, 32u * p.K) : desc(p.B + (uint64_t)n0 * p.K, min(p.N - n0, 16u * NT) * p.K);

    // ---- global -> LDS: instruction j of a group's wavefront v takes kilobyte j * G + v of the stage, activations first; a
    // row's 16-byte pieces lie at piece ^ (row / Q).  Tiled weights: sixteen rows of a piece side by side, as they come.
    constexpr uint32_t PR = RB / 16, RPI = 64 / PR, Q = RB < 256 ? 256 / RB : 1;  // pieces a row, rows an instruction
    const uint32_t group = G == 1 ? wave : 0, v = G == 1 ? 0 : wave;
    const uint32_t r0 = v * RPI + lane / PR, row0 = r0 * p.K;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds + group * (DEPTH * kStage) + v * 1024;
    auto load = [&](uint32_t step, uint32_t slot) {
        const uint32_t k = (step * (8 / G) + group) * RB;
        uint32_t off[2];  // (of even and odd instructions: rows 16 apart swizzle alike)
        bool in[2];
#pragma unroll
        for (int o = 0; o < 2; ++o) {
            off[o] = k + ((lane % PR) ^ ((o * (G * RPI) + r0) % 16 / Q)) * 16;
            in[o] = off[o] < p.K;  // K % 32 == 0: a 16-byte piece is all in or all out
        }
#pragma unroll
        for (int j = 0; j < L; ++j) {
            const int jw = j - MT * U;
            uint32_t from = kOobOffset;
            if (TILED && jw >= 0) {
                const uint32_t piece = (uint32_t)(jw % U * G + v) * 4 + (lane >> 4), half = NT == 2 ? (uint32_t)(jw / U) : n0 / 16 & 1u;
                if (k + piece * 16 < p.K) from = (k / 32 + piece / 2) * 1024 + ((piece & 1u) * 32 + half * 16 + l16) * 16;
            } else if (in[j % 2]) {
                from = row0 + (uint32_t)(jw < 0 ? j : jw) * (G * RPI) * p.K + off[j % 2];
            }
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(lds0 + slot + j * (G * 1024)), "v"(from),
                         "s"(jw < 0 ? dX : dW)
                         : "memory", "m0");
        }
    };
    static_assert(G * RPI == 8 || G * RPI == 16, "the two swizzles above");
    // ---- LDS -> registers: 64 bytes of a row make a fragment
    v4i x[MT][U], w[NT][U];
    const uint8_t *const own = lds + group * (DEPTH * kStage);
    auto read = [&](uint32_t slot) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t piece = (v * U + u) * 4 + g, swizzled = l16 * RB + (piece ^ (l16 / Q)) * 16;
#pragma unroll
            for (int n = 0; n < NT; ++n)
                w[n][u] = *reinterpret_cast<const v4i *>(own + slot + (MT + n) * (16 * RB) + (TILED ? piece * 256 + l16 * 16 : swizzled));
#pragma unroll
            for (int m = 0; m < MT; ++m) x[m][u] = *reinterpret_cast<const v4i *>(own + slot + m * (16 * RB) + swizzled);
        }
    };
    v4i acc[NT][MT];
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[n][m] = v4i{0, 0, 0, 0};
    const uint32_t steps = (p.K + 8 / G * RB - 1) / (8 / G * RB);
#pragma unroll
    for (int s = 0; s < DEPTH; ++s) load(s, s * kStage);

    // the parameters of the outputs this thread finishes, behind the first steps' operands
    const uint32_t src_lane = (tid >> 2) & 63u, er = tid & 3u, fg = tid >> 8;
    const uint32_t my_m = m0 + (src_lane & 15u), my_c = n0 + (src_lane >> 4) * 4 + er;
    float sc[FT], zc[FT], bs[FT], sr[FT], zr[FT];
    if (FUSED) {
#pragma unroll
        for (int f = 0; f < FT; ++f) {
            const uint32_t t = min(fg + 2 * f, (uint32_t)(MT * NT - 1));
            const uint32_t n = min(my_c + t / MT * 16, p.N - 1), m = min(my_m + t % MT * 16, p.M - 1);
            sc[f] = p.epi.s_col[n];
            zc[f] = p.epi.z_col[n];
            bs[f] = BIAS ? p.epi.bias[n] : 0.f;
            sr[f] = p.epi.s_row[m];
            zr[f] = p.epi.z_row[m];
        }
    }
    uint32_t slot = 0;
    for (uint32_t st = 0; st < steps; ++st) {
        // this step's loads are here (those of the next DEPTH - 1 may be in flight; other loads only make the wait longer)
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((DEPTH - 1) * L) : "memory");
        if (G > 1) asm volatile("s_barrier" ::: "memory");  // (and everybody's)
        read(slot);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // read: the place takes the step DEPTH further on
        if (G > 1) asm volatile("s_barrier" ::: "memory");
        load(st + DEPTH, slot);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int n = 0; n < NT; ++n) acc[n][m] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[n][u], x[m][u], acc[n][m], 0, 0, 0);
        slot = slot + kStage == DEPTH * kStage ? 0 : slot + kStage;
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    v4i *const part = reinterpret_cast<v4i *>(lds);
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < MT; ++m) part[((n * MT + m) * 8 + wave) * 64 + lane] = acc[n][m];
    __syncthreads();
    const int *const sums = reinterpret_cast<const int *>(lds) + src_lane * 4 + er;
#pragma unroll
    for (int f = 0; f < FT; ++f) {
        const uint32_t t = fg + 2 * f;
        if (t < (uint32_t)(MT * NT)) {
            int sum = 0;
#pragma unroll
            for (int i = 0; i < 8; ++i) sum += sums[(t * 8 + i) * 256];
            const uint32_t m = my_m + t % MT * 16, n = my_c + t / MT * 16;
            if (m < p.M && n < p.N) {
                if (FUSED) {
                    float o = dequant_hprec_one(sum, sr[f], zr[f], sc[f], zc[f]);
                    if (BIAS) o = o + bs[f];
                    p.y[(uint64_t)m * p.N + n] = o;
                } else {
                    p.C[(uint64_t)m * p.N + n] = sum;
                }
            }
        }
    }
}

// Shapes of the LDS kernel.  Measured against the kernels that would run otherwise, every weight out of the caches (a pool of 720 MB,
// 640 MB of other data read before each run: with a few copies of the weight 16 x 11008 x 4096 seemed 10.9 -> 10.4 us and is
// 10.7 -> 12.8), on 5400 shapes each of the tiled copy and the weight as stored, times as fast:
//  - one round of workgroups: the weight as stored, a cache line per lane in the other kernels, 1.0 - 3.6; the copy with rows in
//    several groups 1.05 - 3.0, and with rows longer than 4096 elements, which the decode kernel does not hold, 1.0 - 3.5 (up
//    to four rows of 16384 elements 0.9 - 1.15).
//  - tiled, rows in one group of up to 4096 elements, whose decode kernel keeps the activations of up to 2048 or 4096 elements in
//    registers: ahead or level where those are not full (16 x 4096 columns: K 512 / 1024 / 2080 / 4096 1.04 / 1.07 / 1.12 /
//    1.11, but 1248 0.95 (most of a stage is padding) and 2048 0.93; 24 rows 1.0 / 1.0 / 0.98 / 1.10 / 1.08, 2048 0.91), with two column tiles a workgroup (more than 4096 columns) only for short
//    rows, registers that are half empty, or many rows (8192 columns: 16 x 1024 1.03, x 2080 1.05, x 4096 0.95; 32 x 512 1.03, x 2560
//    1.05, x 4096 0.93; 64 x 2560 1.24, x 4096 1.18; 40 x 3072 1.03, x 4096 0.96).
//  - up to 16 rows in several rounds, the last of which may leave most compute units idle (9000 columns: 282 workgroups): the weight as
//    stored 0.97 - 2.0 (16384 x 4096 0.93); the copy 1.01 - 1.25 up to 768 elements and 16384 columns (1024 .. 4096: 0.8 - 1.1)
//    and 1.0 - 1.6 from 4097 to 6144; longer rows, against the skinny kernel, 0.94 - 1.2 at eight rows (11008 x 8192 0.98, 13824
//    x 8192 1.13, x 16384 0.85 - 1.12) and 1.0 - 1.35 at sixteen, less where the second round is a few workgroups (8200 columns:
//    0.88 at eight, 0.93 - 1.1 at twelve).
inline bool lds8_takes(uint32_t M, uint32_t N, uint32_t K, bool tiled)
{
    if (M == 0 || (M < 5 && K <= 4096) || K == 0 || K > 65536 || ((uint64_t)N + 32) * K >= 0xFFFFFF00ull) return false;
    const LdsShape t = lds_shape(M, N);
    if (t.rows == 0) return false;
    const uint32_t groups = (M + 16 * t.rows - 1) / (16 * t.rows);
    const uint64_t workgroups = (uint64_t)groups * ((N + 16 * t.cols - 1) / (16 * t.cols));
    if (workgroups > 256) {
        if (M > 16 || N > 65536) return false;
        if (!tiled) return N <= 12288 || K <= 2560 || K > 4096;
        if (K <= 4096) return K <= 768 && N <= 16384;
        return K <= 7168 || M > 8 || (workgroups > 272 && K <= 12288);
    }
    if (!tiled || groups > 1) return true;
    if (K > 4096) return M > 4 || K <= 12288;
    if (K > 2048) return t.cols == 1 || K <= 2560 || M > 40 || (M > 32 && K <= 3072);
    return K <= (t.cols == 1 || M <= 16 || M > 48 ? 1024u : 512u) || (t.cols == 1 && M <= 16 && K > 1536 && (K <= 1920 || M <= 12));
}

template <bool FUSED, bool BIAS, bool TILED>
static void launch_lds8(Gemm8Params &p, hipStream_t stream)
{
    const LdsShape t = lds_shape(p.M, p.N);
    // groups of rows, and 2^16 over them: (at * m) >> 16 == at / groups while at * (groups - 1) < 2^16 (one round)
    const uint32_t groups = (p.M + 16 * t.rows - 1) / (16 * t.rows), tiles = (p.N + 16 * t.cols - 1) / (16 * t.cols);
    p.tiles_m = groups | ((65535 + groups) / groups) << 9;
    const dim3 grid((tiles * groups + 7) / 8 * 8);
#define DUQ_LDS8(MT)                                                                                                            \
    if (t.rows == MT && t.cols == 1) DUQ_LAUNCH_HEAD((gemm_s8_lds_kernel<MT, 1, FUSED, BIAS, TILED>), grid, dim3(512), 0, stream, p); \
    if (t.rows == MT && t.cols == 2) DUQ_LAUNCH_HEAD((gemm_s8_lds_kernel<MT, 2, FUSED, BIAS, TILED>), grid, dim3(512), 0, stream, p);
    DUQ_LDS8(1)
    DUQ_LDS8(2)
    DUQ_LDS8(3)
    DUQ_LDS8(4)
#undef DUQ_LDS8
}

// ---------------------------------------------------------------------------------
// skinny kernel (M <= 32): bound by reading the weight once from HBM
// ---------------------------------------------------------------------------------
// A workgroup owns 16 weight rows; its four wavefronts split K in contiguous quarters and meet in LDS at the end, so
// N / 16 workgroups fill the chip at decode sizes.  v_mfma_i32_16x16x64_i8 with the weights on the "A" side: lane
// (r = lane % 16, kb = lane / 16) holds 16 bytes of row r at k = 64*j + 16*kb for step j, from the row-major weight
// (16 rows x 64 contiguous bytes per load) or from the tiled copy (four runs of 256 contiguous bytes per load).  The
// activations (MT tiles of 16 rows) use the same layout on the "B" side, straight from global memory: they are
// small and stay in L2.  A ring of kSkinnyRing steps per operand is in flight per lane and each register is
// refetched right after its MFMA, so the whole K quarter of a 4096-long row is requested before the first MFMA.
constexpr int kSkinnyRing = 16;

template <int MT, bool FUSED, bool BIAS, bool TILED>
__global__ __launch_bounds__(256) void gemm_s8_skinny_kernel(DUQ_HEAD_DECL, Gemm8Params tail)
{
    Gemm8Params p = with_head(tail, DUQ_HEAD_USE);
    to_global(p.A);
    to_global(p.B);
    to_global(p.C);
    to_global(p.y);
    __shared__ v4i part[4][MT][64];
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63u, wave = tid >> 6;
    const uint32_t l16 = lane & 15u, kb = lane >> 4;
    const uint32_t n0 = blockIdx.x * 16;
    const uint32_t steps = (p.K + 63) / 64;
    const uint32_t spw = (steps + 3) / 4;  // steps per wavefront
    const uint32_t j0 = wave * spw;

    // row-major: the descriptor covers this workgroup's rows (rows past N read as zero).  Tiled: it covers the 32-row
    // tile (zero-padded past N) of which these 16 rows are the lower or upper half
    const __amdgpu_buffer_rsrc_t rWt = TILED ? make_rsrc(p.B + (uint64_t)(n0 / 32) * 32 * p.K, 32u * p.K)
                                             : make_rsrc(p.B + (uint64_t)n0 * p.K, min(p.N - n0, 16u) * p.K);
    const __amdgpu_buffer_rsrc_t rX = make_rsrc(p.A, p.M * p.K);  // rows past M read as zero
    const bool wrow_ok = n0 + l16 < p.N;
    // byte offset of this lane's 16 bytes of step j: row-major  r*K + 64*j + 16*kb;
    // tiled (step ks = 2*j + kb/2, half h = kb%2, row r + 16*(n0/16 % 2) of the tile)  ks*1024 + (h*32 + row)*16
    const uint32_t wlane = TILED ? (kb >> 1) * 1024 + ((kb & 1u) * 32 + l16 + (n0 & 16u)) * 16 : l16 * p.K + kb * 16;
    auto load_w = [&](uint32_t j) -> v4i {
        const uint32_t k = j * 64 + kb * 16;
        const bool ok = wrow_ok && j < j0 + spw && k < p.K;
        return __builtin_bit_cast(v4i, buf_load16_aux<DUQ_S8_SKINNY_WLOAD_AUX>(rWt, ok ? wlane + (TILED ? j * 2048 : j * 64) : kOobOffset, 0));
    };
    auto load_x = [&](int mt, uint32_t j) -> v4i {
        const uint32_t k = j * 64 + kb * 16;
        const bool ok = j < j0 + spw && k < p.K;
        return __builtin_bit_cast(v4i, buf_load16(rX, ok ? (mt * 16 + l16) * p.K + k : kOobOffset, 0));
    };

    v4i w[kSkinnyRing], x[MT][kSkinnyRing];
#pragma unroll
    for (int u = 0; u < kSkinnyRing; ++u) {
        w[u] = load_w(j0 + u);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) x[mt][u] = load_x(mt, j0 + u);
    }
    v4i acc[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt] = v4i{0, 0, 0, 0};
    for (uint32_t g = 0; g < spw; g += kSkinnyRing) {
#pragma unroll
        for (int u = 0; u < kSkinnyRing; ++u) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) acc[mt] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[u], x[mt][u], acc[mt], 0, 0, 0);
            const uint32_t j = j0 + g + kSkinnyRing + u;  // past the wavefront's range: reads as zero
            w[u] = load_w(j);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) x[mt][u] = load_x(mt, j);
        }
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) part[wave][mt][lane] = acc[mt];
    __syncthreads();
    // lane (m = lane % 16, q = lane / 16) of tile mt holds C[mt*16 + m][n0 + 4*q + (0..3)]: MT * 64 threads finish
    if (tid >= MT * 64) return;
    const uint32_t mt = tid >> 6;
    v4i sum = part[0][mt][lane];
#pragma unroll
    for (int w2 = 1; w2 < 4; ++w2) {
        const v4i o = part[w2][mt][lane];
#pragma unroll
        for (int r = 0; r < 4; ++r) sum[r] += o[r];
    }
    const uint32_t m = mt * 16 + l16, n = n0 + kb * 4;
    if (m >= p.M || n >= p.N) return;
    const void *outp = FUSED ? (const void *)p.y : (const void *)p.C;
    const bool vec_ok = p.N % 4 == 0 && reinterpret_cast<uintptr_t>(outp) % 16 == 0 && n + 3 < p.N;
    if (FUSED) {
        const float sr = p.epi.s_row[m], zr = p.epi.z_row[m];
        v4f32 v;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t nn = min(n + r, p.N - 1);
            float o = dequant_hprec_one(sum[r], sr, zr, p.epi.s_col[nn], p.epi.z_col[nn]);
            if (BIAS) o = o + p.epi.bias[nn];
            v[r] = o;
        }
        float *dst = p.y + (uint64_t)m * p.N + n;
        if (vec_ok) {
            *reinterpret_cast<v4f32 *>(dst) = v;
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (n + r < p.N) dst[r] = v[r];
        }
    } else {
        int32_t *dst = p.C + (uint64_t)m * p.N + n;
        if (vec_ok) {
            *reinterpret_cast<v4i *>(dst) = sum;
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (n + r < p.N) dst[r] = sum[r];
        }
    }
}

// ---------------------------------------------------------------------------------
// decode kernel (5 <= M <= 64 on the row-major weight): one round of workgroups, activations held in registers
// ---------------------------------------------------------------------------------
// The 4-bit MFMA decode kernel's shape for int8 (src/kernels/gemm.cu:46-81 at small M): eight wavefronts split K
// for one 16-column tile (wavefront v owns the 64-byte row segments [v*SEGS, (v+1)*SEGS)); lane (l16, g) holds
// bytes [g*16, +16) of each segment, of weight row l16 of the tile (MFMA "A" side) and of activation rows
// 16*t + l16 of the MT row tiles ("B" side), the operand layout of v_mfma_i32_16x16x64_i8.  A lane keeps its
// activation fragments in registers for the whole launch and a workgroup owns p.tiles_n consecutive column tiles
// with two tiles' weights in flight (two register sets alternate), so a launch is one round of at most 256
// workgroups and the activations (as many bytes as a tile's weights at 16 rows) enter a CU once.  The partial
// tiles meet in LDS; MT * 64 threads finish four consecutive columns of one row each.
//
// RQ > 0 (1, 2, 4 or 8 rows): p.A holds float32 rows and the workgroup quantizes all of them itself, with the arithmetic of
// the row quantizer, while its weights are on the way: 8 / RQ wavefronts per row, which hold it in registers between the
// statistics and the codes; the codes meet in LDS in place of a launch, a write and a read of their own.  What it costs over
// the GEMM alone is the way of M * K floats into every CU (8 x 4096: 1.8 us of 7.1; the arithmetic is 0.5, in the time of
// the weights).  Weights are requested right behind the rows (with a barrier between the two 7.75).
template <int SEGS, int MT, bool FUSED, bool BIAS, bool TILED, int RQ = 0>
__global__ __launch_bounds__(512) void gemm_s8_decode_kernel(DUQ_HEAD_DECL, Gemm8Params tail)
{
    static_assert(RQ == 0 || (MT == 1 && FUSED), "rows quantized here: one row tile");
    Gemm8Params p = with_head(tail, DUQ_HEAD_USE);
    to_global(p.A);
    to_global(p.B);
    to_global(p.C);
    to_global(p.y);
    constexpr int WAVES = 8;
    __shared__ v4i part[2][MT][WAVES][64];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t l16 = lane & 15u, g = lane >> 4;
    const uint32_t ntiles = (p.N + 15) / 16;
    const uint32_t tile0 = blockIdx.x * p.tiles_n;
    const uint32_t tile_end = min(tile0 + p.tiles_n, ntiles);

    // rows past N read as zero (the tiled copy holds whole 32-row tiles, zero-padded); N * K < 2^32 - 32 * K (launcher)
    const __amdgpu_buffer_rsrc_t rW = make_rsrc(p.B, (TILED ? (p.N + 31u) / 32u * 32u : p.N) * p.K);
    const __amdgpu_buffer_rsrc_t rX = make_rsrc(p.A, p.M * p.K);  // rows past M read as zero
    uint32_t koff[SEGS];  // byte offset inside a row, or out of range for pieces past K (K % 32 == 0 and 16 | off)
#pragma unroll
    for (int u = 0; u < SEGS; ++u) {
        const uint32_t off = (wave * SEGS + u) * 64 + g * 16;
        koff[u] = off < p.K ? off : kOobOffset;
    }
    // row-major: 16 rows x 64 contiguous bytes per load instruction.  Tiled copy (fragments of 32 rows x 32 bytes,
    // 1 KB each in lane order (r, h) -> (h * 32 + r) * 16): the 16 bytes of (row, 64 * j + 16 * g) sit in fragment
    // ks = 2 * j + g / 2 at lane (h = g % 2, r = row % 32): four runs of 256 contiguous bytes per instruction
    auto load_tile = [&](uint32_t tile, v4i(&w)[SEGS]) {
        const uint32_t row = tile * 16 + l16;
        const uint32_t nrows = tile < tile_end ? p.N : 0u;
        const uint32_t base = TILED ? (tile >> 1) * 32u * p.K + (g >> 1) * 1024u + ((g & 1u) * 32u + l16 + (tile & 1u) * 16u) * 16u
                                    : row * p.K;
#pragma unroll
        for (int u = 0; u < SEGS; ++u) {
            const uint32_t off = TILED ? base + (wave * SEGS + u) * 2048u : base + koff[u];
            w[u] = __builtin_bit_cast(v4i, buf_load16_aux<DUQ_S8_DEC_WLOAD_AUX>(rW, (row < nrows && koff[u] != kOobOffset) ? off : kOobOffset, 0));
        }
    };
    // loads in the order their data is needed: activations, the first tile's weights, the finishing threads' row
    // parameters
    v4i x[MT][SEGS];
    v4i w0[SEGS], w1[SEGS];
    // thread (mt = tid / 64, lane) finishes C[mt*16 + l16][tile*16 + 4*g + (0..3)]
    const bool finisher = tid < MT * 64;
    const uint32_t m = wave * 16 + l16;
    float sr = 0.f, zr = 0.f;
    if constexpr (RQ == 0) {
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int u = 0; u < SEGS; ++u)
                x[t][u] = __builtin_bit_cast(v4i, buf_load16(rX, koff[u] != kOobOffset ? (t * 16 + l16) * p.K + koff[u] : kOobOffset, 0));
        load_tile(tile0, w0);
        if (FUSED && finisher) {
            const uint32_t mm = min(m, p.M - 1);
            sr = p.epi.s_row[mm], zr = p.epi.z_row[mm];
        }
    } else {
        constexpr uint32_t kStride = 512 * SEGS + 16;  // bytes of a row of codes: sixteen rows' pieces on all banks
        constexpr int WPR = WAVES / RQ, NV = 2 * SEGS / WPR;
        __shared__ __attribute__((aligned(16))) uint8_t codes[RQ * kStride];
        __shared__ float stat[2][WAVES], rowp[2][RQ];
        const uint32_t r = wave / WPR, part = wave % WPR, nvec = p.K >> 2;
        const __amdgpu_buffer_rsrc_t rF = make_rsrc(p.A, p.M * p.K * 4);
        v4f32 v[NV];  // (pieces past the row end are copies of its last one: no statistic changes, no weight meets their codes)
        auto piece = [&](int i) { return (part * NV + i) * 64 + lane; };
#pragma unroll
        for (int i = 0; i < NV; ++i)
            v[i] = __builtin_bit_cast(v4f32, buf_load16(rF, (min(r, p.M - 1) * nvec + min(piece(i), nvec - 1)) * 16, 0));
        load_tile(tile0, w0);
        load_tile(tile0 + 1, w1);
        float lo = INFINITY, hi = -INFINITY;
        bool nan_seen = false;
#pragma unroll
        for (int i = 0; i < NV; ++i) row_stats8(v[i], lo, hi, nan_seen);
        lo = wave_min_f32(lo);
        hi = wave_max_f32(hi);
        if (__builtin_amdgcn_ballot_w64(nan_seen) != 0) lo = hi = __builtin_nanf("");
        if constexpr (WPR > 1) {
            if (lane == 0) stat[0][wave] = lo, stat[1][wave] = hi;
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // (no wait for the weights)
#pragma unroll
            for (int k = 0; k < WPR; ++k) {
                const float l = stat[0][r * WPR + k], h = stat[1][r * WPR + k];
                nan_seen |= l != l;
                lo = fminf(lo, l);
                hi = fmaxf(hi, h);
            }
            if (__builtin_amdgcn_ballot_w64(nan_seen) != 0) lo = hi = __builtin_nanf("");
        }
        const RowCode8 rc(lo, hi);
        if (part == 0 && lane == 0) rowp[0][r] = rc.s, rowp[1][r] = rc.z;
        auto quantize = [&](auto code4) {
#pragma unroll
            for (int i = 0; i < NV; ++i)
                *reinterpret_cast<uint32_t *>(codes + r * kStride + piece(i) * 4) = code4(v[i]);
        };
        if (__builtin_amdgcn_readfirstlane(rc.fast))
            quantize([&](const v4f32 &q) { return rc.quick4(q); });
        else
            quantize([&](const v4f32 &q) { return rc.slow4(q); });
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
        for (int u = 0; u < SEGS; ++u) {
            x[0][u] = *reinterpret_cast<const v4i *>(codes + min(l16, (uint32_t)RQ - 1) * kStride + (wave * SEGS + u) * 64 + g * 16);
        }
        sr = rowp[0][min(m, (uint32_t)RQ - 1)], zr = rowp[1][min(m, (uint32_t)RQ - 1)];
    }
    const void *outp = FUSED ? (const void *)p.y : (const void *)p.C;
    const bool vec_all = p.N % 4 == 0 && reinterpret_cast<uintptr_t>(outp) % 16 == 0;

    auto compute_tile = [&](uint32_t tile, const v4i(&w)[SEGS], uint32_t buf) {
        const uint32_t n = tile * 16 + g * 4;
        float sc[4], zc[4], bs[4];
        if (FUSED && finisher) {  // requested now, used after the matrix work and the barrier
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t nn = min(n + r, p.N - 1);
                sc[r] = p.epi.s_col[nn];
                zc[r] = p.epi.z_col[nn];
                bs[r] = BIAS ? p.epi.bias[nn] : 0.f;
            }
        }
        v4i acc[MT];
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[t] = v4i{0, 0, 0, 0};
#pragma unroll
        for (int u = 0; u < SEGS; ++u)
#pragma unroll
            for (int t = 0; t < MT; ++t) acc[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[u], x[t][u], acc[t], 0, 0, 0);
#pragma unroll
        for (int t = 0; t < MT; ++t) part[buf][t][wave][lane] = acc[t];
        __syncthreads();
        if (finisher) {
            v4i sum = part[buf][wave][0][lane];
#pragma unroll
            for (int w2 = 1; w2 < WAVES; ++w2) {
                const v4i o = part[buf][wave][w2][lane];
#pragma unroll
                for (int r = 0; r < 4; ++r) sum[r] += o[r];
            }
            if (m < p.M && n < p.N) {
                const bool vec_ok = vec_all && n + 3 < p.N;
                if (FUSED) {
                    v4f32 v;
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        float o = dequant_hprec_one(sum[r], sr, zr, sc[r], zc[r]);
                        if (BIAS) o = o + bs[r];
                        v[r] = o;
                    }
                    float *dst = p.y + (uint64_t)m * p.N + n;
                    if (vec_ok) {
                        *reinterpret_cast<v4f32 *>(dst) = v;
                    } else {
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            if (n + r < p.N) dst[r] = v[r];
                    }
                } else {
                    int32_t *dst = p.C + (uint64_t)m * p.N + n;
                    if (vec_ok) {
                        *reinterpret_cast<v4i *>(dst) = sum;
                    } else {
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            if (n + r < p.N) dst[r] = sum[r];
                    }
                }
            }
        }
    };

    // the partial-sum buffers alternate with the register sets: one barrier per tile
    for (uint32_t t = tile0; t < tile_end; t += 2) {
        if (RQ == 0 || t > tile0) load_tile(t + 1, w1);
        compute_tile(t, w0, 0);
        load_tile(t + 2, w0);
        if (t + 1 < tile_end) compute_tile(t + 1, w1, 1);
    }
}

// shapes the decode kernel takes: up to 64 rows of at most 4096 elements (the activation fragments of more would
// not fit in registers next to two sets of weights; with 8192 it measured slower than the skinny kernel: 11.9
// against 10.5 us at 16 x 4096 x 8192), the weight tensor within 32-bit offsets; above 32 rows only up to 1024
// column tiles (64 rows, N = 28672: the 64-row tiles of the GEMM kernel take 27 us, this kernel 33).  Measured
// on the tiled copy, K = 4096, against the skinny kernel (64 rows: the GEMM kernel): N = 4096 M16 6.5 against
// 6.6 us, M32 7.7 against 8.9, M64 11.8 against 22.3; N = 11008 M16 11.1 against 14.7, M32 12.3 against 21.6, M64
// 17.3 against 24.9; N = 28672 M32 26.6 against 47.5; on the row-major weight it is 5-15 % slower than on the copy.
inline bool decode8_takes(uint32_t M, uint32_t N, uint32_t K)
{
    return M <= 64 && K <= 4096 && (M <= 32 || (N + 15) / 16 <= 1024) && ((uint64_t)N + 32) * K < 0xFFFFFF00ull;
}

template <bool FUSED, bool BIAS, bool TILED>
static void launch_decode8(Gemm8Params &p, hipStream_t stream)
{
    const uint32_t ntiles = (p.N + 15) / 16;
    p.tiles_n = (ntiles + 255) / 256;  // column tiles per workgroup: one round of at most 256 workgroups
    const dim3 grid((ntiles + p.tiles_n - 1) / p.tiles_n);
    const uint32_t mt = (p.M + 15) / 16;
#define DUQ_DEC8(S, T) DUQ_LAUNCH_HEAD((gemm_s8_decode_kernel<S, T, FUSED, BIAS, TILED>), grid, dim3(512), 0, stream, p)
    if (p.K > 2048) {
        if (mt == 1) DUQ_DEC8(8, 1);
        else if (mt == 2) DUQ_DEC8(8, 2);
        else if (mt == 3) DUQ_DEC8(8, 3);
        else DUQ_DEC8(8, 4);
    } else {
        if (mt == 1) DUQ_DEC8(4, 1);
        else if (mt == 2) DUQ_DEC8(4, 2);
        else if (mt == 3) DUQ_DEC8(4, 3);
        else DUQ_DEC8(4, 4);
    }
#undef DUQ_DEC8
}

// Up to eight float32 rows of at most 4096 elements: quantizer and GEMM in one launch of the decode kernel.  Against two
// launches with the present quantizer, on the tiled copy (up to four rows: on the weight as stored, whose kernel is the faster
// one there), weights rotated over > 512 MB: 1 x 4096 x 4096 5.4 / 6.5 us, 2 rows 5.65 / 6.75, 4 rows 6.2 / 7.4, 8 rows 7.1 / 8.0,
// 8 x 4096 x 2048 4.35 / 6.3, 8 x 11008 x 4096 11.1 / 12.2, 8 x 28672 x 4096 20.7 / 22.0.
bool quantize_gemm8_fuses(uint32_t M, uint32_t N, uint32_t K) { return M <= 8 && K <= 4096 && decode8_takes(M, N, K); }

template <bool BIAS, bool TILED>
static void launch_decode8_rq(Gemm8Params &p, hipStream_t stream)
{
    const uint32_t ntiles = (p.N + 15) / 16;
    p.tiles_n = (ntiles + 255) / 256;
    const dim3 grid((ntiles + p.tiles_n - 1) / p.tiles_n);
#define DUQ_DEC8(S, R) DUQ_LAUNCH_HEAD((gemm_s8_decode_kernel<S, 1, true, BIAS, TILED, R>), grid, dim3(512), 0, stream, p)
#define DUQ_DEC8R(S)                                                                                                    \
    if (p.M == 1) DUQ_DEC8(S, 1);                                                                                       \
    else if (p.M == 2) DUQ_DEC8(S, 2);                                                                                  \
    else if (p.M <= 4) DUQ_DEC8(S, 4);                                                                                  \
    else DUQ_DEC8(S, 8)
    if (p.K > 2048) {
        DUQ_DEC8R(8);
    } else {
        DUQ_DEC8R(4);
    }
#undef DUQ_DEC8R
#undef DUQ_DEC8
}

// x [M,K] float32, 16-byte aligned; a shape that quantize_gemm8_fuses takes
int launch_quantize_gemm_s8(const float *x, const int8_t *B, bool b_tiled, uint32_t M, uint32_t N, uint32_t K, const float *s_col,
                            const float *z_col, const float *bias, float *y, hipStream_t stream)
{
    Gemm8Params p{reinterpret_cast<const int8_t *>(x), B, M, N, K, 0, nullptr, y, 0, Epi8{nullptr, nullptr, s_col, z_col, bias}};
    if (b_tiled)
        bias ? launch_decode8_rq<true, true>(p, stream) : launch_decode8_rq<false, true>(p, stream);
    else
        bias ? launch_decode8_rq<true, false>(p, stream) : launch_decode8_rq<false, false>(p, stream);
    return (int)hipGetLastError();
}

// ---------------------------------------------------------------------------------
// rows kernel: M <= 4 activation rows on the row-major weight, rows of up to XS KB
// ---------------------------------------------------------------------------------
// The 4-bit rows kernel's shape for int8 (src/kernels/gemm.cu:46-81 at M <= 4): v_dot4_i32_i8 straight on the
// operands, a wavefront owns R weight rows and the whole K range (lane l holds bytes [i*1024 + l*16, +16) of each
// row: a load instruction covers 1 KB of one row and an activation register serves R rows), every weight load of
// the workgroup is requested before anything else, the MR * R partial sums of a lane meet the other lanes' through
// the wavefront's own piece of LDS (no barrier) and a few DPP steps.  A workgroup is four wavefronts: 16 (8 for rows
// longer than 4 KB) weight rows.
template <int MR, int XS, bool FUSED, bool BIAS>
__global__ __launch_bounds__(256) void gemv_s8_rows_kernel(DUQ_HEAD_DECL, Gemm8Params tail)
{
    Gemm8Params p = with_head(tail, DUQ_HEAD_USE);
    to_global(p.A);
    to_global(p.B);
    to_global(p.C);
    to_global(p.y);
    constexpr int R = XS <= 4 ? 4 : 2;  // weight rows per wavefront: at most 16 weight registers of 16 bytes per lane
    constexpr int V = MR * R;           // partial sums per lane: 2 .. 16
    constexpr int LPV = 64 / V;         // lanes that finish one sum
    static_assert((MR == 1 || MR == 2 || MR == 4) && MR * XS <= 16, "activation registers per lane");
    __shared__ __attribute__((aligned(16))) int red[4][V * 64];

    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t n0 = (blockIdx.x * 4 + wave) * R;
    // loads in the order their data is needed: the activations, then every weight byte of this wavefront, then the
    // parameters of the output this lane will finish
    const __amdgpu_buffer_rsrc_t rX = make_rsrc(p.A, p.M * p.K);  // rows past M read as zero
    v4u xr[MR][XS];
#pragma unroll
    for (int m = 0; m < MR; ++m)
#pragma unroll
        for (int i = 0; i < XS; ++i) {
            const uint32_t off = i * 1024 + lane * 16;
            xr[m][i] = buf_load16(rX, off < p.K ? m * p.K + off : kOobOffset, 0);  // K % 32 == 0 and 16 | off
        }
    const __amdgpu_buffer_rsrc_t rW = make_rsrc(p.B + (uint64_t)n0 * p.K, min(p.N - min(n0, p.N), (uint32_t)R) * p.K);
    v4u w[R][XS];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int i = 0; i < XS; ++i) {
            const uint32_t off = i * 1024 + lane * 16;
            w[r][i] = buf_load16_aux<DUQ_S8_ROWS_WLOAD_AUX>(rW, off < p.K ? r * p.K + off : kOobOffset, 0);  // rows past N: beyond the descriptor
        }
    const uint32_t myv = lane / LPV, sub = lane % LPV;
    const uint32_t my_m = myv / R, my_n = n0 + myv % R;
    float sr = 0.f, zr = 0.f, sc = 0.f, zc = 0.f, bias = 0.f;
    if (FUSED) {
        const uint32_t mm = min(my_m, p.M - 1), nn = min(my_n, p.N - 1);
        sr = p.epi.s_row[mm], zr = p.epi.z_row[mm], sc = p.epi.s_col[nn], zc = p.epi.z_col[nn];
        if (BIAS) bias = p.epi.bias[nn];
    }

    int acc[MR][R];
#pragma unroll
    for (int m = 0; m < MR; ++m)
#pragma unroll
        for (int r = 0; r < R; ++r) acc[m][r] = 0;
#pragma unroll
    for (int i = 0; i < XS; ++i)
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int m = 0; m < MR; ++m)
#pragma unroll
                for (int d = 0; d < 4; ++d)
                    acc[m][r] = __builtin_amdgcn_sdot4((int)w[r][i][d], (int)xr[m][i][d], acc[m][r], false);

    // the V sums of 64 lanes each: through this wavefront's piece of LDS (a wavefront's LDS operations execute in
    // order: no barrier), V entries per lane back, then log2(LPV) DPP steps
    int *mine = red[wave];
#pragma unroll
    for (int v = 0; v < V; ++v) mine[v * 64 + lane] = acc[v / R][v % R];
    __builtin_amdgcn_wave_barrier();
    int sum = 0;
#pragma unroll
    for (int e = 0; e < V; ++e) sum += mine[lane * V + e];  // = [myv * 64 + sub * V + e]
    // sum over the LPV consecutive lanes of a group (4 .. 32 lanes)
    sum += __builtin_amdgcn_update_dpp(0, sum, 0xB1, 0xF, 0xF, true);                  // quad_perm [1,0,3,2]
    sum += __builtin_amdgcn_update_dpp(0, sum, 0x4E, 0xF, 0xF, true);                  // quad_perm [2,3,0,1]
    if (LPV >= 8) sum += __builtin_amdgcn_update_dpp(0, sum, 0x141, 0xF, 0xF, true);   // row_half_mirror
    if (LPV >= 16) sum += __builtin_amdgcn_update_dpp(0, sum, 0x140, 0xF, 0xF, true);  // row_mirror
    if (LPV >= 32) sum += __shfl_xor(sum, 16, kWave);
    if (sub == 0 && my_m < p.M && my_n < p.N) {
        if (FUSED) {
            float o = dequant_hprec_one(sum, sr, zr, sc, zc);
            if (BIAS) o = o + bias;
            p.y[(uint64_t)my_m * p.N + my_n] = o;
        } else {
            p.C[(uint64_t)my_m * p.N + my_n] = sum;
        }
    }
}

template <int MR, bool FUSED, bool BIAS>
static void launch_rows8(const Gemm8Params &p, hipStream_t stream)
{
    const uint32_t xs = (p.K + 1023) / 1024;
#define DUQ_ROWS8K(XS)                                                                                              \
    DUQ_LAUNCH_HEAD((gemv_s8_rows_kernel<MR, XS, FUSED, BIAS>), dim3((p.N + 4 * (XS <= 4 ? 4 : 2) - 1) / (4 * (XS <= 4 ? 4 : 2))), \
                       dim3(256), 0, stream, p)
    if (xs <= 2) DUQ_ROWS8K(2);
    else if (xs <= 4) DUQ_ROWS8K(4);
    else if constexpr (MR <= 2) DUQ_ROWS8K(8);
#undef DUQ_ROWS8K
}

// shapes the rows kernel takes: row-major weight, up to four rows of at most 4096 elements (two rows: 8192), the
// weight tensor within 32-bit offsets per descriptor (a descriptor covers one wavefront's rows)
inline bool rows8_takes(uint32_t M, uint32_t K) { return M <= 4 && K <= (M <= 2 ? 8192u : 4096u); }
// split kernel: problems of one round of its 64 x 64 tiles, from 33 rows on where the decode kernel does not reach (tiled
// weights, against the 64 x 128, 64 x 256 and 32 x 256 tiles that ran them: 65 x 4096 x 4096 10.7 against 14.75 us, 128 x 4096
// x 11008 29 / 55, 256 x 2048 x 8192 15.8 / 25.3, 256 x 4096 x 4096 11.3 / 12.4, 40 rows of 8192 on N = 8192 22 / 42), rows
// of at least 1536 elements (x 1024: 6.4 - 7.3 us either way).  Of the decode kernel's shapes those of four row tiles on a
// narrow layer (64 x 4096 x 4096 10.4 / 11.85, 64 x 1024 x 4096 10.3 / 11.1, but 64 x 8192 x 4096 15.0 / 13.9, 48 x 4096 x 4096
// 10.1 / 9.3); of the skinny kernel's 17 rows and more on a wide layer (20 x 11008 x 8192 21.5 / 29.2, but 20 x 8192 x 8192
// 22.5 / 21.75).
inline bool split8_takes(uint32_t M, uint32_t N, uint32_t K)
{
    if (M <= 16 || (uint64_t)((M + 63) / 64) * ((N + 63) / 64) > 256) return false;
    if (decode8_takes(M, N, K)) return M > 48 && K > 2048 && N <= 4096;
    return M <= 32 ? N > 8192 : K >= 1536;
}

// a round of 256 x 256 tiles in rounds of 128 x 256 ones (measured 1.86 - 1.97: 4096 x 4096 x 4096 73.4 against
// 74.4 us, 4096 x 11008 x 4096 188 against 202, 4096 x 8192 x 8192 240 against 251)
#ifndef DUQ_S8_COST256
#define DUQ_S8_COST256 1.95f
#endif
// More than 64 rows on at least 160 tiles of 128 x 256.  A round of 256 workgroups lasts as long as its tile, however few
// tiles it has: about f + c * (K / 256) microseconds, measured (one round, K = 1024 / 4096): 128 x 256 14.8 / 34.5, 96 x 256 12.7 /
// 28.2, 64 x 256 10.6 / 23.2, 64 x 128 6.8 / 14.4; the constants below are of a round among others.  So the cheapest of: 128 x 256 tiles; 96 x 256 tiles (2000 x 6000 x 4096 62.5 -> 54.5
// us, 1536 x 4096 x 4096 30.7 -> 28.2); and, where rows are long enough for the ends not to decide and the model has it 5 % ahead,
// whole rounds of 128 x 256 tiles with the columns that are left in one round of smaller tiles behind them, in the same launch
// (2048 x 11008 x 4096 100.4 -> 94.3, 2048 x 5000 x 8192 105 -> 84.5, 1024 x 11008 x 4096 61 -> 52).
struct Plan8 {
    uint32_t rows;                                        // 128 or 96
    uint32_t cols = 0, rest_rows = 0, rest_cols = 0;      // cols > 0: tiles of 256 columns in whole rounds, and the rest's tile
};
inline Plan8 plan_gemm8(uint32_t M, uint32_t N, uint32_t K, bool fused)
{
    const float n = (float)((K + 255) / 256);
    auto tiles = [&](uint32_t rows, uint32_t width, uint32_t from) { return ((M + rows - 1) / rows) * ((N - from + width - 1) / width); };
    auto rounds = [&](uint32_t t) { return (float)((t + 255) / 256); };
    const float round = n * 1.67f + 6.8f, c128 = rounds(tiles(128, 256, 0)) * round, c96 = rounds(tiles(96, 256, 0)) * (n * 1.29f + 5.4f);
    Plan8 best{c96 < c128 ? 96u : 128u};
    float cost = 0.95f * std::min(c96, c128);
    const uint32_t tm = (M + 127) / 128, whole = tiles(128, 256, 0) / 256, cols = whole * 256 / tm;
    if (!fused || whole == 0 || cols * 256 >= N || K < 2048) return best;
    const uint32_t rr[3] = {96, 64, 64}, rc[3] = {256, 256, 128};
    const float c_us[3] = {1.29f, 1.05f, 0.63f}, f_us[3] = {7.5f, 6.4f, 4.4f};
    for (int k = 0; k < 3; ++k) {
        const float c = (float)whole * round + n * c_us[k] + f_us[k];
        if (tiles(rr[k], rc[k], cols * 256) <= 256 && c < cost) {
            cost = c;
            best = Plan8{128, cols, rr[k], rc[k]};
        }
    }
    return best;
}

template <bool FUSED, bool BIAS, bool TILED>
static void launch_plan8(Gemm8Params &p, hipStream_t stream)
{
    const Plan8 plan = plan_gemm8(p.M, p.N, p.K, FUSED);
    p.tiles_m = (p.M + plan.rows - 1) / plan.rows;
    p.tiles_n = (p.N + 255) / 256;
    if constexpr (FUSED) {
        if (plan.cols) {
            p.tiles_n = plan.cols;
            const uint32_t left = p.N - plan.cols * 256;
            const dim3 grid(p.tiles_m * p.tiles_n +
                            ((p.M + plan.rest_rows - 1) / plan.rest_rows) * ((left + plan.rest_cols - 1) / plan.rest_cols));
            if (plan.rest_rows == 96)
                DUQ_LAUNCH_HEAD((gemm_s8_mixed_kernel<3, 2, BIAS, TILED>), grid, dim3(256), 0, stream, p);
            else if (plan.rest_cols == 256)
                DUQ_LAUNCH_HEAD((gemm_s8_mixed_kernel<2, 2, BIAS, TILED>), grid, dim3(256), 0, stream, p);
            else
                DUQ_LAUNCH_HEAD((gemm_s8_mixed_kernel<2, 1, BIAS, TILED>), grid, dim3(256), 0, stream, p);
            return;
        }
    }
    const dim3 grid(p.tiles_m * p.tiles_n);
    if (plan.rows == 96)
        DUQ_LAUNCH_HEAD((gemm_s8_kernel<3, 2, FUSED, BIAS, TILED>), grid, dim3(256), 0, stream, p);
    else
        DUQ_LAUNCH_HEAD((gemm_s8_kernel<4, 2, FUSED, BIAS, TILED>), grid, dim3(256), 0, stream, p);
}

int select_gemm8_kernel(uint32_t M, uint32_t N, uint32_t K, bool tiled)
{
    if (!tiled && rows8_takes(M, K)) return kKernel8Rows;
    if (lds8_takes(M, N, K, tiled)) return kKernel8Lds;
    if (split8_takes(M, N, K)) return kKernel8Split;
    if (decode8_takes(M, N, K)) return kKernel8Decode;
    return M <= 32 ? kKernel8Skinny : kKernel8Tile;
}

template <bool FUSED, bool BIAS, bool TILED>
static void launch_gemm8_variant(Gemm8Params &p, hipStream_t stream)
{
    switch (select_gemm8_kernel(p.M, p.N, p.K, TILED)) {
    case kKernel8Rows:
        if constexpr (!TILED) {
            if (p.M == 1) launch_rows8<1, FUSED, BIAS>(p, stream);
            else if (p.M == 2) launch_rows8<2, FUSED, BIAS>(p, stream);
            else launch_rows8<4, FUSED, BIAS>(p, stream);
        }
        return;
    case kKernel8Lds:
        launch_lds8<FUSED, BIAS, TILED>(p, stream);
        return;
    case kKernel8Split:
        p.tiles_m = (p.M + 63) / 64;
        p.tiles_n = (p.N + 63) / 64;
        DUQ_LAUNCH_HEAD((gemm_s8_split_kernel<FUSED, BIAS, TILED>), dim3(p.tiles_m * p.tiles_n), dim3(512), 0, stream, p);
        return;
    case kKernel8Decode:
        launch_decode8<FUSED, BIAS, TILED>(p, stream);
        return;
    case kKernel8Skinny: {
        const dim3 grid((p.N + 15) / 16);
        if (p.M <= 16)
            DUQ_LAUNCH_HEAD((gemm_s8_skinny_kernel<1, FUSED, BIAS, TILED>), grid, dim3(256), 0, stream, p);
        else
            DUQ_LAUNCH_HEAD((gemm_s8_skinny_kernel<2, FUSED, BIAS, TILED>), grid, dim3(256), 0, stream, p);
        return;
    }
    default: break;
    }
    p.tiles_n = (p.N + 255) / 256;
    // the tallest tile that still gives most of the 256 CUs a workgroup
    const uint32_t t128 = ((p.M + 127) / 128) * p.tiles_n, t64 = ((p.M + 63) / 64) * p.tiles_n;
    const uint32_t t256 = ((p.M + 255) / 256) * p.tiles_n;
    // 256-row tiles where every CU gets one and their rounds (each DUQ_S8_COST256 rounds of 128-row tiles for twice
    // the outputs) come out cheaper
    if (t256 >= 256 && DUQ_S8_COST256 * (float)((t256 + 255) / 256) < (float)((t128 + 255) / 256)) {
        p.tiles_m = (p.M + 255) / 256;
        DUQ_LAUNCH_HEAD((gemm_s8_kernel<8, 2, FUSED, BIAS, TILED>), dim3(p.tiles_m * p.tiles_n), dim3(256), 0, stream, p);
    } else if (p.M > 64 && t128 >= 160) {
        launch_plan8<FUSED, BIAS, TILED>(p, stream);
    } else if (p.M > 32 && t64 >= 48) {
        p.tiles_m = (p.M + 63) / 64;
        // one round of 64 x 256 tiles would leave CUs idle: 64 x 128 tiles, twice as many (measured 21-24 % faster at
        // 128 such tiles, 9 % at 64)
        if (t64 <= 128) {
            p.tiles_n = (p.N + 127) / 128;
            DUQ_LAUNCH_HEAD((gemm_s8_kernel<2, 1, FUSED, BIAS, TILED>), dim3(p.tiles_m * p.tiles_n), dim3(256), 0, stream, p);
        } else {
            DUQ_LAUNCH_HEAD((gemm_s8_kernel<2, 2, FUSED, BIAS, TILED>), dim3(p.tiles_m * p.tiles_n), dim3(256), 0, stream, p);
        }
    } else {
        p.tiles_m = (p.M + 31) / 32;
        DUQ_LAUNCH_HEAD((gemm_s8_kernel<1, 2, FUSED, BIAS, TILED>), dim3(p.tiles_m * p.tiles_n), dim3(256), 0, stream, p);
    }
}

int launch_gemm_s8(const int8_t *A, const int8_t *B, bool b_tiled, uint32_t M, uint32_t N, uint32_t K, int32_t *C,
                   const float *s_row, const float *z_row, const float *s_col, const float *z_col, const float *bias,
                   float *y, hipStream_t stream)
{
    if (M == 0 || N == 0) return 0;
    Gemm8Params p{A, B, M, N, K, 0, C, y, 0, Epi8{s_row, z_row, s_col, z_col, bias}};
    if (C)
        launch_gemm8_variant<false, false, false>(p, stream);
    else if (b_tiled && bias)
        launch_gemm8_variant<true, true, true>(p, stream);
    else if (b_tiled)
        launch_gemm8_variant<true, false, true>(p, stream);
    else if (bias)
        launch_gemm8_variant<true, true, false>(p, stream);
    else
        launch_gemm8_variant<true, false, false>(p, stream);
    return (int)hipGetLastError();
}

// ---------------------------------------------------------------------------------
// weight [N, K] row-major -> tiled: [ceil(N/32)][K/32][64 lanes][16 bytes], lane (r = lane % 32, h = lane / 32) of
// tile (nt, ks) holding W[32*nt + r][32*ks + 16*h, +16) (zero past row N): each MFMA weight fragment is then one
// contiguous kilobyte, eight cache lines per load instruction instead of thirty-two
// ---------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void weight_tile8_kernel(const int8_t *w, uint32_t N, uint32_t K, int8_t *out)
{
    const uint32_t ksteps = K / 32;
    const uint64_t pieces = (uint64_t)((N + 31) / 32) * ksteps * 64;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < pieces; i += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t ln = (uint32_t)(i & 63u);
        const uint64_t tile = i >> 6;
        const uint32_t ks = (uint32_t)(tile % ksteps), nt = (uint32_t)(tile / ksteps);
        const uint32_t row = nt * 32 + (ln & 31u), k = ks * 32 + (ln >> 5) * 16;
        v4u v = {0u, 0u, 0u, 0u};
        if (row < N) v = *reinterpret_cast<const v4u *>(w + (uint64_t)row * K + k);
        reinterpret_cast<v4u *>(out)[i] = v;
    }
}

int launch_weight_tile8(const int8_t *w, uint32_t N, uint32_t K, int8_t *out, hipStream_t stream)
{
    if (N == 0 || K == 0) return 0;
    const uint64_t pieces = (uint64_t)((N + 31) / 32) * (K / 32) * 64;
    const uint32_t blocks = (uint32_t)std::min<uint64_t>((pieces + 255) / 256, 1u << 20);
    hipLaunchKernelGGL(weight_tile8_kernel, dim3(blocks), dim3(256), 0, stream, w, N, K, out);
    return (int)hipGetLastError();
}

}  // namespace duq
