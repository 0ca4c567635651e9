// Packed-int4 x packed-int4 -> int32 GEMM for gfx950 on v_mfma_i32_16x16x64_i8, with the
// fp16 dequant epilogue fused in (or raw int32 accumulators out).
//
//   C[m,n] = sum_k s4(A[m,k]) * s4(B[n,k])        (src/kernels/gemm.cu:8-43 of the reference)
//
// Nibble -> byte: for a packed word w, (w & 0xF0F0F0F0) holds the four odd-k nibbles as
// bytes equal to 16*s4 (sign included), ((w << 4) & 0xF0F0F0F0) the four even-k ones.
// Both operands are expanded the same way, so every MFMA product is 256*a*b and the
// accumulator is 256*C exactly; one arithmetic shift by 8 recovers C.  |C| <= 64*K, so
// 256*|C| stays below 2^31 for K <= 131008.  Integer accumulation is order-free, so the
// k order inside a tile only has to be the same for A and B.
//
// Four kernels here, and the prefill kernel in duq_prefill.hip, picked by shape in gemm_kernel_for() (up to 64 rows,
// and more on narrow problems, run the kernels of duq_decode.hip as far as they reach):
//  * prefill kernel (duq_prefill.hip): more than 64 rows, long rows, fewer rows on wide layers, tensors of 4 GiB or more,
//    what is left;
//  * stream kernel (the same shapes where rows are short): 64 x 128 tiles, weights from global memory straight to
//    registers, activations expanded once into LDS, v_mfma_i32_32x32x32_i8 with a hand-ordered schedule;
//  * short-row kernel (rows of at most 256 elements): the stream kernel's operand paths without its K pipeline;
//  * skinny kernel (9 <= M <= 16 with 1536 or more column tiles): one workgroup owns 16 output columns, its
//    wavefronts split K, whole-line weight loads turned into fragments through LDS;
//  * dot kernel (M <= 4 with rows of 16385 to 30720 elements, more than 4096 columns): v_dot8_i32_i4 on the packed nibbles, a
//    pure HBM stream.
// In the MFMA kernels the weight operand goes to the MFMA "A" side, so each lane ends up
// with four consecutive output columns of one row.
#include "duq_gemm_common.h"
// Cache policy of the weight loads of the kernels that read every weight byte once: 2 = non-temporal.  Measured:
// skinny kernel 16 x 28672 x 4096 13.2 against 14.1 us, dot kernel 1 x 8192 x 28672 20.9 against 22.8 and 4 x 4096 x
// 20480 11.5 against 13.2.
#ifndef DUQ_SKINNY_WLOAD_AUX
#define DUQ_SKINNY_WLOAD_AUX 2
#endif
#ifndef DUQ_DOT_WLOAD_AUX
#define DUQ_DOT_WLOAD_AUX 2
#endif
#include <type_traits>

namespace duq {

// ---------------------------------------------------------------------------------
// stream kernel (prefill on short rows): weights global -> registers, activations through LDS,
// v_mfma_i32_32x32x32_i8
// ---------------------------------------------------------------------------------
// Tile 64 (M) x 128 (N), 4 wavefronts side by side along N: every wavefront owns 32 weight
// rows that no other wavefront of the workgroup needs, so weight fragments never go through
// LDS: lane (l32, h) loads 16-byte piece i (0..3) = bytes [i*32 + h*16, +16) of the 128-byte
// row segment of a 256-k chunk straight into registers.  The 64 activation rows are shared
// by the four wavefronts: they are expanded to bytes once on the way into LDS (three
// buffers, rows padded to 272 B) and read back as 128-bit fragments.  What bounds it is the wait
// for a chunk's activations, which are loaded and used within one chunk; with two or three workgroups
// on a CU they cover for one another, and with few chunks it matters less than the prefill kernel's
// longer start and end (select_stream_tile draws the line).
//
// The 32x32x32 MFMA keeps the matrix pipe full from a single wavefront per SIMD (32 cycles
// per instruction, 16 per 32768 operations); the 16x16x64 form needs 18 and loses more to
// interleaved vector work.  A chunk is 8 k-steps (piece i, nibble parity) of 2 MFMAs (1
// weight tile x 2 activation tiles).  The order is fixed by hand, a scheduling fence after
// every MFMA, and everything else rides in the MFMA shadows, a few instructions per slot:
//   every step    : the next step's two activation fragments (step 7: the next chunk's);
//   step 2i       : refetch weight piece i for the next chunk (its registers were just
//                   expanded), expand piece i+1;
//   step 1        : fetch the activations two chunks ahead;
//   steps 6, 7    : expand + store those activations into the third LDS buffer;
//   step 6        : expand the next chunk's weight piece 0.
// MFMAs are issued through inline assembly with the accumulators tied to the accumulation
// register file, so they never move.
//
// All global reads are raw buffer loads on per-workgroup descriptors that cover exactly
// the rows of this tile: rows past M or N read as zero without a branch, and the chunk
// offset rides in the scalar offset.  The last chunks use per-piece guarded offsets (a
// piece at or past the row end is redirected out of bounds and reads as zero).
constexpr int kCK = 256;         // k elements per chunk (128 packed bytes per row)
constexpr int kXStride = 272;    // LDS bytes per activation row: 256 expanded + 16 pad


template <int EPI, bool BIAS>
__global__ __launch_bounds__(256) void gemm_s4_stream_kernel(DUQ_HEAD_DECL, GemmParams tail)
{
    GemmParams p = with_head(tail, DUQ_HEAD_USE);
    to_global(p.A);
    to_global(p.B);
    to_global(p.C);
    to_global(p.y);
    constexpr int TM = 2, TN = 1;      // 32-row activation and 32-column weight tiles per wavefront
    constexpr int BM = 32 * TM, BN = 128 * TN;
    constexpr int S = TM * TN;         // MFMA slots per step
    constexpr int NXP = TM;            // 16-byte activation pieces per thread and chunk
    constexpr uint32_t kBuf = BM * kXStride;

    __shared__ __attribute__((aligned(16))) uint8_t lds[3 * kBuf];
    // dual-uniform row-sum epilogue (EPI 5): its parameters, eight words per column of the tile and per row,
    // fetched by the first BN / BM threads before the loop and read back from here after it
    //   column: wlo, whi (first eight bytes of the weight row), s1 | s2 << 16, z1, z2, adj1, adj2, bias
    //   row   : xlo, xhi & 0xFF (first ten codes of the activation row), float(s), z, rx - rxl, rxl
    __shared__ __attribute__((aligned(16))) uint32_t dpar[EPI == 5 ? (BN + BM) * 8 : 4];
    __shared__ uint32_t dwide;  // EPI 5: non-zero when a factor of the corrections leaves the signed 24-bit range

    if (blockIdx.z) batch_shift(p, blockIdx.z);
    uint32_t tile_m, tile_n;
    tile_of_block(blockIdx.x, p.tiles_m, p.tiles_n, tile_m, tile_n);
    const uint32_t m0 = tile_m * BM, n0 = tile_n * BN;
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63u, wave = tid >> 6;
    const uint32_t l32 = lane & 31u, h = lane >> 5;
    const uint32_t wm0 = m0, wn0 = n0 + wave * (32 * TN);
    const uint32_t kbytes = p.K >> 1;
    const uint32_t nfull = p.K / kCK;
    const uint32_t nchunks = (p.K + kCK - 1) / kCK;

    if constexpr (EPI == 5) {
        if (tid == 0) dwide = 0;
        __syncthreads();
        bool wide = false;
        if (tid < (uint32_t)BN) {
            const uint32_t n = min(n0 + tid, p.N - 1);
            const v2u head = *reinterpret_cast<const v2u *>(p.B + (uint64_t)n * kbytes);
            uint32_t *d = dpar + tid * 8;
            d[0] = head[0];
            d[1] = head[1];
            d[2] = (uint32_t)p.epi.s_col_1[n] | ((uint32_t)p.epi.s_col_2[n] << 16);
            d[3] = (uint32_t)rint_i32((float)bits_to_f16(p.epi.z_col_1[n]));
            d[4] = (uint32_t)rint_i32((float)bits_to_f16(p.epi.z_col_2[n]));
            d[5] = (uint32_t)p.epi.rs_col[n];
            d[6] = (uint32_t)p.epi.rs_col_2[n];
            d[7] = BIAS ? (uint32_t)p.epi.bias[n] : 0u;
            wide = !(fits_i24(d[3]) && fits_i24(d[4]) && fits_i24(d[5]) && fits_i24(d[6]));
        }
        if (tid < (uint32_t)BM) {
            const uint32_t m = min(m0 + tid, p.M - 1);
            const v2u head = *reinterpret_cast<const v2u *>(p.A + (uint64_t)m * kbytes);
            const uint32_t xlo = head[0], xhi = head[1] & 0xFFu;  // input columns 0..7 and 8, 9
            const uint32_t rxl = (uint32_t)__builtin_amdgcn_sdot8((int)xhi, 0x11111111, __builtin_amdgcn_sdot8((int)xlo, 0x11111111, 0, false), false);
            uint32_t *d = dpar + (BN + tid) * 8;
            d[0] = xlo;
            d[1] = xhi;
            d[2] = __builtin_bit_cast(uint32_t, (float)bits_to_f16(p.epi.s_row[m]));
            d[3] = (uint32_t)rint_i32((float)bits_to_f16(p.epi.z_row[m]));
            d[4] = (uint32_t)p.epi.rs_row[m] - rxl;
            d[5] = rxl;
            wide = wide || !(fits_i24(d[3]) && fits_i24(d[4]));
        }
        if (wide) dwide = 1;  // (same value from every writer)
        // (the barrier that ends the prologue below orders these writes before the epilogue's reads)
    }

    const __amdgpu_buffer_rsrc_t rW = make_rsrc(p.B + (uint64_t)n0 * kbytes, min(p.N - n0, (uint32_t)BN) * kbytes);
    const __amdgpu_buffer_rsrc_t rX = make_rsrc(p.A + (uint64_t)m0 * kbytes, min(p.M - m0, (uint32_t)BM) * kbytes);

    uint32_t woff[TN];
#pragma unroll
    for (int t = 0; t < TN; ++t) woff[t] = (wave * (32 * TN) + t * 32 + l32) * kbytes + h * 16;
    uint32_t xoff[NXP], xlds[NXP];
    const uint32_t xq = tid & 7u;  // which 16-byte piece of the 128-byte row segment
#pragma unroll
    for (int i = 0; i < NXP; ++i) {
        const uint32_t row = (tid >> 3) + i * 32;
        xoff[i] = row * kbytes + xq * 16;
        xlds[i] = row * kXStride + xq * 32;
    }

    v4u wreg[TN][4];      // raw weight pieces [tile][piece]
    v4u xreg[NXP];        // raw activation pieces
    v4u wexp[2][2][TN];   // expanded weights [piece & 1][parity][tile]
    v4i fx[2][TM];        // activation fragments [step & 1][tile]
    v16i acc[TN][TM];
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
        for (int b = 0; b < TM; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[t][b][r] = 0;

    // fragment of step (i, par) for activation tile b: + b*32*kXStride + i*64 + par*16
    const uint32_t fragX = l32 * kXStride + h * 32;

    auto expand_word = [&](const v4u &raw, v4u &even, v4u &odd, int w) {
        even[w] = (raw[w] << 4) & kNibbleMask;
        odd[w] = raw[w] & kNibbleMask;
    };

    // GUARD = false: every chunk fetched is complete, plain offsets.
    auto body = [&](auto guard, uint32_t c, uint32_t cur, uint32_t nxt, uint32_t nx2) {
        constexpr bool G = decltype(guard)::value;
        const uint32_t koff1 = (c + 1) * (kCK / 2), koff2 = (c + 2) * (kCK / 2);
        const bool okx = !G || (koff2 + xq * 16 < kbytes);  // K % 64 == 0: a piece is all in or all out
        v4u xe, xo;
#pragma unroll
        for (int step = 0; step < 8; ++step) {
            const int i = step >> 1, par = step & 1;
            const bool okw = !G || (koff1 + i * 32 + h * 16 < kbytes);
#pragma unroll
            for (int slot = 0; slot < S; ++slot) {
                const int b = slot / TN, t = slot % TN;
                asm volatile("v_mfma_i32_32x32x32_i8 %0, %1, %2, %0"
                             : "+a"(acc[t][b])
                             : "v"(wexp[i & 1][par][t]), "v"(fx[step & 1][b]));
                __builtin_amdgcn_sched_barrier(0);
                // ---- side work in the shadow of this MFMA
                if (slot < TM) {  // next step's activation fragment for tile `slot`
                    const uint8_t *src = step < 7 ? lds + cur + fragX + ((step + 1) >> 1) * 64 + ((step + 1) & 1) * 16
                                                  : lds + nxt + fragX;
                    fx[(step + 1) & 1][slot] = *reinterpret_cast<const v4i *>(src + slot * 32 * kXStride);
                }
                if (par == 0 && slot < TN)  // piece i was expanded earlier: refetch it for the next chunk
                    wreg[slot][i] = buf_load16(rW, okw ? woff[slot] + i * 32 : kOobOffset, koff1);
                if (step == 1 && slot < NXP)  // activations two chunks ahead
                    xreg[slot] = buf_load16(rX, okx ? xoff[slot] : kOobOffset, koff2);
                // expand the next weight piece of tile `par`: its four words over the last four slots (or
                // two / one per slot when a step has fewer than four slots)
                if (par < TN) {
                    const int np = (i + 1) & 3;  // pieces 1, 2, 3 of this chunk, then piece 0 of the next
#pragma unroll
                    for (int w = 0; w < 4; ++w)
                        if ((S >= 4 ? S - 4 + w : w * S / 4) == slot)
                            expand_word(wreg[par < TN ? par : 0][np], wexp[(i + 1) & 1][0][par < TN ? par : 0],
                                        wexp[(i + 1) & 1][1][par < TN ? par : 0], w);
                }
                if (step >= 8 - NXP) {  // activations two chunks ahead -> third LDS buffer, one piece per step
#pragma unroll
                    for (int w = 0; w < 4; ++w)
                        if ((S >= 4 ? w : w * S / 4) == slot) {
                            expand_word(xreg[step - (8 - NXP)], xe, xo, w);
                            if (w == 3) {
                                *reinterpret_cast<v4u *>(lds + nx2 + xlds[step - (8 - NXP)]) = xe;
                                *reinterpret_cast<v4u *>(lds + nx2 + xlds[step - (8 - NXP)] + 16) = xo;
                            }
                        }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __syncthreads();
    };

    using Plain = std::false_type;
    using Guarded = std::true_type;

    // ---- prologue: chunks 0 and 1 activations -> LDS, chunk 0 weights -> registers
    {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const bool okw = i * 32 + h * 16 < kbytes;
#pragma unroll
            for (int t = 0; t < TN; ++t) wreg[t][i] = buf_load16(rW, okw ? woff[t] + i * 32 : kOobOffset, 0);
        }
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const bool okx = q * (kCK / 2) + xq * 16 < kbytes;
#pragma unroll
            for (int i = 0; i < NXP; ++i) xreg[i] = buf_load16(rX, okx ? xoff[i] : kOobOffset, q * (kCK / 2));
#pragma unroll
            for (int i = 0; i < NXP; ++i) {
                v4u ev, od;
                expand_nibbles(xreg[i], ev, od);
                *reinterpret_cast<v4u *>(lds + q * kBuf + xlds[i]) = ev;
                *reinterpret_cast<v4u *>(lds + q * kBuf + xlds[i] + 16) = od;
            }
        }
#pragma unroll
        for (int t = 0; t < TN; ++t) expand_nibbles(wreg[t][0], wexp[0][0][t], wexp[0][1][t]);
        __syncthreads();
#pragma unroll
        for (int b = 0; b < TM; ++b) fx[0][b] = *reinterpret_cast<const v4i *>(lds + fragX + b * 32 * kXStride);
    }

    // ---- epilogue parameters: fetched now so that their latency hides behind the main loop
    constexpr bool kLdsParams = false;
#include "duq_stream_epilogue_fetch.inc"
    fetch_params();

    uint32_t cur = 0, nxt = kBuf, nx2 = 2 * kBuf;
    auto rotate = [&]() {
        const uint32_t t = cur;
        cur = nxt;
        nxt = nx2;
        nx2 = t;
    };
    uint32_t c = 0;
    for (; c + 2 < nfull; ++c) {  // steady state: chunks c+1 and c+2 are complete ones
        body(Plain{}, c, cur, nxt, nx2);
        rotate();
    }
    for (; c < nchunks; ++c) {  // last chunks: guarded fetches (a fetch past K reads zeros, unused)
        body(Guarded{}, c, cur, nxt, nx2);
        rotate();
    }
    // the MFMAs above are opaque to the compiler's hazard tracking: let the last ones retire
    // before the accumulators are read
    asm volatile("s_nop 15\n\ts_nop 15\n\ts_nop 15" ::: "memory");

    constexpr bool kWideStore = false, kFloatBits = false;
    uint8_t *const wstage = lds + wave * (BM * (64 * TN + 16));
#include "duq_stream_epilogue_store.inc"
}

// ---------------------------------------------------------------------------------
// short-row kernel: K <= 256 (one chunk), many tiles; batched products of short rows
// ---------------------------------------------------------------------------------
// The stream kernel's tile (32*TM rows x 256 columns, four wavefronts side by side along N, weights global ->
// registers, activations expanded into LDS, v_mfma_i32_32x32x32_i8, the same epilogue) without its K pipeline: a
// problem whose rows hold at most 256 elements is one chunk, and a launch is its output stores (a 2048 x 2048 x 128
// product moves 0.5 MB in and 8 MB out).  One activation buffer that doubles as the epilogue's staging area (37 KB
// of LDS at 64 rows), only the steps the row length needs, whole-row stores; up to four workgroups share a CU and
// overlap one another's loads, matrix work and stores.  (Persistent workgroups that request the next tile's operands
// before the current tile's epilogue measured slower, 93 against 86 us on 32 products of 2048 x 2048 x 128: the
// loop-carried wait for those loads also waits for the stores issued after them.)  The epilogue's per-row parameters go
// through LDS, one 16-byte read for four rows, instead of a register per row and parameter: 112 registers instead of
// 148 and no loads of single values at the tile's head (32 products of 2048 x 2048 x 128, asymmetric: 71 -> 67 us;
// K = 64: 60 -> 52).  What bounds it now is the mix: 268 MB of stores take 39 us at the rate of a plain fill, the vector
// work 30 us of issue, and the launch 48 - 58 (into buffers already in the last-level cache, or not).
template <int TM, int EPI, bool BIAS>
__global__ __launch_bounds__(256, 2) void gemm_s4_shortk_kernel(DUQ_HEAD_DECL, GemmParams tail)
{
    GemmParams p = with_head(tail, DUQ_HEAD_USE);
    to_global(p.A);
    to_global(p.B);
    to_global(p.C);
    to_global(p.y);
    constexpr int BM = 32 * TM, BN = 256, TN = 2;
    constexpr int NXP = TM;  // 16-byte activation pieces per thread
    constexpr uint32_t kBuf = BM * kXStride, kStage = 4 * BM * 144;
    __shared__ __attribute__((aligned(16))) uint8_t lds[kBuf > kStage ? kBuf : kStage];
    uint32_t *const dpar = nullptr;  // named by the shared epilogue text for an epilogue this kernel never runs
    const uint32_t dwide = 0;

    if (blockIdx.z) batch_shift(p, blockIdx.z);
    // every XCD a contiguous range of tiles, column blocks fastest: whole output rows leave from one XCD (8 products of 4000 x
    // 4000 x 128: 52.0 -> 48.4 us, 12 of 1111 x 1111 x 128 14.5 -> 14.0, 32 of 2048 x 2048 x 128 49.0 -> 47.9)
    const uint32_t ntiles = p.tiles_m * p.tiles_n, per = ntiles / 8, rem = ntiles % 8, xcd = blockIdx.x % 8, local = blockIdx.x / 8;
    const uint32_t id = xcd < rem ? xcd * (per + 1) + local : rem * (per + 1) + (xcd - rem) * per + local;
    const uint32_t m0 = (id / p.tiles_n) * BM, n0 = (id % p.tiles_n) * BN;
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63u, wave = tid >> 6;
    const uint32_t l32 = lane & 31u, h = lane >> 5;
    const uint32_t wm0 = m0, wn0 = n0 + wave * (32 * TN);
    const uint32_t kbytes = p.K >> 1;  // <= 128

    const __amdgpu_buffer_rsrc_t rW = make_rsrc(p.B + (uint64_t)n0 * kbytes, min(p.N - n0, (uint32_t)BN) * kbytes);
    const __amdgpu_buffer_rsrc_t rX = make_rsrc(p.A + (uint64_t)m0 * kbytes, min(p.M - m0, (uint32_t)BM) * kbytes);

    // weights: lane (l32, h) of weight tile j holds piece i = bytes [i*32 + h*16, +16) of row wave*64 + j*32 + l32
    v4u wreg[TN][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const bool okw = i * 32 + h * 16 < kbytes;  // K % 64 == 0: a piece is all in or all out
#pragma unroll
        for (int j = 0; j < TN; ++j)
            wreg[j][i] = buf_load16(rW, okw ? (wave * 64 + j * 32 + l32) * kbytes + i * 32 + h * 16 : kOobOffset, 0);
    }
    // activations: thread (row = tid / 8 + 32 * j, piece = tid % 8) -> expanded into LDS (pieces past K as zeros)
    const uint32_t xq = tid & 7u;
    v4u xreg[NXP];
#pragma unroll
    for (int j = 0; j < NXP; ++j) {
        const uint32_t row = (tid >> 3) + j * 32;
        xreg[j] = buf_load16(rX, xq * 16 < kbytes ? row * kbytes + xq * 16 : kOobOffset, 0);
    }
    constexpr bool kLdsParams = true;
#include "duq_stream_epilogue_fetch.inc"
    fetch_params();
#pragma unroll
    for (int j = 0; j < NXP; ++j) {
        const uint32_t row = (tid >> 3) + j * 32;
        v4u ev, od;
        expand_nibbles(xreg[j], ev, od);
        *reinterpret_cast<v4u *>(lds + row * kXStride + xq * 32) = ev;
        *reinterpret_cast<v4u *>(lds + row * kXStride + xq * 32 + 16) = od;
    }
    __syncthreads();

    // The accumulators of the binary16 epilogues start at the bits of kF32Base: at most 256 products of at most 64, carried x
    // 256, stay within 2^22, so that they are the float kF32Base + sum all along (one subtraction in place of a conversion
    // and a scaling per output).
    constexpr bool kFloatBits = EPI >= 0 && EPI != 4;
    uint32_t start = kFloatBits ? __builtin_bit_cast(uint32_t, kF32Base) : 0u;
    v16i acc0;
    if (kFloatBits) asm volatile("" : "+v"(start));  // (one tuple for all four, not sixteen constants each)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc0[r] = (int)start;
    v16i acc[TN][TM];
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int b = 0; b < TM; ++b) acc[j][b] = acc0;
    // step (i, par): weight operand = even (par 0) or odd (par 1) nibbles of piece i, activation fragment at
    // + i*64 + par*16 of the row; both sides pair the same k values
    const uint32_t fragX = l32 * kXStride + h * 32;
    auto steps = [&](int i0, int i1) {
#pragma unroll
        for (int i = i0; i < i1; ++i) {
            v4u we[TN], wo[TN];
#pragma unroll
            for (int j = 0; j < TN; ++j) expand_nibbles(wreg[j][i], we[j], wo[j]);
#pragma unroll
            for (int par = 0; par < 2; ++par) {
                v4i fx[TM];
#pragma unroll
                for (int b = 0; b < TM; ++b)
                    fx[b] = *reinterpret_cast<const v4i *>(lds + fragX + b * 32 * kXStride + i * 64 + par * 16);
#pragma unroll
                for (int b = 0; b < TM; ++b)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
                        acc[j][b] = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(v4i, par ? wo[j] : we[j]), fx[b],
                                                                          acc[j][b], 0, 0, 0);
            }
        }
    };
    steps(0, 2);                   // K >= 64 always: pieces 0 and 1 (one of them zeros when K = 64)
    if (kbytes > 64) steps(2, 4);  // rows of 192 or 256 elements
    // (the activation buffer becomes the staging area of the epilogue, which waits for every wavefront first)
    constexpr bool kWideStore = true;
    uint8_t *const wstage = lds + wave * (BM * (64 * TN + 16));
#include "duq_stream_epilogue_store.inc"
}

// ---------------------------------------------------------------------------------
// skinny kernel (9 <= M <= 16 on wide problems: 1536 or more 16-column tiles, K <= 4096)
// ---------------------------------------------------------------------------------
// Workgroup = four wavefronts that split K; it walks `tiles_per_wg` consecutive 16-column
// tiles.  Wavefront w owns 64-byte row segments [w*S, (w+1)*S), S <= 8: lane (l16, g) holds
// bytes [g*16, +16) of each.  The activation fragments of that k range do not depend on the
// column tile, so they are loaded and expanded ONCE per workgroup and stay in registers;
// per tile only the weights stream in (the next tile's loads are issued before the current
// tile's MFMAs), two MFMAs per 16-byte weight piece (even k, odd k).  Partial sums of the
// wavefronts meet in LDS (double buffered: one barrier per tile).
// Weight loads fetch whole cache lines: an instruction covers 8 rows x 128 contiguous bytes instead of the
// MFMA layout's 16 rows x 64 (half a line each); the wavefront turns the tile into the MFMA's lane layout
// through its own 8 KB of LDS (one 128-bit write and one 128-bit read per load; no barrier: the piece is
// private to the wavefront and a wavefront's LDS operations execute in order).  Slot s of a row's line holds
// its 16-byte piece s ^ ((row / 2) % 8), which makes the 16 rows x 16 bytes of a fragment read cover every bank
// once.  Measured 4-9 % faster than MFMA-layout loads from 512 column tiles on; smaller problems run the
// decode kernels (duq_decode.hip), where the extra LDS hop is not hidden.
constexpr int kSkinnyWaves = 4;
constexpr int kSkinnySegs = 8;  // 64-byte segments per wavefront = 128-bit weight loads in flight per lane

template <int EPI, bool BIAS>
__global__ __launch_bounds__(kSkinnyWaves * 64) void gemm_s4_skinny_kernel(DUQ_HEAD_DECL, GemmParams tail)
{
    GemmParams p = with_head(tail, DUQ_HEAD_USE);
    to_global(p.A);
    to_global(p.B);
    to_global(p.C);
    to_global(p.y);
    __shared__ v4i part[2][kSkinnyWaves][64];
    __shared__ __attribute__((aligned(16))) uint8_t turn[kSkinnyWaves * 8192];
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63u, wave = tid >> 6;
    const uint32_t l16 = lane & 15u, g = lane >> 4;
    const uint32_t r8 = lane >> 3, j8 = lane & 7u;
    const uint32_t kbytes = p.K >> 1;
    const uint32_t segs = (kbytes + 63) / 64;
    const uint32_t seg0 = wave * kSkinnySegs;  // kSkinnyWaves * kSkinnySegs >= segs: rows of at most 4096 elements
    const uint32_t tiles_per_wg = p.tiles_m;   // (field reused: column tiles per workgroup)
    const uint32_t ntiles = (p.N + 15) / 16;
    const uint32_t tile0 = blockIdx.x * tiles_per_wg;
    const uint32_t tile_end = min(tile0 + tiles_per_wg, ntiles);

    // 32-bit byte offsets over the whole tensors: the dispatcher only comes here while N * K / 2 < 2^32 - 256
    const __amdgpu_buffer_rsrc_t rW = make_rsrc(p.B, p.N * kbytes);  // rows past N read as zero
    const __amdgpu_buffer_rsrc_t rX = make_rsrc(p.A, p.M * kbytes);  // rows past M read as zero

    // activations of this wavefront's k range: once per workgroup
    v4u xe[kSkinnySegs], xo[kSkinnySegs];
#pragma unroll
    for (int u = 0; u < kSkinnySegs; ++u) {
        const uint32_t off = (seg0 + u) * 64 + g * 16;
        const bool ok = seg0 + u < segs && off < kbytes;
        const v4u x = buf_load16(rX, ok ? l16 * kbytes + off : kOobOffset, 0);
        expand_nibbles(x, xe[u], xo[u]);
    }

    auto load_tile = [&](uint32_t tile, v4u(&w)[kSkinnySegs]) {
        // load u = 2 * line + half: rows 8 * half + r8 of the tile, slot j8 of line `line` of this wavefront's range
#pragma unroll
        for (int u = 0; u < kSkinnySegs; ++u) {
            const uint32_t rt = (u & 1) * 8 + r8, row = tile * 16 + rt;
            const uint32_t off = seg0 * 64 + (u >> 1) * 128 + ((j8 ^ ((rt >> 1) & 7u)) << 4);
            const bool ok = tile < tile_end && row < p.N && off < kbytes;
            w[u] = buf_load16_aux<DUQ_SKINNY_WLOAD_AUX>(rW, ok ? row * kbytes + off : kOobOffset, 0);
        }
    };
    auto compute_tile = [&](uint32_t tile, const v4u(&w)[kSkinnySegs], uint32_t buf) {
        v4i acc = v4i{0, 0, 0, 0};
        uint8_t *mine = turn + wave * 8192;
#pragma unroll
        for (int u = 0; u < kSkinnySegs; ++u) *reinterpret_cast<v4u *>(mine + u * 1024 + lane * 16) = w[u];
#pragma unroll
        for (int u = 0; u < kSkinnySegs; ++u) {
            // segment u = 64 bytes: half (u % 2) of line u / 2; this lane's row l16 sits in load 2 * line + l16 / 8
            const uint32_t piece = (u & 1) * 4 + g;
            const v4u raw = *reinterpret_cast<const v4u *>(mine + ((u >> 1) * 2 + (l16 >> 3)) * 1024 + (l16 & 7u) * 128 +
                                                           ((piece ^ ((l16 >> 1) & 7u)) << 4));
            v4u we, wo;
            expand_nibbles(raw, we, wo);
            acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(v4i, we), __builtin_bit_cast(v4i, xe[u]), acc,
                                                        0, 0, 0);
            acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(v4i, wo), __builtin_bit_cast(v4i, xo[u]), acc,
                                                        0, 0, 0);
        }
        // every wavefront parks its 16 x 16 partial tile, then the first 256 threads each
        // finish one output element (sum over wavefronts, epilogue, store): no wavefront
        // is a serial bottleneck
        part[buf][wave][lane] = acc;
        __syncthreads();
        if (tid < 256) {
            const uint32_t src_lane = tid >> 2, r = tid & 3u;
            int sum = 0;
#pragma unroll
            for (int w2 = 0; w2 < kSkinnyWaves; ++w2) sum += part[buf][w2][src_lane][r];
            sum >>= 8;
            const uint32_t m = src_lane & 15u, n = tile * 16 + (src_lane >> 4) * 4 + r;
            if (m < p.M && n < p.N) {
                if (EPI < 0) {
                    p.C[(uint64_t)m * p.N + n] = sum;
                } else {
                    constexpr int MODE = EPI < 0 ? 0 : EPI;
                    const ColParams c = load_col<MODE, BIAS>(p.epi.s_col_1, p.epi.z_col_1, p.epi.s_col_2,
                                                             p.epi.z_col_2, p.epi.bias, n, p.epi.rs_col);
                    p.y[(uint64_t)m * p.N + n] = dequant_one<MODE, BIAS>(sum, load_row<MODE>(p.epi, m), c);
                }
            }
        }
    };

    // two register sets alternate so that one tile's loads are in flight during the other's MFMAs
    v4u w0[kSkinnySegs], w1[kSkinnySegs];
    load_tile(tile0, w0);
    for (uint32_t t = tile0; t < tile_end; t += 2) {
        load_tile(t + 1, w1);
        compute_tile(t, w0, 0);
        load_tile(t + 2, w0);
        if (t + 1 < tile_end) compute_tile(t + 1, w1, 1);
    }
}

// ---------------------------------------------------------------------------------
// dot kernel (M <= 4, rows longer than 16384 elements): weight streaming on v_dot8_i32_i4
// ---------------------------------------------------------------------------------
// The signed 4-bit dot product instruction consumes packed nibbles as they lie in memory,
// so nothing is expanded and no MFMA is needed: the kernel is a pure HBM stream.
// Workgroup = 4 wavefronts = 8 weight rows, K split four ways.  Lane (r8, j) walks its
// quarter of row r8 in 128-byte steps, loading bytes [step*128 + j*16, +16): one wavefront
// load is eight full cache lines.  Eight loads per lane are kept in flight (a register
// ring), and with ~40 VGPRs eight wavefronts fit on a SIMD, so a CU keeps > 100 KB of
// weights in flight.  The M activation rows sit in LDS (lanes of different rows read the
// same address: a broadcast).  Partial sums meet through three lane shuffles and one LDS hop.
constexpr int kDotRing = 8;

template <int MROWS, int EPI, bool BIAS>
__global__ __launch_bounds__(256) void gemv_s4_dot_kernel(DUQ_HEAD_DECL, GemmParams tail)
{
    GemmParams p = with_head(tail, DUQ_HEAD_USE);
    to_global(p.A);
    to_global(p.B);
    to_global(p.C);
    to_global(p.y);
    extern __shared__ __attribute__((aligned(16))) uint8_t xs[];  // [MROWS][xstride] packed activations
    __shared__ int part[4][8][MROWS];
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63u, wave = tid >> 6;
    const uint32_t r8 = lane >> 3, j = lane & 7u;
    const uint32_t kbytes = p.K >> 1;
    const uint32_t nsteps_all = (kbytes + 127) / 128;
    const uint32_t xstride = nsteps_all * 128;
    const uint32_t per = (nsteps_all + 3) / 4;
    const uint32_t step0 = wave * per;
    const uint32_t nsteps = step0 < nsteps_all ? min(per, nsteps_all - step0) : 0;
    const uint32_t n = blockIdx.x * 8 + r8;

    const __amdgpu_buffer_rsrc_t rW = make_rsrc(p.B, p.N * kbytes);  // rows past N read as zero
    const uint32_t wbase = n * kbytes + j * 16;

    auto w_off = [&](uint32_t s) -> uint32_t {  // step s of this wavefront's slice
        const uint32_t off = (step0 + s) * 128 + j * 16;
        return (s < nsteps && off < kbytes && n < p.N) ? wbase + (step0 + s) * 128 : kOobOffset;
    };

    v4u ring[kDotRing];
#pragma unroll
    for (int u = 0; u < kDotRing; ++u) ring[u] = buf_load16_aux<DUQ_DOT_WLOAD_AUX>(rW, w_off(u), 0);

    // activations -> LDS (all rows, whole K), zero beyond the row end
    for (uint32_t i = tid; i < MROWS * (xstride / 16); i += 256) {
        const uint32_t m = i / (xstride / 16), o = (i % (xstride / 16)) * 16;
        v4u v = v4u{0u, 0u, 0u, 0u};
        if (m < p.M && o < kbytes) v = *reinterpret_cast<const v4u *>(p.A + (uint64_t)m * kbytes + o);
        *reinterpret_cast<v4u *>(xs + m * xstride + o) = v;
    }
    __syncthreads();

    int acc[MROWS];
#pragma unroll
    for (int m = 0; m < MROWS; ++m) acc[m] = 0;

    for (uint32_t s = 0; s < nsteps; s += kDotRing) {
#pragma unroll
        for (int u = 0; u < kDotRing; ++u) {
            const v4u w = ring[u];
            ring[u] = buf_load16_aux<DUQ_DOT_WLOAD_AUX>(rW, w_off(s + u + kDotRing), 0);
            const uint32_t xo = (step0 + s + u) * 128 + j * 16;
            if (s + u < nsteps) {
#pragma unroll
                for (int m = 0; m < MROWS; ++m) {
                    const v4u x = *reinterpret_cast<const v4u *>(xs + m * xstride + xo);
#pragma unroll
                    for (int d = 0; d < 4; ++d) acc[m] = __builtin_amdgcn_sdot8((int)w[d], (int)x[d], acc[m], false);
                }
            }
        }
    }

    // the 8 lanes of a row, then the 4 wavefronts
#pragma unroll
    for (int m = 0; m < MROWS; ++m) {
        acc[m] += __shfl_xor(acc[m], 1, kWave);
        acc[m] += __shfl_xor(acc[m], 2, kWave);
        acc[m] += __shfl_xor(acc[m], 4, kWave);
    }
    if (j == 0) {
#pragma unroll
        for (int m = 0; m < MROWS; ++m) part[wave][r8][m] = acc[m];
    }
    __syncthreads();
    if (tid < 8 * MROWS) {
        const uint32_t rr = tid / MROWS, m = tid % MROWS;
        const uint32_t nn = blockIdx.x * 8 + rr;
        if (nn < p.N && m < p.M) {
            const int v = part[0][rr][m] + part[1][rr][m] + part[2][rr][m] + part[3][rr][m];
            if (EPI < 0) {
                p.C[(uint64_t)m * p.N + nn] = v;
            } else {
                constexpr int MODE = EPI < 0 ? 0 : EPI;
                const ColParams c = load_col<MODE, BIAS>(p.epi.s_col_1, p.epi.z_col_1, p.epi.s_col_2, p.epi.z_col_2,
                                                         p.epi.bias, nn, p.epi.rs_col);
                p.y[(uint64_t)m * p.N + nn] = dequant_one<MODE, BIAS>(v, load_row<MODE>(p.epi, m), c);
            }
        }
    }
}

// ---------------------------------------------------------------------------------
// dispatch
// ---------------------------------------------------------------------------------
// Which of the kernels by size takes a shape.  Host arithmetic only, so that the rule can be tested without a GPU:
// every kernel whose weight offsets are 32-bit (decode, dot: row * K/2 + offset, and a buffer descriptor
// over the whole tensor) is reachable only while the packed weights stay below 4 GiB - 256 (the out-of-range
// marker); larger tensors go to the stream / prefill kernels, whose descriptors and pointers are per tile
// (64-bit base, 32-bit offsets inside 256 rows).
int select_gemm_kernel(uint32_t M, uint32_t N, uint32_t K)
{
    const uint64_t wbytes = (uint64_t)N * (K / 2);
    const bool small_offsets = wbytes < 0xFFFFFF00ull && K > 0;
    // (gemm_kernel_for asks takes_wide_kernel and takes_lds_kernel first: what is said here of up to 64 rows and of narrow problems
    // holds for the shapes that those leave.)  Decode: rows kernel for up to four rows (8 KB of every weight row per
    // wavefront); above, the MFMA decode kernel (rows of up to 8192 elements), with two to four row tiles against the same
    // weight fragments for 17..64 rows.  9..16 rows on very wide layers run the skinny kernel (whole-line weight loads, 5 %
    // faster at N = 28672, K = 4096).
    if (M <= 4 && K <= 16384 && small_offsets) return kKernelDecodeRows;
    if (M <= 16 && small_offsets) {
        if (M > 8 && (N + 15) / 16 >= 1536 && K <= 4096) return kKernelSkinny;
        if (K <= 12288) return kKernelDecodeMfma;
    }
    if (M <= 64 && small_offsets) {
        // one round of 64 x 64 tiles of the prefill kernel, whose time hardly depends on rows and columns, is ahead of the
        // decode kernel where that has many row tiles or several column tiles per workgroup.  More than 48 rows: 64 x
        // 11008 x 4096 9.8 against 10.65 us, 64 x 13824 x 1024 6.6 / 8.2; 40 x 11008 x 8192 14.8 / 18.6; 32 x 13824 x 5120 11.8 /
        // 13.6, 32 x 16384 x 8192 18.3 / 20.0 (but 17 x 16384 x 8192 19.3 / 18.4).
        const bool tiles = K <= 4096 ? M > 48 && N > 8192 && K >= 1024
                         : K <= 8192 && (M > 48 ? N >= 3072 : M > 32 ? N >= 5120 : M > 24 && N > 10240);
        if (tiles && N <= 16384) return kKernelStream;
        if (K <= 4096 || (K <= 8192 && M <= 32)) return kKernelDecodeMfma;
        // (wide layers of more than 32 long rows: one round of tiles of the prefill kernel, 48 x 11008 x 11008 20.3 us
        // against 24.0 with 64 x 128 tiles; at N = 4096 the decode kernel is ahead)
        const bool wide = M > 32 && N >= 8192;
        if ((N + 15) / 16 >= 192 && !wide && (K <= 8192 || (K <= 12288 && M <= 48))) return kKernelDecodeMfma;
    }
    const uint32_t xstride = ((K / 2 + 127) / 128) * 128;
    // dot kernel: up to four rows too long for the decode kernels
    if (M <= 4 && small_offsets && 4 * xstride <= 60 * 1024) return kKernelDot;
    // narrow problems, all of which takes_lds_kernel takes: 17..256 rows in groups of 64, 32 or 16 whose column tiles are one
    // round of workgroups, and 5..16 rows of 8193..16384 elements
    const uint32_t rb_max = K <= 4096 ? 4 : (K <= 8192 ? 2 : 1);
    const uint32_t row_groups = ((M + 15) / 16 + rb_max - 1) / rb_max;
    const bool one_round = M > 16 && M <= 256 && (uint64_t)((N + 15) / 16) * row_groups <= 256 && (K > 2048 || M <= 64);
    const bool long_rows = M <= 16 && K > 8192;
    if ((long_rows || one_round) && K <= 16384 && small_offsets) return kKernelLds;
    const uint32_t narrow_tiles = ((M + 63) / 64) * ((N + 127) / 128);
    const bool narrow_round = M > 64 && narrow_tiles >= 64 && narrow_tiles <= 256;
    auto tiles = [&](uint32_t bm, uint32_t bn) { return ((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
    if (narrow_round || (M > 32 && tiles(32, 256) >= 32)) return kKernelStream;
    return kKernelTile;
}

int gemm_kernel_for(uint32_t M, uint32_t N, uint32_t K)
{
    if (takes_wide_kernel(M, N, K)) return kKernelWide;
    if (takes_lds_kernel(M, N, K)) return kKernelLds;
    return select_gemm_kernel(M, N, K);
}

// batch > 1: `batch` problems of one shape, tensors contiguous over the batch, one launch (blockIdx.z is the
// problem): the short-row, stream and prefill kernels only, the tile chosen on the whole batch.
template <int EPI, bool BIAS>
static void launch_epi(GemmParams &p, hipStream_t stream, uint32_t batch = 1)
{
    const int kernel = batch > 1 ? kKernelStream : gemm_kernel_for(p.M, p.N, p.K);
    // (EPI 5, the dual-uniform row-sum epilogue: of the kernels launched here, the stream and prefill kernels have it, and
    // only their shapes come here with it: gemm_fuses_dual_rowsum)
    if constexpr (EPI != 5) {
    if (kernel == kKernelDot) {
        const uint32_t xstride = ((p.K / 2 + 127) / 128) * 128;
        const dim3 grid((p.N + 7) / 8);
        if (p.M == 1)
            DUQ_LAUNCH_HEAD((gemv_s4_dot_kernel<1, EPI, BIAS>), grid, dim3(256), 1 * xstride, stream, p);
        else if (p.M == 2)
            DUQ_LAUNCH_HEAD((gemv_s4_dot_kernel<2, EPI, BIAS>), grid, dim3(256), 2 * xstride, stream, p);
        else
            DUQ_LAUNCH_HEAD((gemv_s4_dot_kernel<4, EPI, BIAS>), grid, dim3(256), 4 * xstride, stream, p);
        return;
    }
    if (kernel == kKernelSkinny) {
        // several column tiles per workgroup (activations are fetched and expanded once per workgroup); at least
        // ~2 workgroups per CU stay
        const uint32_t ntiles = (p.N + 15) / 16, tpw = ntiles >= 6144 ? 8 : 4;
        p.tiles_m = tpw;
        DUQ_LAUNCH_HEAD((gemm_s4_skinny_kernel<EPI, BIAS>), dim3((ntiles + tpw - 1) / tpw), dim3(kSkinnyWaves * 64), 0, stream, p);
        return;
    }
    }
    if constexpr (EPI != 5) {
        if (p.K <= 256) {
            // rows of at most 256 elements: one chunk, the launch is its output stores: the short-row kernel with 64-row
            // tiles (measured on 32 products of 2048 x 2048 x 128: 86 us against 95 us on the stream kernel's 64-row tiles),
            // 32-row ones for a few rows (one query per head)
            const uint32_t bm = p.M <= 32 ? 32 : 64;
            p.tiles_m = (p.M + bm - 1) / bm;
            p.tiles_n = (p.N + 255) / 256;
            const dim3 grid(p.tiles_m * p.tiles_n, 1, batch);
            if (bm == 32)
                DUQ_LAUNCH_HEAD((gemm_s4_shortk_kernel<1, EPI, BIAS>), grid, dim3(256), 0, stream, p);
            else
                DUQ_LAUNCH_HEAD((gemm_s4_shortk_kernel<2, EPI, BIAS>), grid, dim3(256), 0, stream, p);
            return;
        }
    }
    const StreamTile tile = select_stream_tile(p.M, p.N, p.K, batch, EPI == 5);
    if (tile.stream && (EPI < 0 || !tile.main_cols)) {
        p.tiles_m = (p.M + 63) / 64;
        p.tiles_n = (p.N + 127) / 128;
        DUQ_LAUNCH_HEAD((gemm_s4_stream_kernel<EPI, BIAS>), dim3(p.tiles_m * p.tiles_n, 1, batch), dim3(256), 0, stream, p);
    } else {
        (void)launch_prefill(p, tile, EPI >= 0, stream, batch);
    }
}

int launch_gemm_s4(const uint8_t *A, const uint8_t *B, uint32_t M, uint32_t N, uint32_t K, int32_t *out_acc,
                   const Epilogue *epi, uint16_t *y, hipStream_t stream)
{
    return launch_gemm_s4_batched(A, B, M, N, K, 1, out_acc, epi, y, stream);
}

int launch_gemm_s4_batched(const uint8_t *A, const uint8_t *B, uint32_t M, uint32_t N, uint32_t K, uint32_t batch,
                           int32_t *out_acc, const Epilogue *epi, uint16_t *y, hipStream_t stream)
{
    if (M == 0 || N == 0 || batch == 0) return 0;
    if (batch == 1) {
        const int kernel = gemm_kernel_for(M, N, K);
        if (kernel == kKernelDecodeRows || kernel == kKernelDecodeMfma || kernel == kKernelWide || kernel == kKernelLds ||
            (epi && epi->mode == 5 && takes_lds_kernel(M, N, K, true)))
            return launch_decode_s4(A, B, M, N, K, out_acc, epi, y, stream);
    }
    GemmParams p{};
    p.A = A;
    p.B = B;
    p.M = M;
    p.N = N;
    p.K = K;
    p.problems = batch;
    p.C = out_acc;
    p.y = y;
    if (epi) p.epi = *epi;
    if (out_acc) {
        launch_epi<-1, false>(p, stream, batch);
    } else {
        const bool bias = epi->bias != nullptr;
#define DUQ_GEMM(MODE)                             \
    case MODE:                                     \
        if (bias)                                  \
            launch_epi<MODE, true>(p, stream, batch);  \
        else                                       \
            launch_epi<MODE, false>(p, stream, batch); \
        break;
        switch (epi->mode) {
            DUQ_GEMM(0)
            DUQ_GEMM(1)
            DUQ_GEMM(2)
            DUQ_GEMM(3)
            DUQ_GEMM(4)
        case 5:
            if (batch != 1 || !gemm_fuses_dual_rowsum(M, N, K)) return (int)hipErrorInvalidValue;
            if (bias)
                launch_epi<5, true>(p, stream, 1);
            else
                launch_epi<5, false>(p, stream, 1);
            break;
        default:
            return (int)hipErrorInvalidValue;
        }
#undef DUQ_GEMM
    }
    return (int)hipGetLastError();
}

}  // namespace duq
