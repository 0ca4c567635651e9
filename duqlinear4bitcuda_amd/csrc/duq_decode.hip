// Decode kernels (M <= 64 activation rows): weight streaming for problems of a few MB,
// where a launch lives for two or three microseconds and what counts is that every byte is requested
// in the kernel's first instructions and nothing else sits on the critical path.
//
//   C[m,n] = sum_k s4(A[m,k]) * s4(B[n,k])        (src/kernels/gemm.cu:8-43 of the reference, at M <= 16)
//
// The first two
//  * issue every weight load of the workgroup before anything else (no ring: the whole share of a
//    workgroup, 16-32 KB, is in flight at once),
//  * fetch the epilogue parameters of the outputs a lane will store right behind them, so that no
//    dependent memory round trip follows the arithmetic,
//  * take the activations pre-quantized (packed nibbles, the reference's operator boundary); the rows kernel
//    also takes them as binary16 (FUSEQ): the workgroup then computes the per-token scales and codes itself
//    while its weights are in flight (SymQuantizer.forward, qlinear4bit/nn/quantizer.py:10-16, and
//    src/kernels/quant.cu:11-45, through the same RowQuant code as the stand-alone quantizer), which makes
//    quantize + GEMM + dequant one launch.  (Up to four rows only: every workgroup reads all the rows, and from
//    eight rows on that is more bytes into a CU than its share of the weights.)
//
//  rows kernel (M <= 4): v_dot8_i32_i4 on the packed nibbles.  A wavefront owns four weight rows and the
//    whole K range: lane l holds bytes [i*1024 + l*16, +16) of each row, so a load instruction covers 1 KB
//    of one row and an activation register serves four rows.  The 4*M partial sums of a lane meet the other
//    lanes' through the wavefront's own piece of LDS (no barrier) and a few DPP steps.
//  MFMA kernel (5 <= M <= 64, several column tiles per CU, K <= 8192): v_mfma_i32_16x16x64_i8, eight wavefronts split K
//    for one 16-column tile, one to four tiles of 16 rows against the same weight fragments, the partial tiles meet in LDS, 256 threads finish
//    one output each per row tile; one round of at most 256 workgroups with several column tiles each.
//  wide kernel (5 <= M <= 64, many column tiles per CU, K <= 8192): the MFMA kernel's plan with the weights through LDS.
//  LDS kernel (one or two column tiles and up to four row tiles per workgroup, any K): the same MFMAs, both operands through LDS in whole
//    cache lines, K in a loop.
#include "duq_decode_common.h"

// Wavefronts per workgroup of the rows kernel when it quantizes its rows itself (binary16 in).  The quantize phase is
// vector arithmetic (about 27 instructions per eight elements), the same for every workgroup, and sits between the
// arrival of the activations and the dot products: a wavefront alone on its SIMD issues it at half the rate that
// two reach together.  Measured (us, N = K = 4096 unless said): two rows 3.25 with four wavefronts, 3.21 with eight;
// three / four rows 4.11 / 4.17 with four, 3.67 / 3.68 with eight (and with sixteen); four rows of 8192 / 11008
// elements 7.5 / 8.9 with four, 6.5 / 7.1 with sixteen; eight rows 5.0 with eight, 5.1 with sixteen.
#ifndef DUQ_DEC_FUSEQ_WAVES
#define DUQ_DEC_FUSEQ_WAVES 8     // eight rows; and several tiles per workgroup
#endif
#ifndef DUQ_DEC_FUSEQ_WAVES_M4
#define DUQ_DEC_FUSEQ_WAVES_M4 8  // three or four rows of up to 4096 elements
#endif
#ifndef DUQ_DEC_FUSEQ_WAVES_M4L
#define DUQ_DEC_FUSEQ_WAVES_M4L 16  // of more
#endif
#ifndef DUQ_DEC_FUSEQ_WAVES_M2
#define DUQ_DEC_FUSEQ_WAVES_M2 4
#endif
#ifndef DUQ_DEC_R
#define DUQ_DEC_R 4
#endif
// Cache policy of the rows kernel's weight loads (and of the read probe that mirrors them): 2 = non-temporal.  A
// load instruction of that kernel covers whole cache lines that nobody reads again (measured, one row: N = K = 4096
// 3.00 against 3.08 us, N = 28672 K = 8192 19.6 against 21.2).  The MFMA kernel reads a line in two instructions (64
// bytes of a row each) and loses with it (16 rows, N = K = 4096: 4.13 against 3.90 us): it keeps the default.
#ifndef DUQ_DEC_WLOAD_AUX
#define DUQ_DEC_WLOAD_AUX 2
#endif
#ifndef DUQ_DEC_WAVES
#define DUQ_DEC_WAVES 8
#endif
// 8-element units whose quantization chains are interleaved in the kernels that quantize their rows themselves
#ifndef DUQ_DEC_QUANT_GROUP
#define DUQ_DEC_QUANT_GROUP 8
#endif
namespace duq {

namespace {

// ---------------------------------------------------------------------------------
// rows kernel: M <= MR <= 4 (8 with binary16 activations quantized inside), K <= XS * 2048
// ---------------------------------------------------------------------------------
// WAVES wavefronts of R = 16 / WAVES weight rows each: 16 weight rows ("a tile") per workgroup either way.  Eight
// wavefronts help when the workgroup quantizes four activation rows itself and a CU holds several workgroups
// (launcher).  MULTI: a workgroup owns p.tiles_per_wg consecutive tiles and keeps two tiles' weights in flight
// (two register sets that alternate), so that a launch is one round of at most 256 workgroups: the activations
// are fetched, and with FUSEQ quantized, once per CU and not once per tile.
template <int MR, int XS, bool FUSEQ, int EPI, int WAVES = 4, bool MULTI = false>
__global__ __launch_bounds__(WAVES * 64) void gemv_s4_rows_kernel(DUQ_HEAD_DECL, DecodeParams tail)
{
    const DecodeParams p = with_head(tail, DUQ_HEAD_USE);
    constexpr int R = 4 * DUQ_DEC_R / WAVES;  // weight rows per wavefront
    constexpr int V = MR * R;        // partial sums per lane: 4, 8 or 16
    constexpr int LPV = 64 / V;      // lanes that finish one sum: 16, 8 or 4
    constexpr int MODE = EPI < 0 ? 0 : EPI;
    constexpr uint32_t XSTRIDE = XS * 1024;
    static_assert(MR == 1 || MR == 2 || MR == 4 || (MR == 8 && WAVES >= 8), "rows");
    static_assert(WAVES == 4 || WAVES == 8 || WAVES == 16, "wavefronts per workgroup");
    static_assert(V >= 4 && V <= 16 && (XS * MR * 4) % WAVES == 0, "partial sums per lane, quantize units per lane");
    __shared__ __attribute__((aligned(16))) int red[WAVES][V * 64];
    __shared__ __attribute__((aligned(16))) uint8_t xs[FUSEQ ? MR * XSTRIDE : 16];
    __shared__ uint32_t rmax[WAVES];
    __shared__ float rlo[WAVES], rhi[WAVES];
    __shared__ int rsum[WAVES];
    __shared__ uint16_t srow[MR], zrow[MR];
    __shared__ int rsrow[MR];
    // binary16 rows in: the epilogue decides the quantizer (SymQuantizer for the symmetric epilogues, AsymQuantizer
    // for the asymmetric ones; the row-sum epilogue takes the signed-shifted codes, code - 8 and zero - 8, and the
    // per-token sum of the shifted codes)
    constexpr bool ASYMQ = FUSEQ && (MODE == 1 || MODE == 3 || MODE == 4 || MODE == 5);
    constexpr bool SHIFTQ = FUSEQ && (MODE == 4 || MODE == 5);
    using ColRec = typename EpiRec<MODE>::Col;
    using RowRec = typename EpiRec<MODE>::Row;

    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t kbytes = p.K >> 1;
    const uint32_t tile0 = MULTI ? blockIdx.x * p.tiles_per_wg : blockIdx.x;
    const uint32_t tile_end = MULTI ? min(tile0 + p.tiles_per_wg, (p.N + 4 * DUQ_DEC_R - 1) / (4 * DUQ_DEC_R)) : tile0 + 1;

    // ---- loads, in the order their data is needed (loads return in order: waiting for one waits for every
    // earlier one): the activations first, then every weight byte of this wavefront's first tile, then the
    // parameters of the output this lane will finish
    // activations: lane l needs bytes [i*1024 + l*16, +16) of every row
    v4u xr[MR][XS];
    // Four rows of 12289 to 16384 elements come out of LDS in two halves: all of them beside the weights are more than
    // the 128 registers that sixteen wavefronts leave each, and the asymmetric quantizers spilled.  Measured (us, four
    // rows, 4096 columns x 16384, whole against halves): Linear4bitASQ 11.2 -> 9.9, Linear4bitASQRowSum 11.4 -> 10.4,
    // LinearQuant4bitDUASQRowSum 12.8 -> 11.1, Linear4bitSQ 9.5 -> 9.6.
    constexpr bool kHalves = FUSEQ && MR == 4 && XS >= 8 && !MULTI;
    constexpr int WPR = WAVES / MR;           // wavefronts that share a row in the quantize phase
    constexpr int UPL = FUSEQ ? XS * MR * 4 / WAVES : 1;  // 8-element units per lane in the quantize phase
    const uint32_t qrow = wave / WPR, qpart = wave % WPR;
    v4u raw[UPL];
    const uint32_t nunits = p.K >> 3;
    if (!FUSEQ) {
        const __amdgpu_buffer_rsrc_t rX = make_rsrc(p.A, p.M * kbytes);  // rows past M read as zero
#pragma unroll
        for (int m = 0; m < MR; ++m)
#pragma unroll
            for (int i = 0; i < XS; ++i) {
                const uint32_t off = i * 1024 + lane * 16;
                xr[m][i] = buf_load16(rX, off < kbytes ? m * kbytes + off : kOobOffset, 0);
            }
    } else {
        // the workgroup quantizes the MR rows into LDS: WPR = WAVES / MR wavefronts share a row, wavefront `part` of
        // a row owns its 8-element units part*64 + lane, + 64*WPR, ...
        const __amdgpu_buffer_rsrc_t rX = make_rsrc(p.X, p.M * p.K * 2);  // rows past M read as zero
#pragma unroll
        for (int j = 0; j < UPL; ++j) {
            const uint32_t c = qpart * 64 + lane + j * (64 * WPR);
            raw[j] = buf_load16(rX, c < nunits ? (qrow * p.K + c * 8) * 2 : kOobOffset, 0);
        }
    }
    // Eight wavefronts that quantize: all of them request their activations before any requests weights (the CU
    // serves requests in order, and a wavefront whose activations queue behind another's weights holds up the
    // whole workgroup at the staging barrier below; measured at 8 rows, K = 4096: N = 4096 5.6 against 6.2 us,
    // N = 11008 8.2 against 8.5; with four wavefronts it changes nothing)
    if (FUSEQ && WAVES >= 8) __builtin_amdgcn_s_barrier();
    const __amdgpu_buffer_rsrc_t rW = make_rsrc(p.B, p.N * kbytes);
    // the weights of tile t for this wavefront (tiles past the workgroup's last read as zero, unused)
    auto load_w = [&](uint32_t tile, v4u(&w)[R][XS]) {
        const uint32_t n0 = (tile * WAVES + wave) * R;
        const uint32_t nrows = (!MULTI || tile < tile_end) ? p.N : 0u;
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int i = 0; i < XS; ++i) {
                const uint32_t off = i * 1024 + lane * 16;
                // K % 64 == 0: a 16-byte piece is all in or all out
                const bool ok = off < kbytes && n0 + r < nrows;
                w[r][i] = __builtin_bit_cast(
                    v4u, __builtin_amdgcn_raw_buffer_load_b128(rW, (int)(ok ? (n0 + r) * kbytes + off : kOobOffset), 0, DUQ_DEC_WLOAD_AUX));
            }
    };
    v4u w0[R][XS], w1[MULTI ? R : 1][MULTI ? XS : 1];
    load_w(tile0, w0);
    const uint32_t myv = lane / LPV, sub = lane % LPV;
    const uint32_t my_m = myv / R, my_r = wave * R + myv % R;  // my_r: weight row inside a tile
    const bool bias = p.epi.bias != nullptr;
    auto load_cp = [&](uint32_t tile) {
        ColRec c{};
        if (EPI >= 0) c = load_col_rt<MODE>(p.epi, min(tile * (4 * DUQ_DEC_R) + my_r, p.N - 1), bias, p.B, kbytes);
        return c;
    };
    ColRec cp = load_cp(tile0);
    RowRec rp{};
    if (EPI >= 0 && !FUSEQ) rp = load_row_rt<MODE>(p.epi, min(my_m, p.M - 1), p.A, kbytes);

    // what the quantize phase needs of the kernel arguments, fetched here under the vector loads above: a scalar
    // load issued where the value is first used (the compiler sinks it into the branch that uses it) is waited for on
    // its own, and a fetch of kernel arguments costs about half a microsecond (measured: 4 rows, N = K = 4096, 5.5
    // against 4.9 us)
    const float q_clip = p.clip;
    const int q_qmax = p.qmax;
    uint8_t *const q_out = p.q_out;
    uint16_t *const s_out = p.s_out, *const z_out = p.z_out;
    int32_t *const rs_out = p.rs_out;
    if (FUSEQ)
        asm volatile("" ::"s"(q_clip), "s"(q_qmax), "s"(q_out), "s"(s_out), "s"(z_out), "s"(rs_out));
    // (the output pointers arrive in registers)
    const auto c_out = as_global(p.C);
    const auto y_out = as_global(p.y);

    if (FUSEQ) {
        // statistics of this wavefront's share of its row.  Units past the row end read as zero: that changes no
        // maximum of |x|, but it would change a minimum or a maximum, so the asymmetric form skips them.
        PkMinMax st;
#pragma unroll
        for (int j = 0; j < UPL; ++j)
            if (!ASYMQ || qpart * 64 + lane + j * (64 * WPR) < nunits) st.add8(raw[j]);
        uint32_t m16;
        float lo = 0.f, hi = 0.f;
        if (!ASYMQ) {
            m16 = wave_max_u32(st.absmax_bits());
        } else {
            st.wave_reduce();
            m16 = st.absmax_bits();
            lo = st.min_f32();
            hi = st.max_f32();
        }
        if (WPR > 1) {  // the row's statistics cross its wavefronts through LDS
            if (lane == 0) {
                rmax[wave] = m16;
                if (ASYMQ) {
                    rlo[wave] = lo;
                    rhi[wave] = hi;
                }
            }
            __syncthreads();
            m16 = rmax[qrow * WPR];
            if (ASYMQ) {
                lo = rlo[qrow * WPR];
                hi = rhi[qrow * WPR];
            }
#pragma unroll
            for (int i = 1; i < WPR; ++i) {
                m16 = max(m16, rmax[qrow * WPR + i]);
                if (ASYMQ) {
                    lo = fminf(lo, rlo[qrow * WPR + i]);
                    hi = fmaxf(hi, rhi[qrow * WPR + i]);
                }
            }
        }
        if (ASYMQ && m16 > 0x7C00u) lo = hi = __builtin_nanf("");  // torch's min / max return NaN for a row that holds one
        int code_sum = 0;
        // rows past M (the last rows of the MR the kernel is built for) are neither quantized nor used
        if (qrow < p.M) {
            RowQuant<ASYMQ> rq;
            rq.init(m16, lo, hi, q_clip, q_qmax);
            const bool copy_out = blockIdx.x == 0;
            uint32_t words[UPL];
            quant_in_groups<(XS >= 8 ? 4 : DUQ_DEC_QUANT_GROUP)>(rq, raw, words);  // (long rows: registers)
#pragma unroll
            for (int j = 0; j < UPL; ++j) {
                const uint32_t c = qpart * 64 + lane + j * (64 * WPR);
                if (c < nunits) {
                    uint32_t word = words[j];
                    if (SHIFTQ) {
                        // eight unsigned codes: sum them, then u - 8 as a signed nibble is u with bit 3 flipped
                        const uint32_t pairs = (word & 0x0F0F0F0Fu) + ((word >> 4) & 0x0F0F0F0Fu);
                        code_sum = (int)__builtin_amdgcn_udot4(pairs, 0x01010101u, (uint32_t)code_sum, false);
                        word ^= 0x88888888u;
                    }
                    *reinterpret_cast<uint32_t *>(xs + qrow * XSTRIDE + c * 4) = word;
                    if (copy_out && q_out) reinterpret_cast<uint32_t *>(q_out + (uint64_t)qrow * kbytes)[c] = word;
                }
            }
            if (SHIFTQ) {
                code_sum = wave_sum_i32(code_sum);
                if (lane == 0) rsum[wave] = code_sum;
            }
            if (qpart == 0 && lane == 0) {
                const f16 z = SHIFTQ ? rq.z - (f16)8.0f : rq.z;
                srow[qrow] = f16_to_bits(rq.s);
                if (ASYMQ) zrow[qrow] = f16_to_bits(z);
                if (copy_out && s_out) s_out[qrow] = f16_to_bits(rq.s);
                if (ASYMQ && copy_out && z_out) z_out[qrow] = f16_to_bits(z);
            }
        }
        __syncthreads();
        if (SHIFTQ) {
            // per-token sum of the shifted codes: the parts of a row's wavefronts, minus 8 per element
            if (tid < (uint32_t)MR && tid < p.M) {
                int t = -8 * (int)p.K;
#pragma unroll
                for (int i = 0; i < WPR; ++i) t += rsum[tid * WPR + i];
                rsrow[tid] = t;
                if (blockIdx.x == 0 && rs_out) rs_out[tid] = t;
            }
            __syncthreads();
        }
        // (bytes past the row end are never written: the weights read as zero there)
#pragma unroll
        for (int m = 0; m < MR; ++m)
#pragma unroll
            for (int i = 0; i < (kHalves ? XS / 2 : XS); ++i) xr[m][i] = load16(xs + m * XSTRIDE + i * 1024 + lane * 16);
        const uint32_t rm = min(my_m, (uint32_t)MR - 1);
        if constexpr (MODE == 5) {
            // the row record from the codes this workgroup just wrote
            const v2u head = *reinterpret_cast<const v2u *>(xs + rm * XSTRIDE);
            rp.xlo = head[0];
            rp.xhi = head[1] & 0xFFu;
            rp.zx = (uint32_t)rint_i32((float)bits_to_f16(zrow[rm]));
            rp.sx = (float)bits_to_f16(srow[rm]);
            rp.rxl = dual_head_sum(rp.xlo, rp.xhi);
            rp.rxr = (uint32_t)rsrow[rm] - rp.rxl;
        } else {
            rp.s = bits_to_f16(srow[rm]);
            if (ASYMQ) rp.z = bits_to_f16(zrow[rm]);
            if (SHIFTQ) rp.rs = rsrow[rm];
        }
    }

    auto do_tile = [&](uint32_t tile, const v4u(&w)[R][XS], const ColRec &c) {
        // ---- dot products on the packed nibbles
        int acc[MR][R];
#pragma unroll
        for (int m = 0; m < MR; ++m)
#pragma unroll
            for (int r = 0; r < R; ++r) acc[m][r] = 0;
#pragma unroll
        for (int i = 0; i < XS; ++i) {
            if (kHalves && i == XS / 2) {
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int m = 0; m < MR; ++m)
#pragma unroll
                    for (int h = XS / 2; h < XS; ++h) xr[m][h] = load16(xs + m * XSTRIDE + h * 1024 + lane * 16);
            }
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int m = 0; m < MR; ++m)
#pragma unroll
                    for (int d = 0; d < 4; ++d)
                        acc[m][r] = __builtin_amdgcn_sdot8((int)w[r][i][d], (int)xr[m][i][d], acc[m][r], false);
        }

        // ---- the V sums of 64 lanes each: through this wavefront's piece of LDS (a wavefront's LDS operations
        // execute in order: no barrier), V entries per lane back, then log2(LPV) DPP steps
        int *mine = red[wave];
#pragma unroll
        for (int v = 0; v < V; ++v) mine[v * 64 + lane] = acc[v / R][v % R];
        __builtin_amdgcn_wave_barrier();
        int sum = 0;
#pragma unroll
        for (int e = 0; e < V / 4; ++e) {
            const v4i t = *reinterpret_cast<const v4i *>(&mine[lane * V + e * 4]);  // = [myv * 64 + sub * V + e * 4]
            sum += (t[0] + t[1]) + (t[2] + t[3]);
        }
        __builtin_amdgcn_wave_barrier();
        sum = group_sum<LPV>(sum);
        const uint32_t my_n = tile * (4 * DUQ_DEC_R) + my_r;
        if (sub == 0 && my_m < p.M && my_n < p.N) {
            if (EPI < 0)
                c_out[(uint64_t)my_m * p.N + my_n] = sum;
            else
                y_out[(uint64_t)my_m * p.N + my_n] = dequant_rt<MODE>(sum, rp, c, bias);
        }
    };

    if constexpr (!MULTI) {
        do_tile(tile0, w0, cp);
    } else {
        for (uint32_t t = tile0; t < tile_end; t += 2) {
            load_w(t + 1, w1);
            const ColRec cp1 = load_cp(t + 1 < tile_end ? t + 1 : t);
            do_tile(t, w0, cp);
            load_w(t + 2, w0);
            cp = load_cp(t + 2 < tile_end ? t + 2 : t);
            if (t + 1 < tile_end) do_tile(t + 1, w1, cp1);
        }
    }
}

// ---------------------------------------------------------------------------------
// MFMA kernel: M <= 16 * MT, K <= WAVES * SEGS * 128 <= 12288
// ---------------------------------------------------------------------------------
// WAVES wavefronts split K: wavefront v owns the 64-byte row segments [v*SEGS, (v+1)*SEGS); lane (l16, g)
// holds bytes [g*16, +16) of each, of weight row l16 of the tile (MFMA "A" side) and of activation rows
// 16*t + l16 of the MT row tiles ("B" side), so it ends up with four consecutive output columns of those rows.
// A weight fragment is expanded once and meets all MT activation fragments: more rows cost matrix instructions
// and registers (MT * SEGS * 4 for the packed activations), not weight traffic.  Nibble -> byte as in the
// GEMM kernels: (w & 0xF0F0F0F0) is the four odd-k nibbles times 16, ((w << 4) & 0xF0F0F0F0) the even ones;
// every product is 256 * a * b and one arithmetic shift recovers the sum.
template <int WAVES, int SEGS, int EPI, int MT = 1>
__global__ __launch_bounds__(WAVES * 64) void gemm_s4_decode_kernel(DUQ_HEAD_DECL, DecodeParams tail)
{
    const DecodeParams p = with_head(tail, DUQ_HEAD_USE);
    constexpr int MODE = EPI < 0 ? 0 : EPI;
    static_assert(WAVES == 4 || WAVES == 8, "wavefronts per workgroup");
    static_assert(MT >= 1 && MT <= 4, "16-row activation tiles");
    constexpr int NG = WAVES / 4;             // groups of 256 finishing threads
    constexpr int FT = (MT + NG - 1) / NG;    // row tiles a finishing thread completes
    __shared__ v4i part[2][MT][WAVES][64];

    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t l16 = lane & 15u, g = lane >> 4;
    const uint32_t kbytes = p.K >> 1;
    const uint32_t seg0 = wave * SEGS;
    const uint32_t ntiles = (p.N + 15) / 16;
    const uint32_t tile0 = blockIdx.x * p.tiles_per_wg;
    const uint32_t tile_end = min(tile0 + p.tiles_per_wg, ntiles);

    const __amdgpu_buffer_rsrc_t rW = make_rsrc(p.B, p.N * kbytes);  // rows past N read as zero
    uint32_t koff[SEGS];  // byte offset inside a row, or out of range for pieces past K
#pragma unroll
    for (int u = 0; u < SEGS; ++u) {
        const uint32_t off = (seg0 + u) * 64 + g * 16;
        koff[u] = off < kbytes ? off : kOobOffset;
    }
    auto load_tile = [&](uint32_t tile, v4u(&w)[SEGS]) {
        const uint32_t row = tile * 16 + l16;
        const bool rok = tile < tile_end && row < p.N;
#pragma unroll
        for (int u = 0; u < SEGS; ++u)
            w[u] = buf_load16(rW, (rok && koff[u] != kOobOffset) ? row * kbytes + koff[u] : kOobOffset, 0);
    };

    // ---- loads in the order their data is needed (loads return in order): the activation fragments of this
    // wavefront's k range (packed; expanded when used), the first tile's weights, the parameters of the outputs
    // this thread will finish
    v4u xp[MT][SEGS];
    const __amdgpu_buffer_rsrc_t rX = make_rsrc(p.A, p.M * kbytes);  // rows past M read as zero
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int u = 0; u < SEGS; ++u)
            xp[t][u] = buf_load16(rX, koff[u] != kOobOffset ? (t * 16 + l16) * kbytes + koff[u] : kOobOffset, 0);
    v4u w0[SEGS], w1[SEGS];
    load_tile(tile0, w0);

    // threads finish one output per row tile they own: element er of MFMA lane src_lane; the 256-thread group
    // fg owns row tiles fg, fg + NG, ...
    const uint32_t src_lane = (tid >> 2) & 63u, er = tid & 3u, fg = tid >> 8;
    const uint32_t my_m = src_lane & 15u, my_c = (src_lane >> 4) * 4 + er;
    const bool bias = p.epi.bias != nullptr;
    const bool finisher = fg < (uint32_t)MT;
    using ColRec = typename EpiRec<MODE>::Col;
    using RowRec = typename EpiRec<MODE>::Row;
    ColRec cp{};
    RowRec rp[FT];
    auto load_cp = [&](uint32_t tile) {
        ColRec c{};
        if (EPI >= 0 && finisher) c = load_col_rt<MODE>(p.epi, min(tile * 16 + my_c, p.N - 1), bias, p.B, kbytes);
        return c;
    };
    cp = load_cp(tile0);
    // (the output pointers arrive in registers)
    const auto c_out = as_global(p.C);
    const auto y_out = as_global(p.y);
#pragma unroll
    for (int f = 0; f < FT; ++f) {
        rp[f] = RowRec{};
        if (EPI >= 0 && finisher)
            rp[f] = load_row_rt<MODE>(p.epi, min((fg + f * NG) * 16 + my_m, p.M - 1), p.A, kbytes);
    }

    auto compute_tile = [&](uint32_t tile, const v4u(&w)[SEGS], uint32_t buf) {
        const ColRec cpn = load_cp(tile + 1 < tile_end ? tile + 1 : tile);  // next tile's, under this tile's work
        v4i acc[MT];
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[t] = v4i{0, 0, 0, 0};
#pragma unroll
        for (int u = 0; u < SEGS; ++u) {
            v4u we, wo;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                we[q] = (w[u][q] << 4) & kNibbleMaskD;
                wo[q] = w[u][q] & kNibbleMaskD;
            }
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                v4u xe, xo, xv = xp[t][u];
                // many fragments: keep their expansion here (hoisted out of the tile loop it would double the
                // registers they take)
                if (MT * SEGS > 16) asm volatile("" : "+v"(xv));
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    xe[q] = (xv[q] << 4) & kNibbleMaskD;
                    xo[q] = xv[q] & kNibbleMaskD;
                }
                acc[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(v4i, we), __builtin_bit_cast(v4i, xe), acc[t], 0, 0, 0);
                acc[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(v4i, wo), __builtin_bit_cast(v4i, xo), acc[t], 0, 0, 0);
            }
        }
#pragma unroll
        for (int t = 0; t < MT; ++t) part[buf][t][wave][lane] = acc[t];
        __syncthreads();
#pragma unroll
        for (int f = 0; f < FT; ++f) {
            const uint32_t t = fg + f * NG;
            if (t < (uint32_t)MT) {
                int sum = 0;
#pragma unroll
                for (int w2 = 0; w2 < WAVES; ++w2) sum += part[buf][t][w2][src_lane][er];
                sum >>= 8;
                const uint32_t m = t * 16 + my_m, n = tile * 16 + my_c;
                if (m < p.M && n < p.N) {
                    if (EPI < 0)
                        c_out[(uint64_t)m * p.N + n] = sum;
                    else
                        y_out[(uint64_t)m * p.N + n] = dequant_rt<MODE>(sum, rp[f], cp, bias);
                }
            }
        }
        cp = cpn;
    };

    // two register sets alternate so that one tile's loads are in flight during the other's MFMAs; the
    // partial-sum buffers alternate too: one barrier per tile
    for (uint32_t t = tile0; t < tile_end; t += 2) {
        load_tile(t + 1, w1);
        compute_tile(t, w0, 0);
        load_tile(t + 2, w0);
        if (t + 1 < tile_end) compute_tile(t + 1, w1, 1);
    }
}

// ---------------------------------------------------------------------------------
// LDS kernel: up to 64 rows of any length, more on narrow problems (what takes_lds_kernel gives it)
// ---------------------------------------------------------------------------------
// A fragment of the MFMA takes sixteen bytes of each of sixteen rows from sixteen neighbouring lanes, and a load in that
// layout touches a cache line per lane: the kernel above requests its operands at about 29 bytes per ns and CU, a quarter of
// what a CU can take in (131 KB a workgroup at 16 x 4096 x 8192), and a launch of few rows lasts as long as that.  Here both
// operands come through LDS without registers, in instructions of whole 128- or 512-byte pieces of a row; eight wavefronts
// split K, each reads its fragments out of LDS, and the walk over K is a loop, so that rows may be of any length.  Sixteen
// columns per workgroup: a wavefront's stages are its own, 128 bytes of every
// kilobyte of a row, and nothing waits for another wavefront until the sums meet.  32 columns: the
// activations are a third less of what enters a CU, and the wavefronts share stages of 512 bytes a row, which 64 rows need
// (8192 x 28672: 29 us against 42 with 64-byte pieces of their own, which are half lines).  Measured against what ran before
// (N x K, weights out of the caches, us): 16 rows 4096 x 4096 4.25 -> 4.05, x 8192 7.4 -> 5.6, x 11008 9.2 -> 6.9, 2606 x 26944 32.3 ->
// 14.7, 8192 x 28672 32.2 -> 22.8; 64 rows 7.2 -> 6.0, 13.9 -> 8.3, 17.9 -> 10.1, 40.8 -> 20.4, 40.6 -> 30.7.  Groups of rows in workgroups
// of their own, where a column range leaves compute units without work: 64 x 1024 x 8192 8.1 -> 4.7, 128 x 1024 x 8192 8.2 -> 5.75,
// 256 x 2048 x 4096 9.3 -> 7.3, 96 x 4096 x 11008 15.9 -> 11.4 (64 x 64 tiles of the prefill kernel: half the workgroups and twice
// the operands each).
template <int MT, int NT, int EPI>
__global__ __launch_bounds__(512) void gemm_s4_lds_kernel(DUQ_HEAD_DECL, DecodeParams tail)
{
    const DecodeParams p = with_head(tail, DUQ_HEAD_USE);
    using Tile = LdsTile<MT, NT>;
    constexpr int MODE = EPI < 0 ? 0 : EPI;
    constexpr int WAVES = 8, G = Tile::G, U = Tile::U, L = Tile::L, DEPTH = Tile::DEPTH, NG = WAVES / 4;
    constexpr uint32_t RB = Tile::RB, kStage = Tile::kStage;
    constexpr int FT = (MT * NT + NG - 1) / NG;  // output tiles a group of 256 threads finishes
    static_assert(DEPTH >= 2 && DEPTH * L <= 63, "vmcnt");
    __shared__ __attribute__((aligned(256))) uint8_t lds[Tile::kLds];
    using ColRec = typename EpiRec<MODE>::Col;
    using RowRec = typename EpiRec<MODE>::Row;

    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t l16 = lane & 15u, g = lane >> 4;
    const uint32_t kbytes = p.K >> 1;
    // groups of 16 * MT rows share the weights of a column tile: consecutive in `at`, an eighth of which runs on one XCD
    const uint32_t groups = p.tiles_per_wg & 0x1FFu, per_xcd = ((p.N + 16 * NT - 1) / (16 * NT) * groups + 7) / 8;
    const uint32_t at = blockIdx.x % 8 * per_xcd + blockIdx.x / 8, tile = at * (p.tiles_per_wg >> 9) >> 16;  // (tile = at / groups)
    const uint32_t col0 = tile * (16 * NT), m0 = (at - tile * groups) * (16 * MT);
    if (col0 >= p.N) return;
    const auto desc = [](const uint8_t *base, uint32_t bytes) {
        const uint64_t a = reinterpret_cast<uint64_t>(base);
        return v4u{(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a), (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)(a >> 32) & 0xFFFFu)),
                   (uint32_t)__builtin_amdgcn_readfirstlane((int)bytes), 0x00020000u};
    };
    const v4u dX = desc(p.A + (uint64_t)m0 * kbytes, min(p.M - m0, 16u * MT) * kbytes);  // rows past M and N read as zero
    const v4u dW = desc(p.B + (uint64_t)col0 * kbytes, min(p.N - col0, 16u * NT) * kbytes);

    // ---- global -> LDS: instruction j of a group's wavefront v takes kilobyte j * G + v of the stage, activations first; a
    // row's 16-byte pieces lie at piece ^ (row / Q), so that the sixteen rows of a fragment read sixteen places
    constexpr uint32_t PR = RB / 16, RPI = 64 / PR, Q = RB < 256 ? 256 / RB : 1;  // pieces a row, rows an instruction
    const uint32_t group = G == 1 ? wave : 0, v = G == 1 ? 0 : wave;
    const uint32_t r0 = v * RPI + lane / PR, row0 = r0 * kbytes;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds + group * (DEPTH * kStage) + v * 1024;
    auto load = [&](uint32_t step, uint32_t slot) {
        const uint32_t k = (step * (WAVES / G) + group) * RB;
        uint32_t at[2];  // (of even and odd instructions: rows 16 apart swizzle alike)
        bool in[2];
#pragma unroll
        for (int o = 0; o < 2; ++o) {
            at[o] = k + ((lane % PR) ^ ((o * (G * RPI) + r0) % 16 / Q)) * 16;
            in[o] = at[o] < kbytes;  // K % 64 == 0: a 16-byte piece is all in or all out
        }
#pragma unroll
        for (int j = 0; j < L; ++j) {
            const uint32_t rows = (j < MT * U ? j : j - MT * U) * (G * RPI);
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(lds0 + slot + j * (G * 1024)),
                         "v"(in[j % 2] ? row0 + rows * kbytes + at[j % 2] : kOobOffset), "s"(j < MT * U ? dX : dW)
                         : "memory", "m0");
        }
    };
    static_assert(G * RPI == 8 || G * RPI == 16, "the two swizzles above");
    // ---- LDS -> registers: 64 bytes of a row make a fragment (two MFMAs)
    v4u x[MT][U], w[NT][U];
    const uint8_t *const own = lds + group * (DEPTH * kStage) + l16 * RB;
    auto read = [&](uint32_t slot) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint8_t *const at = own + slot + (((v * U + u) * 4 + g) ^ (l16 / Q)) * 16;
#pragma unroll
            for (int n = 0; n < NT; ++n) w[n][u] = *reinterpret_cast<const v4u *>(at + (MT + n) * (16 * RB));
#pragma unroll
            for (int m = 0; m < MT; ++m) x[m][u] = *reinterpret_cast<const v4u *>(at + m * (16 * RB));
        }
    };
    v4i acc[NT][MT];
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[n][m] = v4i{0, 0, 0, 0};
    auto compute = [&]() {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            v4u we[NT], wo[NT];
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    we[n][q] = (w[n][u][q] << 4) & kNibbleMaskD;
                    wo[n][q] = w[n][u][q] & kNibbleMaskD;
                }
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                v4u xe, xo;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    xe[q] = (x[m][u][q] << 4) & kNibbleMaskD;
                    xo[q] = x[m][u][q] & kNibbleMaskD;
                }
#pragma unroll
                for (int n = 0; n < NT; ++n) {
                    acc[n][m] = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(v4i, we[n]), __builtin_bit_cast(v4i, xe), acc[n][m], 0, 0, 0);
                    acc[n][m] = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(v4i, wo[n]), __builtin_bit_cast(v4i, xo), acc[n][m], 0, 0, 0);
                }
            }
        }
    };
    const uint32_t steps = (kbytes + WAVES / G * RB - 1) / (WAVES / G * RB);
#pragma unroll
    for (int s = 0; s < DEPTH; ++s) load(s, s * kStage);

    // the parameters of the outputs this thread finishes, behind the first steps' operands
    const uint32_t src_lane = (tid >> 2) & 63u, er = tid & 3u, fg = tid >> 8;
    const uint32_t my_m = src_lane & 15u, my_c = (src_lane >> 4) * 4 + er;
    const bool bias = p.epi.bias != nullptr;
    const auto c_out = as_global(p.C);
    const auto y_out = as_global(p.y);
    ColRec cp[FT];
    RowRec rp[FT];
#pragma unroll
    for (int f = 0; f < FT; ++f) {
        const uint32_t t = min(fg + NG * f, (uint32_t)(MT * NT - 1));
        cp[f] = ColRec{};
        rp[f] = RowRec{};
        if (EPI >= 0) {
            cp[f] = load_col_rt<MODE>(p.epi, min(col0 + t / MT * 16 + my_c, p.N - 1), bias, p.B, kbytes);
            rp[f] = load_row_rt<MODE>(p.epi, min(m0 + t % MT * 16 + my_m, p.M - 1), p.A, kbytes);
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
        compute();
        slot = slot + kStage == DEPTH * kStage ? 0 : slot + kStage;
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    v4i *const part = reinterpret_cast<v4i *>(lds);
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < MT; ++m) part[((n * MT + m) * WAVES + wave) * 64 + lane] = acc[n][m];
    __syncthreads();
    const int *const sums = reinterpret_cast<const int *>(lds) + src_lane * 4 + er;
#pragma unroll
    for (int f = 0; f < FT; ++f) {
        const uint32_t t = fg + NG * f;
        if (t < (uint32_t)(MT * NT)) {
            int sum = 0;
#pragma unroll
            for (int v = 0; v < WAVES; ++v) sum += sums[(t * WAVES + v) * 256];
            sum >>= 8;
            const uint32_t m = m0 + t % MT * 16 + my_m, n = col0 + t / MT * 16 + my_c;
            if (m < p.M && n < p.N) {
                if (EPI < 0)
                    c_out[(uint64_t)m * p.N + n] = sum;
                else
                    y_out[(uint64_t)m * p.N + n] = dequant_rt<MODE>(sum, rp[f], cp[f], bias);
            }
        }
    }
}

// ---------------------------------------------------------------------------------
// wide kernel: 5 <= M <= 64, more than 8192 columns, K <= 8192 (what takes_wide_kernel gives it)
// ---------------------------------------------------------------------------------
// The MFMA kernel's plan, several column tiles per workgroup against activations held in registers, with the LDS kernel's way
// in: weights arrive in whole cache lines, without registers, and six to eight steps of 2 KB per wavefront are in flight
// whatever tile they belong to, so that no tile begins with a wait.  The activations take the same way, as the first steps of
// the sequence.  What bounds a launch is the reading of the weights, 4.7 TB/s at 16 x 28672 x 8192 (4.05 before).  A load whose
// result the compiler waits for would empty that queue: eight wavefronts only load and multiply, and four others fetch the
// parameters, add up the eight partial tiles and store, one tile behind.  Measured (us, weights out of the caches): 16 x 28672 x
// 8192 29.0 -> 24.9, x 16384 x 8192 17.5 -> 15.3, 24 x 28672 x 8192 30.3 -> 27.4, 32 x 11008 x 4096 8.6 -> 7.8, 48 x 11008 x 2048 7.6 -> 6.8.
template <int MT, int KS>
struct WideTile {
    static constexpr int kPart = MT * 8 * 1024;                              // one tile's partial sums
    static constexpr int DEPTH = (160 * 1024 - 2 * kPart) / (8 * 2048) < 8 ? (160 * 1024 - 2 * kPart) / (8 * 2048) : 8;  // steps in flight
    static constexpr int kLds = 2 * kPart + 8 * DEPTH * 2048;
    static_assert(kLds <= 160 * 1024, "LDS");
};
template <int MT, int KS, int EPI>
__global__ __launch_bounds__(768) void gemm_s4_wide_kernel(DUQ_HEAD_DECL, DecodeParams tail)
{
    const DecodeParams p = with_head(tail, DUQ_HEAD_USE);
    using Tile = WideTile<MT, KS>;
    constexpr int MODE = EPI < 0 ? 0 : EPI;
    constexpr int DEPTH = Tile::DEPTH;
    constexpr uint32_t kStage = 2048, kPart = Tile::kPart;
    __shared__ __attribute__((aligned(256))) uint8_t lds[Tile::kLds];
    using ColRec = typename EpiRec<MODE>::Col;
    using RowRec = typename EpiRec<MODE>::Row;

    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t kbytes = p.K >> 1;
    const uint32_t ntiles = (p.N + 15) / 16;
    const uint32_t tile0 = blockIdx.x * p.tiles_per_wg, count = min(p.tiles_per_wg, ntiles - tile0);
    if (wave < 8) {
        const uint32_t l16 = lane & 15u, g = lane >> 4;
        const auto desc = [](const uint8_t *base, uint32_t bytes) {
            const uint64_t a = reinterpret_cast<uint64_t>(base);
            return v4u{(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a), (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)(a >> 32) & 0xFFFFu)),
                       (uint32_t)__builtin_amdgcn_readfirstlane((int)bytes), 0x00020000u};
        };
        const v4u dX = desc(p.A, p.M * kbytes);  // rows past M and N read as zero
        const v4u dW = desc(p.B + (uint64_t)tile0 * 16 * kbytes, min(p.N - tile0 * 16, count * 16) * kbytes);
        // ---- global -> LDS, two instructions of eight rows: sixteen rows' 128 bytes of kilobyte ks; pieces lie at piece ^ (row / 2)
        const uint32_t r0 = lane >> 3, even = ((lane & 7u) ^ (r0 >> 1)) * 16, odd = even ^ 64u;
        const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds + 2 * kPart + wave * (DEPTH * kStage);
        auto load = [&](const v4u d, uint32_t tile, uint32_t ks, uint32_t slot) {
            const uint32_t k = ks * 1024 + wave * 128, row0 = (tile * 16 + r0) * kbytes;
            const uint32_t off0 = k + even < kbytes ? row0 + k + even : kOobOffset;  // K % 64 == 0: a piece is all in or all out
            const uint32_t off1 = k + odd < kbytes ? row0 + 8 * kbytes + k + odd : kOobOffset;
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(lds0 + slot), "v"(off0), "s"(d) : "memory", "m0");
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(lds0 + slot + 1024), "v"(off1), "s"(d) : "memory", "m0");
        };
        // the sequence of steps: KS of every row tile of the activations, then KS of every column tile
        const uint8_t *const own = lds + 2 * kPart + wave * (DEPTH * kStage) + l16 * 128;
        uint32_t slot = 0;
        auto step = [&](v4u(&f)[2], auto &&next) {
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"((DEPTH - 1) * 2) : "memory");
#pragma unroll
            for (int u = 0; u < 2; ++u) f[u] = *reinterpret_cast<const v4u *>(own + slot + ((u * 4 + g) ^ (l16 >> 1)) * 16);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // read: the place takes the step DEPTH further on
            next(slot);
            slot = slot + kStage == DEPTH * kStage ? 0 : slot + kStage;
        };
        auto load_step = [&](uint32_t i, uint32_t to) {  // i: constant in the two loops below
            if (i < MT * KS)
                load(dX, i / KS, i % KS, to);
            else
                load(dW, (i - MT * KS) / KS, (i - MT * KS) % KS, to);
        };
#pragma unroll
        for (int i = 0; i < DEPTH; ++i) load_step(i, i * kStage);
        v4u x[MT][KS][2];
#pragma unroll
        for (int i = 0; i < MT * KS; ++i) step(x[i / KS][i % KS], [&](uint32_t to) { load_step(i + DEPTH, to); });
        for (uint32_t t = 0; t < count; ++t) {
            v4i acc[MT];
#pragma unroll
            for (int m = 0; m < MT; ++m) acc[m] = v4i{0, 0, 0, 0};
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                v4u w[2];
                step(w, [&](uint32_t to) { load(dW, t + (ks + DEPTH) / KS, (ks + DEPTH) % KS, to); });
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    v4u we, wo;
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        we[q] = (w[u][q] << 4) & kNibbleMaskD;
                        wo[q] = w[u][q] & kNibbleMaskD;
                    }
#pragma unroll
                    for (int m = 0; m < MT; ++m) {
                        v4u xe, xo, xv = x[m][ks][u];
                        if (MT * KS > 4) asm volatile("" : "+v"(xv));  // (expanded here: hoisted out of the loop it would double the registers)
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            xe[q] = (xv[q] << 4) & kNibbleMaskD;
                            xo[q] = xv[q] & kNibbleMaskD;
                        }
                        acc[m] = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(v4i, we), __builtin_bit_cast(v4i, xe), acc[m], 0, 0, 0);
                        acc[m] = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(v4i, wo), __builtin_bit_cast(v4i, xo), acc[m], 0, 0, 0);
                        if (MT * KS > 4) __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
            v4i *const part = reinterpret_cast<v4i *>(lds + (t & 1u) * kPart);
#pragma unroll
            for (int m = 0; m < MT; ++m) part[(m * 8 + wave) * 64 + lane] = acc[m];
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the loads past the end)
    } else {
        // ---- four wavefronts finish the tiles: one output per thread and row tile, element er of MFMA lane src_lane
        const uint32_t src_lane = (tid >> 2) & 63u, er = tid & 3u;
        const uint32_t my_m = src_lane & 15u, my_c = (src_lane >> 4) * 4 + er;
        const bool bias = p.epi.bias != nullptr;
        const auto c_out = as_global(p.C);
        const auto y_out = as_global(p.y);
        RowRec rp[MT];
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            rp[m] = RowRec{};
            if (EPI >= 0) rp[m] = load_row_rt<MODE>(p.epi, min(m * 16 + my_m, p.M - 1), p.A, kbytes);
        }
        auto load_cp = [&](uint32_t t) {
            ColRec c{};
            if (EPI >= 0) c = load_col_rt<MODE>(p.epi, min((tile0 + t) * 16 + my_c, p.N - 1), bias, p.B, kbytes);
            return c;
        };
        ColRec cp = load_cp(0);
        for (uint32_t t = 0; t < count; ++t) {
            const ColRec next = load_cp(min(t + 1, count - 1));
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            const int *const sums = reinterpret_cast<const int *>(lds + (t & 1u) * kPart) + src_lane * 4 + er;
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                int sum = 0;
#pragma unroll
                for (int v = 0; v < 8; ++v) sum += sums[(m * 8 + v) * 256];
                sum >>= 8;
                const uint32_t row = m * 16 + my_m, n = (tile0 + t) * 16 + my_c;
                if (row < p.M && n < p.N) {
                    if (EPI < 0)
                        c_out[(uint64_t)row * p.N + n] = sum;
                    else
                        y_out[(uint64_t)row * p.N + n] = dequant_rt<MODE>(sum, rp[m], cp, bias);
                }
            }
            cp = next;
        }
    }
}

// ---------------------------------------------------------------------------------
// dispatch
// ---------------------------------------------------------------------------------
// Every dispatcher below returns whether it launched a kernel: a shape or mode that no instantiated template
// covers launches nothing, and the entry points turn that into an error instead of returning success with the
// output unwritten.
template <int MR, int XS, bool FUSEQ>
bool launch_rows_mode(DecodeParams &p, int epi, hipStream_t stream)
{
    const uint32_t ntiles = (p.N + 4 * DUQ_DEC_R - 1) / (4 * DUQ_DEC_R);  // 16 weight rows per tile
    // One tile per workgroup.  Four rows quantized in the kernel, more than 256 tiles: every workgroup quantizes
    // the rows again, so one round of at most 256 workgroups of eight wavefronts with several tiles each when two
    // register sets of weights fit (rows of at most 8192 elements; measured at K = 4096: N = 6144 5.76 against
    // 6.21 us, N = 11008 7.18 against 7.73).  On pre-quantized rows, or with one or two rows, several tiles per
    // workgroup measured 3-15 % slower than one (four wavefronts per CU keep too few loads in flight): not used
    // there.
    constexpr bool kCanMulti = FUSEQ && MR >= 4 && XS <= (MR == 4 ? 4 : 2);
    const bool multi = kCanMulti && ntiles > 256;
    p.tiles_per_wg = multi ? (ntiles + 255) / 256 : 1;
    const dim3 grid((ntiles + p.tiles_per_wg - 1) / p.tiles_per_wg);
    // wavefronts per workgroup: four, or with three or more rows to quantize WQ (DUQ_DEC_FUSEQ_WAVES above)
    constexpr int WQ = !FUSEQ || MR == 1 ? 4
                       : MR == 2         ? DUQ_DEC_FUSEQ_WAVES_M2
                       : MR == 8         ? DUQ_DEC_FUSEQ_WAVES
                                         : (XS >= 4 ? DUQ_DEC_FUSEQ_WAVES_M4L : DUQ_DEC_FUSEQ_WAVES_M4);
    constexpr int WMULTI = DUQ_DEC_FUSEQ_WAVES;
    bool launched = false;
#define DUQ_ROWS(E)                                                                                              \
    if (multi) {                                                                                                 \
        if constexpr (kCanMulti) {                                                                               \
            DUQ_LAUNCH_HEAD((gemv_s4_rows_kernel<MR, XS, FUSEQ, E, WMULTI, true>), grid, dim3(WMULTI * 64), 0, stream, p); \
            launched = true;                                                                                     \
        }                                                                                                        \
    } else {                                                                                                     \
        DUQ_LAUNCH_HEAD((gemv_s4_rows_kernel<MR, XS, FUSEQ, E, WQ>), grid, dim3(WQ * 64), 0, stream, p);              \
        launched = true;                                                                                         \
    }
    switch (epi) {
    case 0: DUQ_ROWS(0) break;
    case 1: DUQ_ROWS(1) break;
    case 2: DUQ_ROWS(2) break;
    case 3: DUQ_ROWS(3) break;
    case 4: DUQ_ROWS(4) break;
    case 5: DUQ_ROWS(5) break;
    default:
        if constexpr (!FUSEQ) {
            if (epi == -1) { DUQ_ROWS(-1) }
        }
    }
#undef DUQ_ROWS
    return launched;
}

template <int MR, bool FUSEQ>
bool launch_rows_xs(DecodeParams &p, int epi, hipStream_t stream)
{
    const uint32_t kbytes = p.K / 2;
    if (kbytes <= 2048) return launch_rows_mode<MR, 2, FUSEQ>(p, epi, stream);
    if constexpr (MR <= 4) {  // (eight longer rows: quant_gemm_shape)
        if (kbytes <= 4096) return launch_rows_mode<MR, 4, FUSEQ>(p, epi, stream);
        if (kbytes <= 6144) return launch_rows_mode<MR, 6, FUSEQ>(p, epi, stream);
        if (kbytes <= 8192) return launch_rows_mode<MR, 8, FUSEQ>(p, epi, stream);
    }
    return false;
}

template <int WAVES, int SEGS, int MT = 1>
bool launch_mfma_mode(const DecodeParams &p, int epi, hipStream_t stream)
{
    const uint32_t ntiles = (p.N + 15) / 16;
    const dim3 grid((ntiles + p.tiles_per_wg - 1) / p.tiles_per_wg);
#define DUQ_DEC(E) \
    DUQ_LAUNCH_HEAD((gemm_s4_decode_kernel<WAVES, SEGS, E, MT>), grid, dim3(WAVES * 64), 0, stream, p)
    switch (epi) {
    case -1: DUQ_DEC(-1); break;
    case 0: DUQ_DEC(0); break;
    case 1: DUQ_DEC(1); break;
    case 2: DUQ_DEC(2); break;
    case 3: DUQ_DEC(3); break;
    case 4: DUQ_DEC(4); break;
    case 5: DUQ_DEC(5); break;
    default: return false;
    }
#undef DUQ_DEC
    return true;
}

template <bool FUSEQ>
bool launch_decode_any(DecodeParams &p, int epi, hipStream_t stream)
{
    const uint32_t kbytes = p.K / 2;
    if (decode_uses_rows_kernel(p.M)) {
        if (p.M == 1) return launch_rows_xs<1, FUSEQ>(p, epi, stream);
        if (p.M == 2) return launch_rows_xs<2, FUSEQ>(p, epi, stream);
        return launch_rows_xs<4, FUSEQ>(p, epi, stream);
    }
    if constexpr (FUSEQ) {
        return p.M <= 8 && launch_rows_xs<8, true>(p, epi, stream);  // 5..8 rows on more columns than quant_gemm_shape has
    } else {
        const uint32_t ntiles = (p.N + 15) / 16;
        p.tiles_per_wg = decode_tiles_per_workgroup(ntiles);
        constexpr int W = DUQ_DEC_WAVES, S = 32 / W;  // 64-byte segments per wavefront for 2 KB of a row
        const uint32_t mt = (p.M + 15) / 16;
        // rows of up to 4096 / 8192 elements: S, 2 S segments per wavefront; the row tiles whose fragments fit in registers
        // next to two sets of weights (what gemm_kernel_for leaves here)
        if (mt > 4 || kbytes > 4096) return false;
        if (kbytes <= 2048) {
            if (mt == 1) return launch_mfma_mode<W, S, 1>(p, epi, stream);
            if (mt == 2) return launch_mfma_mode<W, S, 2>(p, epi, stream);
            if (mt == 3) return launch_mfma_mode<W, S, 3>(p, epi, stream);
            return launch_mfma_mode<W, S, 4>(p, epi, stream);
        }
        if (mt == 1) return launch_mfma_mode<W, 2 * S, 1>(p, epi, stream);
        if (mt == 2) return launch_mfma_mode<W, 2 * S, 2>(p, epi, stream);
        return false;
    }
}

template <int MT, int NT>
bool launch_lds_mode(DecodeParams &p, int epi, hipStream_t stream)
{
    // groups of rows, and 2^16 over them: (at * m) >> 16 == at / groups while at * (groups - 1) < 2^16
    const uint32_t groups = (p.M + 16 * MT - 1) / (16 * MT), tiles = (p.N + 16 * NT - 1) / (16 * NT);
    if (groups > 1 && groups * tiles > 256) return false;
    p.tiles_per_wg = groups | ((65535 + groups) / groups) << 9;
    const dim3 grid((tiles * groups + 7) / 8 * 8);
#define DUQ_DEC(E) DUQ_LAUNCH_HEAD((gemm_s4_lds_kernel<MT, NT, E>), grid, dim3(512), 0, stream, p)
    switch (epi) {
    case -1: DUQ_DEC(-1); break;
    case 0: DUQ_DEC(0); break;
    case 1: DUQ_DEC(1); break;
    case 2: DUQ_DEC(2); break;
    case 3: DUQ_DEC(3); break;
    case 4: DUQ_DEC(4); break;
    case 5: DUQ_DEC(5); break;
    default: return false;
    }
#undef DUQ_DEC
    return true;
}

template <int MT, int KS>
bool launch_wide_mode(DecodeParams &p, int epi, hipStream_t stream)
{
    const uint32_t ntiles = (p.N + 15) / 16;
    p.tiles_per_wg = decode_tiles_per_workgroup(ntiles);
    const dim3 grid((ntiles + p.tiles_per_wg - 1) / p.tiles_per_wg);
#define DUQ_DEC(E) DUQ_LAUNCH_HEAD((gemm_s4_wide_kernel<MT, KS, E>), grid, dim3(768), 0, stream, p)
    switch (epi) {
    case -1: DUQ_DEC(-1); break;
    case 0: DUQ_DEC(0); break;
    case 1: DUQ_DEC(1); break;
    case 2: DUQ_DEC(2); break;
    case 3: DUQ_DEC(3); break;
    case 4: DUQ_DEC(4); break;
    case 5: DUQ_DEC(5); break;
    default: return false;
    }
#undef DUQ_DEC
    return true;
}

bool launch_wide_any(DecodeParams &p, int epi, hipStream_t stream)
{
    const uint32_t mt = (p.M + 15) / 16, ks = p.K <= 2048 ? 1 : p.K <= 4096 ? 2 : 4;  // kilobytes of a row
    if (mt == 1 && ks == 4) return launch_wide_mode<1, 4>(p, epi, stream);
    if (mt == 2 && ks == 4) return launch_wide_mode<2, 4>(p, epi, stream);
    if (mt == 2 && ks == 2) return launch_wide_mode<2, 2>(p, epi, stream);
    if (mt == 2) return launch_wide_mode<2, 1>(p, epi, stream);
    if (mt == 3 && ks == 1) return launch_wide_mode<3, 1>(p, epi, stream);
    if (mt == 4 && ks == 1) return launch_wide_mode<4, 1>(p, epi, stream);
    return false;
}

bool launch_lds_any(DecodeParams &p, int epi, hipStream_t stream)
{
    const LdsShape tile = lds_shape(p.M, p.N);
#define DUQ_LDS(MT) (tile.cols == 2 ? launch_lds_mode<MT, 2>(p, epi, stream) : launch_lds_mode<MT, 1>(p, epi, stream))
    switch (tile.rows) {
    case 1: return DUQ_LDS(1);
    case 2: return DUQ_LDS(2);
    case 3: return DUQ_LDS(3);
    case 4: return DUQ_LDS(4);
    default: return false;
    }
#undef DUQ_LDS
}

}  // namespace

// Measurement aid: the rows kernel's access pattern without its arithmetic (every lane requests 8 x 16 bytes up
// front, a load instruction covers 1 KB, one workgroup per 32 KB) over `bytes` of memory, nothing stored.  What
// this takes for N * K / 2 bytes is the floor of a decode launch of that size on the part.
__global__ __launch_bounds__(256) void probe_read_kernel(const v4u *src, uint32_t nvec, uint32_t *sink)
{
    const uint32_t gw = (blockIdx.x * 256 + threadIdx.x) >> 6, lane = threadIdx.x & 63u;
    const __amdgpu_buffer_rsrc_t r = make_rsrc(src, nvec * 16);
    v4u v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const uint32_t idx = gw * 512 + i * 64 + lane;
        v[i] = __builtin_bit_cast(
            v4u, __builtin_amdgcn_raw_buffer_load_b128(r, (int)(idx < nvec ? idx * 16 : kOobOffset), 0, DUQ_DEC_WLOAD_AUX));
    }
    uint32_t x = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) x ^= (v[i][0] ^ v[i][1]) ^ (v[i][2] ^ v[i][3]);
    if (x == 0x9E3779B9u && sink) sink[gw & 63u] = x;  // keeps the loads alive; practically never taken
}

int launch_probe_read(const void *src, uint64_t bytes, uint32_t *sink, hipStream_t stream)
{
    const uint32_t nvec = (uint32_t)(bytes / 16);
    if (nvec == 0) return 0;
    const uint32_t waves = (nvec + 511) / 512;
    hipLaunchKernelGGL(probe_read_kernel, dim3((waves + 3) / 4), dim3(256), 0, stream, static_cast<const v4u *>(src), nvec,
                       sink);
    return (int)hipGetLastError();
}

int launch_decode_s4(const uint8_t *A, const uint8_t *B, uint32_t M, uint32_t N, uint32_t K, int32_t *out_acc,
                     const Epilogue *epi, uint16_t *y, hipStream_t stream)
{
    DecodeParams p{};
    p.A = A;
    p.B = B;
    p.M = M;
    p.N = N;
    p.K = K;
    p.C = out_acc;
    p.y = y;
    if (epi) p.epi = *epi;
    const int mode = out_acc ? -1 : epi->mode;
    if (!(takes_wide_kernel(M, N, K) ? launch_wide_any(p, mode, stream) : takes_lds_kernel(M, N, K, mode == 5) ? launch_lds_any(p, mode, stream) : launch_decode_any<false>(p, mode, stream))) return (int)hipErrorInvalidValue;
    return (int)hipGetLastError();
}

int launch_decode_fp16in(const uint16_t *x, float clip, int qmax, const uint8_t *B, uint32_t M, uint32_t N, uint32_t K,
                         const Epilogue &epi, uint16_t *y, uint8_t *q_out, uint16_t *s_out, uint16_t *z_out,
                         int32_t *rs_out, hipStream_t stream)
{
    DecodeParams p{};
    p.X = x;
    p.B = B;
    p.M = M;
    p.N = N;
    p.K = K;
    p.y = y;
    p.epi = epi;
    p.clip = clip;
    p.qmax = qmax;
    p.q_out = q_out;
    p.s_out = s_out;
    p.z_out = z_out;
    p.rs_out = rs_out;
    if (!launch_decode_any<true>(p, epi.mode, stream)) return (int)hipErrorInvalidValue;
    return (int)hipGetLastError();
}

}  // namespace duq
