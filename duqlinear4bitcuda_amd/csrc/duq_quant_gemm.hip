// Quantizer, GEMM and dequant of a few dozen rows in one launch: binary16 activations in.
//
// A workgroup quantizes the rows of its tile itself, through the same RowQuant code as the stand-alone quantizer (scale:
// qlinear4bit/nn/quantizer.py:13, codes: src/kernels/quant.cu:11-45, :99-132), while its whole share of the weights comes to LDS.
// As two launches a step of few or short rows cost 8.2 us of host time, and in a graph 4.7 at least, more than its work: 46 rows 1231 x
// 1216 8.3 -> 5.7 called eagerly, 5.6 -> 4.3 in a graph.  What bounds it: every workgroup repeats the quantizer's vector work for its
// rows, about 31 instructions per eight elements (2.2 us for the 65536 elements a workgroup can have), behind one trip to memory
// and its fetch of the rows (128 KB there, 1.2 us); then the launch.  So a tile is as few rows as one round of workgroups allows.
#include "duq_decode_common.h"

namespace duq {

namespace {

// The first 56 bytes (through y) reach the kernel in registers (DUQ_HEAD_DECL / with_head).
struct QuantGemmParams {
    const uint16_t *X;  // binary16 activations [M, K]
    const uint8_t *B;   // packed weights [N, K/2]
    uint32_t M, N, K;
    uint32_t groups;    // of rows, and 2^16 over them from bit 9 on
    uint32_t chunks;    // of columns, in a workgroup
    float clip;
    int qmax;
    uint32_t reserved;
    uint16_t *y;
    Epilogue epi;       // (what concerns rows is not read: the kernel computes it)
    uint8_t *q_out;     // optional: the packed codes [M, K/2], scales, zero points and sums of the rows (written by the workgroups
    uint16_t *s_out, *z_out;  // of the first columns)
    int32_t *rs_out;
};
static_assert(offsetof(QuantGemmParams, epi) == kHeadBytes, "the fields delivered in registers");

// ROWS rows of eight wavefronts in one or two passes (the first one's codes are made while the second one's rows arrive), each row
// held by 512 * PASSES / ROWS lanes, UPL units of eight elements a lane.
template <int ROWS, int PASSES, int UPL, int NT, int BUFS, bool SPLIT>
struct QuantTile {
    static constexpr int LPR = 512 * PASSES / ROWS, RPI = 64 / LPR, MT = (ROWS + 15) / 16;  // lanes of a row, rows of a wavefront and pass, row tiles
    static_assert(LPR >= 8 && LPR <= 64, "lanes of a row");
    static constexpr int KB = LPR * UPL * 4;                      // bytes of the longest packed row
    // SPLIT: the wavefronts split K, a wavefront multiplies SLICE bytes of every row of the tile at a time.  Otherwise each has one of the
    // eight 16 x 16 tiles, and all of K.
    static constexpr int SLICE = SPLIT && KB / 8 < 128 ? KB / 8 : 128;
    static constexpr int V = SPLIT ? 8 : 1, S = KB / V / SLICE, U = SLICE / 64;  // wavefronts and slices of one along K, 64-byte fragments in a slice
    static constexpr int XSTRIDE = KB + 16;                       // (the rows of a fragment read fall on different banks)
    static constexpr int kX = ROWS * XSTRIDE, kW = NT * 16 * KB /* of one buffer */, kPart = SPLIT ? NT * MT * 8 * 1024 : 0;
    static_assert(U >= 1 && (SPLIT || MT * NT == 8), "work for every wavefront");
    static_assert(kX + BUFS * kW + kPart <= 159 * 1024, "LDS");
};

// Eight wavefronts quantize and then multiply, four others only fetch the weights (a wavefront's wait for its activations would
// otherwise be a wait for the weights it requested too).  Sums as in the other decode kernels: the wavefronts split K, eight
// partial tiles meet in LDS.  A workgroup takes p.chunks times NT column tiles, with BUFS = 2 the next ones' weights on their way
// while it multiplies.
template <int ROWS, int PASSES, int UPL, int NT, int BUFS, bool SPLIT, int EPI>
__global__ __launch_bounds__(768) void quant_gemm_s4_kernel(DUQ_HEAD_DECL, QuantGemmParams tail)
{
    const QuantGemmParams p = with_head(tail, DUQ_HEAD_USE);
    using Tile = QuantTile<ROWS, PASSES, UPL, NT, BUFS, SPLIT>;
    constexpr int LPR = Tile::LPR, RPI = Tile::RPI, MT = Tile::MT, V = Tile::V, S = Tile::S, U = Tile::U;
    constexpr uint32_t SLICE = Tile::SLICE, XSTRIDE = Tile::XSTRIDE;
    constexpr bool ASYM = EPI == 1 || EPI == 3 || EPI == 4 || EPI == 5, SHIFT = EPI == 4 || EPI == 5;
    __shared__ __attribute__((aligned(256))) uint8_t lds_w[BUFS * Tile::kW];
    __shared__ __attribute__((aligned(16))) uint8_t xs[Tile::kX];
    __shared__ v4i part[SPLIT ? NT : 1][SPLIT ? MT : 1][8][SPLIT ? 64 : 1];
    __shared__ uint16_t srow[MT * 16], zrow[MT * 16];
    __shared__ int rsrow[MT * 16];
    using ColRec = typename EpiRec<EPI>::Col;
    using RowRec = typename EpiRec<EPI>::Row;

    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t l16 = lane & 15u, g = lane >> 4;
    const uint32_t kbytes = p.K >> 1;
    // groups of ROWS rows share the weights of a column range: consecutive in `at`, an eighth of which runs on one XCD
    const uint32_t width = 16 * NT * (BUFS == 1 ? 1 : p.chunks);
    const uint32_t groups = p.groups & 0x1FFu, per_xcd = ((p.N + width - 1) / width * groups + 7) / 8;
    const uint32_t at = blockIdx.x % 8 * per_xcd + blockIdx.x / 8, tile = at * (p.groups >> 9) >> 16;  // (tile = at / groups)
    const uint32_t col0 = tile * width, m0 = (at - tile * groups) * ROWS;
    if (col0 >= p.N) return;
    const uint32_t chunks = BUFS == 1 ? 1 : min(p.chunks, (p.N - col0 + 16 * NT - 1) / (16 * NT));
    auto sync = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

    // ---- the wavefronts that fetch: instruction i takes kilobyte i of [column tile][slice][wavefront], rows of SLICE bytes whose
    // 16-byte pieces lie at piece ^ (row / Q), so that the sixteen rows of a fragment read sixteen places
    constexpr uint32_t PR = SLICE / 16, RPW = 64 / PR, Q = 256 / SLICE;   // pieces a row, rows an instruction
    if (wave >= 8) {
        const uint64_t a = reinterpret_cast<uint64_t>(p.B + (uint64_t)col0 * kbytes);
        const v4u dW = {(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a), (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)(a >> 32) & 0xFFFFu)),
                        (uint32_t)__builtin_amdgcn_readfirstlane((int)(min(p.N - col0, width) * kbytes)), 0x00020000u};  // rows past N read as zero
        const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds_w;
        constexpr uint32_t kInstr = Tile::kW / 1024;
        static_assert(kInstr % 4 == 0 && BUFS * (kInstr / 4) <= 63, "vmcnt");
        auto fetch = [&](uint32_t chunk) {
#pragma unroll
            for (uint32_t j = 0; j < kInstr / 4; ++j) {
                const uint32_t i = j * 4 + (wave - 8);
                const uint32_t r = i % (16 / RPW) * RPW + lane / PR, v = i / (16 / RPW) % V, s = i / (16 / RPW) / V % S, n = i / (16 / RPW) / V / S;
                const uint32_t k = (s * V + v) * SLICE + ((lane % PR) ^ (r / Q)) * 16;
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(lds0 + (chunk % BUFS) * Tile::kW + i * 1024),
                             "v"(k < kbytes ? ((chunk * NT + n) * 16 + r) * kbytes + k : kOobOffset), "s"(dW)
                             : "memory", "m0");
            }
        };
        if (ROWS == 8) __builtin_amdgcn_s_barrier();  // (behind the requests for the activations, which are needed first)
        fetch(0);
        if (BUFS == 1) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            sync();  // the weights are here, and everybody's codes
            if (SPLIT) sync();  // the partial sums are written
        } else if (SPLIT) {
            fetch(1);  // (rows past the workgroup's read as zero)
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kInstr / 4) : "memory");
            sync();
            for (uint32_t c = 0; c < chunks; ++c) {
                if (c > 0) sync();  // the last chunk's partial sums are read
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                sync();  // this chunk's partial sums are written (its weights read), and the next one's weights are here
                fetch(c + 2);
            }
        } else {
            fetch(1);
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

    // ---- the wavefronts that quantize: lane l holds units l % LPR, + LPR, ... of row l / LPR of this wavefront's
    const uint32_t nunits = p.K >> 3, u0 = lane % LPR;
    const __amdgpu_buffer_rsrc_t rX = make_rsrc(p.X + (uint64_t)m0 * p.K, min(p.M - m0, (uint32_t)ROWS) * p.K * 2);  // rows past M read as zero
    v4u raw[PASSES][UPL];
#pragma unroll
    for (int s = 0; s < PASSES; ++s) {
        const uint32_t x0 = (((s * 8 + wave) * RPI + lane / LPR) * p.K + u0 * 8) * 2;
#pragma unroll
        for (int j = 0; j < UPL; ++j) raw[s][j] = buf_load16(rX, u0 + j * LPR < nunits ? x0 + j * (LPR * 16) : kOobOffset, 0);
    }
    if (ROWS == 8) __builtin_amdgcn_s_barrier();
    // the parameters of the outputs this thread finishes, behind them.  SPLIT: 256 threads take half of the column tiles (one row
    // tile), or half of the row tiles; otherwise a lane holds four columns of a row of its wavefront's tile
    constexpr int FN = !SPLIT ? 4 : MT == 1 ? (NT + 1) / 2 : NT, FM = !SPLIT || MT == 1 ? 1 : MT / 2;
    const uint32_t src_lane = (tid >> 2) & 63u, er = tid & 3u, fg = tid >> 8;
    const uint32_t my_m = SPLIT ? src_lane & 15u : l16, my_c = (src_lane >> 4) * 4 + er;
    const bool bias = p.epi.bias != nullptr;
    const auto y_out = as_global(p.y);
    ColRec cp[FN], cpn[FN];
    auto column = [&](uint32_t chunk, int f) {
        return col0 + (SPLIT ? (chunk * NT + (MT == 1 ? f * 2 + fg : f)) * 16 + my_c : (chunk * NT + wave / MT) * 16 + g * 4 + f);
    };
    auto fetch_columns = [&](uint32_t chunk, ColRec(&c)[FN]) {
#pragma unroll
        for (int f = 0; f < FN; ++f) c[f] = load_col_rt<EPI>(p.epi, min(column(chunk, f), p.N - 1), bias, p.B, kbytes);
    };
    fetch_columns(0, cp);
#pragma unroll
    for (int s = 0; s < PASSES; ++s) {
        const uint32_t qrow = (s * 8 + wave) * RPI + lane / LPR;
        const bool live = m0 + qrow < p.M;
        if (RPI == 1 && !live) break;
        // (units past the row end read as zero: no maximum of |x| changes, a minimum or maximum would)
        PkMinMax st;
#pragma unroll
        for (int j = 0; j < UPL; ++j)
            if (!ASYM || u0 + j * LPR < nunits) st.add8(raw[s][j]);
        uint32_t m16;
        float lo = 0.f, hi = 0.f;
        if constexpr (!ASYM) {
            m16 = lanes_reduce<LPR>(st.absmax_bits(), [](uint32_t x, uint32_t y) { return max(x, y); });
        } else {
            st.mx = lanes_reduce<LPR>(st.mx, [](uint32_t x, uint32_t y) {
                asm("v_pk_maximum3_f16 %0, %0, %1, %1" : "+v"(x) : "v"(y));
                return x;
            });
            st.mn = lanes_reduce<LPR>(st.mn, [](uint32_t x, uint32_t y) {
                asm("v_pk_minimum3_f16 %0, %0, %1, %1" : "+v"(x) : "v"(y));
                return x;
            });
            m16 = st.absmax_bits();
            lo = st.min_f32();
            hi = st.max_f32();
            if (m16 > 0x7C00u) lo = hi = __builtin_nanf("");  // torch's min / max return NaN for a row that holds one
            if (RPI > 1 && !live) hi = 15.f;  // (zeros alone would send the rows beside them down the element-wise path)
        }
        RowQuant<ASYM, RPI == 1> rq;
        rq.init(m16, lo, hi, p.clip, p.qmax);
        int code_sum = 0;
        uint8_t *const to = xs + qrow * XSTRIDE;
        auto put = [&](uint32_t c, uint32_t word) {
            if (c >= nunits) return;
            if (SHIFT) {
                word ^= 0x88888888u;  // u - 8 as a signed nibble is u with bit 3 flipped
                code_sum = __builtin_amdgcn_sdot8((int)word, 0x11111111, code_sum, false);
            }
            *reinterpret_cast<uint32_t *>(to + c * 4) = word;
        };
        if (rq.fast) {
#pragma unroll
            for (int j0 = 0; j0 < UPL; j0 += 4) {
                if ((uint32_t)(j0 * LPR) >= nunits) break;
                v4u in[4];
                uint32_t words[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) in[j] = raw[s][j0 + j];
                rq.quant_units_packed(in, words);
#pragma unroll
                for (int j = 0; j < 4; ++j) put(u0 + (j0 + j) * LPR, words[j]);
            }
        } else {  // a row with a NaN or an infinity: element by element, in a loop that fetches them again
#pragma unroll 1
            for (uint32_t c = u0; c < nunits; c += 4 * LPR) {
                v4u in[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) in[j] = buf_load16(rX, c + j * LPR < nunits ? (qrow * p.K + (c + j * LPR) * 8) * 2 : kOobOffset, 0);
#pragma unroll
                for (int j = 0; j < 4; ++j) put(c + j * LPR, quant8_exact<ASYM>(in[j], rq.rcp, rq.qmax, rq.zi));
            }
        }
        if (SHIFT) code_sum = (int)lanes_reduce<LPR>((uint32_t)code_sum, [](uint32_t x, uint32_t y) { return x + y; });
        if (u0 == 0) {
            srow[qrow] = f16_to_bits(rq.s);
            if (ASYM) zrow[qrow] = f16_to_bits(SHIFT ? rq.z - (f16)8.0f : rq.z);
            if (SHIFT) rsrow[qrow] = code_sum;
        }
    }
    if (SPLIT || BUFS == 1) sync();

    // ---- products of this wavefront's slices of the rows
    // (bytes past the row end, and rows past M, hold anything: the weights read as zero there, and a row's codes only reach that
    // row's outputs)
    // (one tile to a wavefront, several chunks: its rows' fragments stay in registers, expanded)
    constexpr bool kHold = !SPLIT && BUFS > 1;
    v4u he[kHold ? S * U : 1], ho[kHold ? S * U : 1];
    if constexpr (kHold) {
        sync();  // the codes are here, and the first chunk's weights
#pragma unroll
        for (int f = 0; f < S * U; ++f) {
            const v4u x = load16(xs + (wave % MT * 16 + l16) * XSTRIDE + f * 64 + g * 16);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                he[f][q] = (x[q] << 4) & kNibbleMaskD;
                ho[f][q] = x[q] & kNibbleMaskD;
            }
        }
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
            if ((s * V + v) * SLICE >= kbytes) break;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                v4u xe[AM], xo[AM];
#pragma unroll
                for (int m = 0; m < AM; ++m) {
                    if (kHold) {
                        xe[m] = he[s * U + u];
                        xo[m] = ho[s * U + u];
                        continue;
                    }
                    const v4u x = load16(xr + m * (16 * XSTRIDE) + s * (V * SLICE) + u * 64);
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        xe[m][q] = (x[q] << 4) & kNibbleMaskD;
                        xo[m][q] = x[q] & kNibbleMaskD;
                    }
                }
#pragma unroll
                for (int n = 0; n < AN; ++n) {
                    const v4u w = load16(ws + (n * S + s) * (V * 16 * SLICE) + ((u * 4 + g) ^ (l16 / Q)) * 16);
                    v4u we, wo;
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        we[q] = (w[q] << 4) & kNibbleMaskD;
                        wo[q] = w[q] & kNibbleMaskD;
                    }
#pragma unroll
                    for (int m = 0; m < AM; ++m) {
                        acc[n][m] = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(v4i, we), __builtin_bit_cast(v4i, xe[m]), acc[n][m], 0, 0, 0);
                        acc[n][m] = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(v4i, wo), __builtin_bit_cast(v4i, xo[m]), acc[n][m], 0, 0, 0);
                    }
                }
            }
        }
        if constexpr (SPLIT) {
            if (BUFS > 1 && chunk > 0) sync();
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
            RowRec rp{};
            if (ROWS >= 16 || row < ROWS) {
                if constexpr (EPI == 5) {
                    const v2u head = *reinterpret_cast<const v2u *>(xs + row * XSTRIDE);
                    rp.xlo = head[0];
                    rp.xhi = head[1] & 0xFFu;
                    rp.zx = (uint32_t)rint_i32((float)bits_to_f16(zrow[row]));
                    rp.sx = (float)bits_to_f16(srow[row]);
                    rp.rxl = dual_head_sum(rp.xlo, rp.xhi);
                    rp.rxr = (uint32_t)rsrow[row] - rp.rxl;
                } else {
                    rp.s = bits_to_f16(srow[row]);
                    if (ASYM) rp.z = bits_to_f16(zrow[row]);
                    if (SHIFT) rp.rs = rsrow[row];
                }
            }
            const uint32_t m = m0 + row;
            uint16_t out[FN];
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
                sum >>= 8;
                out[f] = dequant_rt<EPI>(sum, rp, cp[f], bias);
                const uint32_t n = column(chunk, f);
                if (SPLIT && m < p.M && n < p.N && (ROWS >= 16 || row < ROWS)) y_out[(uint64_t)m * p.N + n] = out[f];
            }
            if constexpr (!SPLIT) {
                const uint32_t n = column(chunk, 0);
                if (m < p.M && n < p.N) {
                    typedef v2u v2u_any __attribute__((aligned(2)));
                    const auto to = y_out + (uint64_t)m * p.N + n;
                    if (n + 3 < p.N) {
                        *(__attribute__((address_space(1))) v2u_any *)to = v2u{(uint32_t)out[0] | (uint32_t)out[1] << 16, (uint32_t)out[2] | (uint32_t)out[3] << 16};
                    } else {
#pragma unroll
                        for (int f = 0; f < 4; ++f)
                            if (n + f < p.N) to[f] = out[f];
                    }
                }
            }
        }
        if (BUFS > 1)
#pragma unroll
            for (int f = 0; f < FN; ++f) cp[f] = cpn[f];
    }

    // ---- what the caller asked for of the quantizer
    if (col0 != 0) return;
    const uint32_t rows = min(p.M - m0, (uint32_t)ROWS);
    if (p.q_out)
        for (uint32_t r = wave; r < rows; r += 8)
            for (uint32_t c = lane; c < nunits; c += 64)
                reinterpret_cast<uint32_t *>(p.q_out + (uint64_t)(m0 + r) * kbytes)[c] = *reinterpret_cast<const uint32_t *>(xs + r * XSTRIDE + c * 4);
    if (tid < rows) {
        if (p.s_out) p.s_out[m0 + tid] = srow[tid];
        if (ASYM && p.z_out) p.z_out[m0 + tid] = zrow[tid];
        if (SHIFT && p.rs_out) p.rs_out[m0 + tid] = rsrow[tid];
    }
}

template <int ROWS, int PASSES, int UPL, int NT, int BUFS, bool SPLIT>
bool launch_shape(QuantGemmParams &p, uint32_t chunks, hipStream_t stream)
{
    using Tile = QuantTile<ROWS, PASSES, UPL, NT, BUFS, SPLIT>;
    // groups of rows, and 2^16 over them: (at * m) >> 16 == at / groups while at * (groups - 1) < 2^16
    const uint32_t width = 16 * NT * chunks;
    const uint64_t groups = (p.M + ROWS - 1) / ROWS, tiles = (p.N + width - 1) / width;
    if (groups > 64 || (groups > 1 && (groups * tiles + 8) * (groups - 1) >= 65536) || p.K > 2 * Tile::KB || (uint64_t)width * (p.K / 2) >= kOobOffset) return false;
    p.groups = (uint32_t)groups | (uint32_t)((65535 + groups) / groups) << 9;
    p.chunks = chunks;
    const dim3 grid((uint32_t)((tiles * groups + 7) / 8 * 8));
#define DUQ_QG(E) DUQ_LAUNCH_HEAD((quant_gemm_s4_kernel<ROWS, PASSES, UPL, NT, BUFS, SPLIT, E>), grid, dim3(768), 0, stream, p)
    switch (p.epi.mode) {
    case 0: DUQ_QG(0); break;
    case 1: DUQ_QG(1); break;
    case 2: DUQ_QG(2); break;
    case 3: DUQ_QG(3); break;
    case 4: DUQ_QG(4); break;
    case 5: DUQ_QG(5); break;
    default: return false;
    }
#undef DUQ_QG
    return true;
}

}  // namespace

int launch_quant_gemm(QuantGemmShape s, const uint16_t *x, float clip, int qmax, const uint8_t *B, uint32_t M, uint32_t N, uint32_t K,
                      const Epilogue &epi, uint16_t *y, uint8_t *q_out, uint16_t *s_out, uint16_t *z_out, int32_t *rs_out,
                      hipStream_t stream)
{
    QuantGemmParams p{x, B, M, N, K, 0, 0, clip, qmax, 0, y, epi, q_out, s_out, z_out, rs_out};
    bool launched = false;
    const bool one_pass = (uint64_t)s.rows * K <= 32768;  // eight units for every lane
#define DUQ_QS(R, P, U, C, B)                                                                                              \
    if (s.rows == R && (R == 8 ? one_pass == (U == 8) : one_pass == (P == 1)) && s.cols == C && (s.chunks > 1) == (B > 1)) \
        launched = launch_shape<R, P, U, C, B, (R / 16 * C < 8)>(p, s.chunks, stream);
    DUQ_QS(8, 1, 8, 1, 1)
    DUQ_QS(8, 1, 8, 2, 1)
    DUQ_QS(8, 1, 8, 3, 1)
    DUQ_QS(8, 1, 16, 1, 1)
    DUQ_QS(16, 1, 8, 1, 1)
    DUQ_QS(16, 1, 8, 2, 1)
    DUQ_QS(16, 1, 8, 3, 1)
    DUQ_QS(16, 1, 8, 8, 1)
    DUQ_QS(16, 2, 8, 2, 1)
    DUQ_QS(16, 2, 8, 3, 1)
    DUQ_QS(16, 2, 8, 1, 2)
    DUQ_QS(32, 1, 8, 4, 1)
    DUQ_QS(32, 1, 8, 4, 2)
#undef DUQ_QS
    return launched ? (int)hipGetLastError() : (int)hipErrorInvalidValue;
}

}  // namespace duq
