// Prefill GEMM on packed int4 operands (v_mfma_i32_32x32x32_i8): both operands travel packed from memory into LDS, every
// wavefront expands the fragments it multiplies.  Definition and nibble arithmetic: duq_gemm.hip.
//
// What bounds it: at 256 x 256 tiles the matrix cores at the clock the part holds under them (4096 x 4096 x 16384: 178 us
// = 3.1 POP/s; a loop of nothing but these MFMAs reaches 3.7 on random operands).  On smaller tiles the two vector
// instructions per word and parity that the expansion costs, and LDS, share the time with the MFMAs (64 x 128 tiles, per
// 256 k: 0.22 us of MFMAs, 0.25 of LDS traffic and loads, 0.25 of expansion; 0.44 together).
//
// Why this shape.  A wavefront that is alone on its SIMD issues a vector instruction every eight cycles, two of them one
// every four: eight wavefronts per workgroup, so that the expansion fits beside the MFMAs.  A fragment of either operand
// costs its expansion once per wavefront that reads it, so a wavefront's own tile is as large as it gets: 64 x 64 or
// 128 x 64 outputs, and on the small tiles the wavefronts of a workgroup split K (KS) instead of the tile, which also
// saves LDS reads; their sums meet in LDS once, at the end.  Operands go to LDS without passing through registers
// (buffer_load ... lds), several stages of them in flight: the loads of a stage have all the stages before it to arrive.
// Before, one 64 x 128 tile kept four wavefronts, whose activations were loaded and used within a chunk (the wait for
// them was 1100 of the 1700 cycles of a 256-k chunk): 512 x 4096 x 11008 (K) 34.7 -> 26.6 us, 77 x 13824 x 5120 19.0 ->
// 14.3, 128 x 4096 x 11008 25.1 -> 19.9, 1024 x 11008 x 4096 55.5 -> 45, 4096 x 4096 x 4096 58 -> 53.5; rows of more than
// 16384 elements, formerly on a kernel of 64 x 64 tiles, 9 x 11008 x 20480 79 -> 31 us, 2048 x 512 x 28672 81 -> 44.6.
//
// Few rows (65..256 on a few thousand columns, 17..64 long ones) leave most CUs without a 64 x 128 tile, and there a
// launch lasts as long as one workgroup's walk over K.  64 x 64 tiles (96 x 64 for 65..96 rows on wide layers) whose eight
// wavefronts each take an eighth of every stage: twice the workgroups, half the walk (0.2 us per 256 k against 0.44),
// for a longer end, since eight partial tiles have to meet (5.5 us with the start against 3.6).  128 x 4096 x 4096 10.5 ->
// 8.7 us, 128 x 4096 x 11008 22.5 -> 16.9, 64 x 4096 x 16384 30.6 -> 22.7, 77 x 4096 x 28672 43.4 -> 32.5 (these narrow ones run
// the LDS kernel of duq_decode.hip by now); 96 x 64: 77 x 13824 x 5120 15.1 -> 14.4 (3.9 TB/s of weights).  A 128 x 64 tile
// measured behind 64 x 128 (512 x 4096 x 4096 13.4 against 12.4).
#include "duq_gemm_common.h"
#include <type_traits>

namespace duq {

// Stages of (BM + BN) rows that fit beside one another in LDS, six at most.
constexpr int stages_of(int bytes) { return 147456 / bytes > 6 ? 6 : 147456 / bytes; }

// WTM x WTN: 32 x 32 tiles of a wavefront.  WM x WN: wavefronts over the rows and columns of the workgroup's tile, KS of
// them over k.  kRowB: bytes of a row in a stage (128 = 256 elements, or 256 where the tile is small: half the barriers).
template <int WTM_, int WTN_, int WM_, int WN_, int KS_, int kRowB_>
struct PrefillTile {
    static constexpr int WTM = WTM_, WTN = WTN_, WM = WM_, WN = WN_, KS = KS_, kRowB = kRowB_;
    static constexpr int BM = 32 * WTM * WM, BN = 32 * WTN * WN;
    static constexpr int NST = stages_of((BM + BN) * kRowB);
    static constexpr uint32_t kStage = (BM + BN) * kRowB;
    static constexpr int TM = KS == 8 ? 1 : KS == 4 ? WTM / 2 : WTM, TN = KS == 1 ? WTN : WTN / 2;  // what a wavefront finishes after the loop
    static constexpr uint32_t kEpiLds = 8 * (32 * TM) * (64 * TN + 16), kXchg = KS == 1 ? 0 : KS == 8 ? WTM * WTN * 4096 : 8 * (KS - 1) * TM * TN * 4096;
    static constexpr uint32_t kLds = NST * kStage > kEpiLds ? (NST * kStage > kXchg ? NST * kStage : kXchg) : (kEpiLds > kXchg ? kEpiLds : kXchg);
};

// The tile of rows m0 .. and columns n0 ...  lds: Tile::kLds bytes; dpar, dwide: staged parameters of EPI 5.
template <typename Tile, int EPI, bool BIAS>
__device__ __forceinline__ void prefill_tile(GemmParams &p, uint8_t *lds, uint32_t *dpar, uint32_t &dwide, const uint32_t m0, const uint32_t n0)
{
    constexpr int WTM = Tile::WTM, WTN = Tile::WTN, WM = Tile::WM, WN = Tile::WN, KS = Tile::KS, kRowB = Tile::kRowB;
    static_assert(WM * WN * KS == 8, "eight wavefronts");
    static_assert(WTN >= 2 && 4 * (WTM + WTN) / (WTM * WTN) <= 4, "the last slot expands words of the last weight tile only");
    constexpr int BM = Tile::BM, BN = Tile::BN, NST = Tile::NST;
    constexpr uint32_t kStage = Tile::kStage;
    constexpr int RPL = 1024 / kRowB, LPR = 64 / RPL;  // rows per load instruction, lanes per row
    constexpr int L = (BM + BN) / (8 * RPL);  // loads per wavefront and stage
    constexpr int LX = BM / (8 * RPL);               // ... of which bring activation rows
    constexpr int STEPS = kRowB / 32 / KS;             // steps of a wavefront per stage
    constexpr int H = WTM * WTN;              // MFMAs per nibble parity of a step
    constexpr int P = WTM + WTN;              // fragments per step
    constexpr int W = 4 * P;                  // words a lane expands per step and parity
    constexpr int T = WTM * WTN;
    constexpr int TM = Tile::TM, TN = Tile::TN;
    constexpr bool LATE = WTM * WTN == 8;     // no registers to spare in the loop: parameters after it
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t l32 = lane & 31u, h = lane >> 5;
    const uint32_t ks = wave / (WM * WN), w4 = wave % (WM * WN);
    const uint32_t wm = w4 / WN, wn = w4 % WN;
    const uint32_t kbytes = p.K >> 1;
    const uint32_t nchunks = (kbytes + kRowB - 1) / kRowB;

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
            const uint32_t rxl = dual_head_sum(xlo, xhi);
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
    }

    // ---- global -> LDS.  Load j of this wavefront brings rows 8 * (8 * j + wave) .. + 7 of the stage (activation rows
    // first, then weight rows; 4 rows of 256 bytes with kRowB = 256), whole cache lines of each.  The instruction puts lane
    // l's 16 bytes at 16 * l behind its base, so it is the lane's SOURCE that swizzles: piece q of row r lies at position
    // q ^ ((r / 2) % 8) of the row's 128 bytes (q ^ (r % 16) of 256), which spreads the sixteen rows x 16 bytes that a
    // fragment read serves at once over all banks.
    const uint32_t lrow = lane / LPR, lpos = lane % LPR;
    auto desc = [](const uint8_t *base, uint32_t bytes) {
        const uint64_t a = reinterpret_cast<uint64_t>(base);
        return v4u{(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a), (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)(a >> 32) & 0xFFFFu)),
                   (uint32_t)__builtin_amdgcn_readfirstlane((int)bytes), 0x00020000u};
    };
    const v4u dX = desc(p.A + (uint64_t)m0 * kbytes, min(p.M - m0, (uint32_t)BM) * kbytes);
    const v4u dW = desc(p.B + (uint64_t)n0 * kbytes, min(p.N - n0, (uint32_t)BN) * kbytes);
    uint32_t voff[L];
    const uint32_t lr = wave * RPL + lrow, piece = lpos ^ (kRowB == 128 ? (lr >> 1) & 7u : lr & 15u);  // (row = 8 * RPL * j + lr)
#pragma unroll
    for (int j = 0; j < L; ++j) voff[j] = ((j < LX ? j : j - LX) * (8 * RPL) + lr) * kbytes + piece * 16;
    const uint32_t tail_bytes = kbytes - (nchunks - 1) * kRowB;  // of the last chunk
    const bool in_tail = piece * 16 < tail_bytes;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds + wave * 1024;
    auto load = [&](int j, uint32_t chunk, uint32_t stage) {
        v4u d = j < LX ? dX : dW;
        d[2] = chunk < nchunks ? d[2] : 0u;  // chunks past the end: every lane out of range, zeros
        const uint32_t off = chunk + 1 < nchunks || in_tail ? voff[j] : kOobOffset;
        const uint32_t m0reg = lds0 + stage + j * 8192, soff = chunk * kRowB;
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(m0reg), "v"(off), "s"(d), "s"(soff)
                     : "memory", "m0");
    };

    // ---- LDS -> registers: fragment f (activation tile f, or weight tile f - WTM), step i of a wavefront: piece
    // 2 * (ks * STEPS + i) + h
    const uint32_t sw = kRowB == 128 ? (l32 >> 1) & 7u : l32 & 15u;
    const uint32_t rx = (wm * (32 * WTM) + l32) * kRowB, rw = (BM + wn * (32 * WTN) + l32) * kRowB;
    uint32_t pos[STEPS];
#pragma unroll
    for (int i = 0; i < STEPS; ++i) pos[i] = ((2 * (ks * STEPS + i) + h) ^ sw) * 16;
    v4u raw[2][P];
    v4u ex[2][P];  // [nibble parity][fragment]
    auto read = [&](int set, int f, int i, uint32_t stage) {
        raw[set][f] = *reinterpret_cast<const v4u *>(lds + stage + (f < WTM ? rx + f * 32 * kRowB : rw + (f - WTM) * 32 * kRowB) + pos[i]);
    };
    // (expanded where it stands: an MFMA is opaque to the compiler, which may otherwise leave an expansion until right before
    // the MFMA that reads it, where it would need two wait states)
    auto expand_word = [&](int par, int set, int f, int w) {
        uint32_t e = (par ? raw[set][f][w] : raw[set][f][w] << 4) & kNibbleMask;
        asm volatile("" : "+v"(e));
        ex[par][f][w] = e;
    };

    v16i accw[WTN][WTM];
#pragma unroll
    for (int t = 0; t < WTN; ++t)
#pragma unroll
        for (int b = 0; b < WTM; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r) accw[t][b][r] = 0;

    // ---- prologue
#pragma unroll
    for (int s = 0; s < NST; ++s)
#pragma unroll
        for (int j = 0; j < L; ++j) load(j, s, s * kStage);
    auto wait_stages = [&](auto allowed) {  // at most `allowed` stages of loads in flight, own LDS reads done, all wavefronts here
        constexpr int N = decltype(allowed)::value * L;
        static_assert(N <= 63, "vmcnt");
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
    };
    // the part of the tile that this wavefront finishes
    // (KS = 8: wavefronts T and up finish nothing, and fetch parameters of the last tile)
    const uint32_t mine = KS == 8 ? min(ks, (uint32_t)T - 1) : ks;
    const uint32_t wm0 = m0 + wm * (32 * WTM) + (mine >> 1) * (32 * TM), wn0 = n0 + wn * (32 * WTN) + (mine & 1u) * (32 * TN);
    // (the 256 x 256 tile stages its parameters in LDS: next to 128 accumulators the eight quads of up to five arrays do not fit
    // in registers, and spilled or not by form: 4096 x 8192 x 4096, dual scales and zero points, 124 us spilled, 104 staged)
    constexpr bool kLdsParams = LATE;
#include "duq_stream_epilogue_fetch.inc"
    if (!LATE) fetch_params();
    if constexpr (STEPS == 1) {
        // a wavefront has one step of every stage, and reads two stages ahead into its registers: the stages of this chunk
        // and the next are free to be loaded once every wavefront has read them
        wait_stages(std::integral_constant<int, NST - 2>{});
#pragma unroll
        for (int f = 0; f < P; ++f) read(0, f, 0, 0);
#pragma unroll
        for (int f = 0; f < P; ++f) read(1, f, 0, kStage);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
        for (int j = 0; j < L; ++j) load(j, NST, 0);
    } else {
        wait_stages(std::integral_constant<int, NST - 1>{});
#pragma unroll
        for (int f = 0; f < P; ++f) read(0, f, 0, 0);
#pragma unroll
        for (int f = 0; f < P; ++f) read(1, f, 1, 0);
    }
#pragma unroll
    for (int f = 0; f < P; ++f)
#pragma unroll
        for (int w = 0; w < 4; ++w) expand_word(0, 0, f, w);

    // ---- main loop (stores and MFMAs are opaque to the compiler, which counts neither: the waits are written out).  A step is H MFMAs on the even nibbles, in whose shadow the odd ones are expanded, and H on the odd
    // ones, in whose shadow the next step's even ones are expanded and the registers that leaves are read for the step
    // after it.  The first read of the next chunk is in step STEPS - 2: that is where the wavefronts wait for it.  All
    // reads of this chunk are done then (every wavefront waited for its own), and its stage takes the chunk NST further on.
    if constexpr (STEPS == 1) {
        // two chunks per turn for the two register sets; a chunk past the end is zeros
        uint32_t st1 = kStage, st2 = 2 % NST * kStage;  // stages of the next chunk and the one after it
#pragma unroll 1
        for (uint32_t c = 0; c < nchunks; c += 2) {
#pragma unroll
            for (int set = 0; set < 2; ++set) {
#pragma unroll
                for (int slot = 0; slot < 2 * H; ++slot) {
                    const int par = slot / H, q = slot % H, b = q / WTN, t = q % WTN;
                    if (slot == H) {
                        wait_stages(std::integral_constant<int, NST - 2>{});
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    asm volatile("v_mfma_i32_32x32x32_i8 %0, %1, %2, %0"
                                 : "+a"(accw[t][b])
                                 : "v"(ex[par][WTM + t]), "v"(ex[par][b]));
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int w = q * W / H; w < (q + 1) * W / H; ++w) expand_word(par ^ 1, par ? set ^ 1 : set, w / 4, w % 4);
#pragma unroll
                    for (int f = 0; f < P; ++f)
                        if (par && q == f * H / P) read(set, f, 0, st2);
#pragma unroll
                    for (int j = 0; j < L; ++j)
                        if (par && q == j * H / L) load(j, c + set + 1 + NST, st1);
                    __builtin_amdgcn_sched_barrier(0);
                }
                st1 = st2;
                st2 = st2 + kStage == NST * kStage ? 0 : st2 + kStage;
            }
        }
    } else {
        uint32_t stage = 0;
#pragma unroll 1
        for (uint32_t c = 0; c < nchunks; ++c) {
            const uint32_t next = stage + kStage == NST * kStage ? 0 : stage + kStage;
#pragma unroll
            for (int i = 0; i < STEPS; ++i) {
                const int set = i & 1;
#pragma unroll
                for (int slot = 0; slot < 2 * H; ++slot) {
                    const int par = slot / H, q = slot % H, b = q / WTN, t = q % WTN;
                    if (i == STEPS - 2 && slot == H) {
                        wait_stages(std::integral_constant<int, NST - 2>{});
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    asm volatile("v_mfma_i32_32x32x32_i8 %0, %1, %2, %0"
                                 : "+a"(accw[t][b])
                                 : "v"(ex[par][WTM + t]), "v"(ex[par][b]));
                    __builtin_amdgcn_sched_barrier(0);
                    // ---- side work in the shadow of this MFMA.  (The words expanded last belong to the last weight tile,
                    // which the MFMA behind them does not read: one that did would need two wait states first.)
#pragma unroll
                    for (int w = q * W / H; w < (q + 1) * W / H; ++w) expand_word(par ^ 1, par ? set ^ 1 : set, w / 4, w % 4);
#pragma unroll
                    for (int f = 0; f < P; ++f)
                        if (par && q == f * H / P) read(set, f, (i + 2) % STEPS, i < STEPS - 2 ? stage : next);
                    if (i >= STEPS - 2) {
#pragma unroll
                        for (int j = 0; j < L; ++j)
                            if ((i - STEPS + 2) * 2 * H + slot == H + j * 3 * H / L) load(j, c + NST, stage);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            stage = next;
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    asm volatile("s_nop 15\n\ts_nop 15\n\ts_nop 15" ::: "memory");

    v16i acc[TN][TM];
    if constexpr (KS == 1) {
#pragma unroll
        for (int t = 0; t < TN; ++t)
#pragma unroll
            for (int b = 0; b < TM; ++b) acc[t][b] = accw[t][b];
    } else if constexpr (KS == 8) {
        // tile 2 * b + t is finished by the wavefront of that number: the others add to its sums in LDS (integers, in any
        // order)
        static_assert(WTN == 2 && T <= 8, "a tile per wavefront");
        int32_t *const red = reinterpret_cast<int32_t *>(lds) + lane;
        __syncthreads();
#pragma unroll
        for (int g = 0; g < T; ++g)
            if ((uint32_t)g == ks)
#pragma unroll
                for (int r = 0; r < 16; ++r) red[(g * 16 + r) * 64] = accw[g & 1][g >> 1][r];
        __syncthreads();
#pragma unroll
        for (int g = 0; g < T; ++g)
            if ((uint32_t)g != ks)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    __hip_atomic_fetch_add(red + (g * 16 + r) * 64, accw[g & 1][g >> 1][r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[0][0][r] = red[(mine * 16 + r) * 64];
    } else {
        // the KS wavefronts of a tile share its outputs out: each hands the sums it does not finish to those that do
        auto at = [&](int dst, uint32_t src, int t, int b) {
            const uint32_t from = src > (uint32_t)dst ? src - 1 : src;  // (nobody hands itself anything)
            return reinterpret_cast<v4i *>(lds + ((((uint32_t)dst * (KS - 1) + from) * (WM * WN) + w4) * (TM * TN) + t * TM + b) * 4096) + lane;
        };
        __syncthreads();
#pragma unroll
        for (int g = 0; g < KS; ++g) {
            if ((uint32_t)g == ks) {
#pragma unroll
                for (int t = 0; t < TN; ++t)
#pragma unroll
                    for (int b = 0; b < TM; ++b) acc[t][b] = accw[(g & 1) * TN + t][(g >> 1) * TM + b];
            } else {
#pragma unroll
                for (int t = 0; t < TN; ++t)
#pragma unroll
                    for (int b = 0; b < TM; ++b)
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            v4i v;
#pragma unroll
                            for (int r = 0; r < 4; ++r) v[r] = accw[(g & 1) * TN + t][(g >> 1) * TM + b][q * 4 + r];
                            at(g, ks, t, b)[q * 64] = v;
                        }
            }
        }
        __syncthreads();
#pragma unroll
        for (int o = 1; o < KS; ++o)
#pragma unroll
            for (int t = 0; t < TN; ++t)
#pragma unroll
                for (int b = 0; b < TM; ++b)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const v4i v = at((int)ks, (ks + o) % KS, t, b)[q * 64];
#pragma unroll
                        for (int r = 0; r < 4; ++r) acc[t][b][q * 4 + r] += v[r];
                    }
    }
    if (LATE) fetch_params();
    if (KS == 8 && ks >= (uint32_t)T) p.M = 0;  // no rows of its own: stores nothing
    uint8_t *const wstage = lds + wave * (32 * TM) * (64 * TN + 16);
    constexpr bool kWideStore = false, kFloatBits = false;
#include "duq_stream_epilogue_store.inc"
}

template <int WTM, int WTN, int WM, int WN, int KS, int kRowB, int EPI, bool BIAS>
__global__ __launch_bounds__(512) void gemm_s4_prefill_kernel(DUQ_HEAD_DECL, GemmParams tail)
{
    using Tile = PrefillTile<WTM, WTN, WM, WN, KS, kRowB>;
    GemmParams p = with_head(tail, DUQ_HEAD_USE);
    to_global(p.A);
    to_global(p.B);
    to_global(p.C);
    to_global(p.y);
    __shared__ __attribute__((aligned(256))) uint8_t lds[Tile::kLds];
    __shared__ __attribute__((aligned(16))) uint32_t dpar[EPI == 5 ? (Tile::BN + Tile::BM) * 8 : 4];
    __shared__ uint32_t dwide;
    if (blockIdx.z) batch_shift(p, blockIdx.z);
    uint32_t tile_m, tile_n;
    tile_of_block(blockIdx.x, p.tiles_m, p.tiles_n, tile_m, tile_n);
    prefill_tile<Tile, EPI, BIAS>(p, lds, dpar, dwide, tile_m * Tile::BM, tile_n * Tile::BN);
}

using Tile64x128 = PrefillTile<2, 2, 1, 2, 4, 256>;
using Tile128x128 = PrefillTile<2, 2, 2, 2, 2, 256>;
using Tile192x128 = PrefillTile<3, 2, 2, 2, 2, 128>;
using Tile128x256 = PrefillTile<2, 2, 2, 4, 1, 128>;
using Tile256x256 = PrefillTile<4, 2, 2, 4, 1, 128>;

// Rounds that do not come out even: p.tiles_m x p.tiles_n tiles of 128 x 256 or 256 x 256, as many as fill whole rounds of 256
// workgroups, and behind them the columns that are left in tiles of another kind.
template <typename Tile, typename Rest, int EPI, bool BIAS>
__global__ __launch_bounds__(512) void gemm_s4_prefill_mixed_kernel(DUQ_HEAD_DECL, GemmParams tail)
{
    GemmParams p = with_head(tail, DUQ_HEAD_USE);
    to_global(p.A);
    to_global(p.B);
    to_global(p.C);
    to_global(p.y);
    __shared__ __attribute__((aligned(256))) uint8_t lds[Tile::kLds > Rest::kLds ? Tile::kLds : Rest::kLds];
    uint32_t none = 0, tile_m, tile_n;
    const uint32_t whole = p.tiles_m * p.tiles_n;
    if (blockIdx.x < whole) {
        tile_of_block(blockIdx.x, p.tiles_m, p.tiles_n, tile_m, tile_n);
        prefill_tile<Tile, EPI, BIAS>(p, lds, &none, none, tile_m * Tile::BM, tile_n * Tile::BN);
    } else {
        const uint32_t n1 = p.tiles_n * Tile::BN;
        tile_of_block(blockIdx.x - whole, (p.M + Rest::BM - 1) / Rest::BM, (p.N - n1 + Rest::BN - 1) / Rest::BN, tile_m, tile_n);
        prefill_tile<Rest, EPI, BIAS>(p, lds, &none, none, tile_m * Rest::BM, n1 + tile_n * Rest::BN);
    }
}

// Whole rounds of such tiles over the first tile.main_cols columns, the rest in other tiles behind them.
template <typename Tile, typename Rest, int EPI, bool BIAS>
static int launch_mixed(GemmParams &p, const StreamTile &tile, hipStream_t stream)
{
    p.tiles_m = (p.M + Tile::BM - 1) / Tile::BM;
    p.tiles_n = tile.main_cols / Tile::BN;
    const uint32_t rest = ((p.M + Rest::BM - 1) / Rest::BM) * ((p.N - tile.main_cols + Rest::BN - 1) / Rest::BN);
    DUQ_LAUNCH_HEAD((gemm_s4_prefill_mixed_kernel<Tile, Rest, EPI, BIAS>), dim3(p.tiles_m * p.tiles_n + rest), dim3(512), 0, stream, p);
    return (int)hipGetLastError();
}

template <typename Tile, int EPI, bool BIAS>
static int launch_mixed(GemmParams &p, const StreamTile &tile, hipStream_t stream)
{
    if constexpr (Tile::BM == 256) {
        if (tile.rest_cols == 256) return launch_mixed<Tile, Tile128x256, EPI, BIAS>(p, tile, stream);
    }
    return tile.rest_rows == 192   ? launch_mixed<Tile, Tile192x128, EPI, BIAS>(p, tile, stream)
           : tile.rest_rows == 128 ? launch_mixed<Tile, Tile128x128, EPI, BIAS>(p, tile, stream)
                                   : launch_mixed<Tile, Tile64x128, EPI, BIAS>(p, tile, stream);
}

template <int EPI, bool BIAS>
static int launch_prefill_epi(GemmParams &p, StreamTile tile, hipStream_t stream, uint32_t batch)
{
    const uint32_t bm = tile.rows, bn = tile.cols;
    if constexpr (EPI >= 0 && EPI != 5) {
        if (tile.main_cols)
            return tile.main_rows == 256 ? launch_mixed<Tile256x256, EPI, BIAS>(p, tile, stream)
                                         : launch_mixed<Tile128x256, EPI, BIAS>(p, tile, stream);
    }
    p.tiles_m = (p.M + bm - 1) / bm;
    p.tiles_n = (p.N + bn - 1) / bn;
    const dim3 grid(p.tiles_m * p.tiles_n, 1, batch);
    if (bm == 64 && bn == 64)
        DUQ_LAUNCH_HEAD((gemm_s4_prefill_kernel<2, 2, 1, 1, 8, 256, EPI, BIAS>), grid, dim3(512), 0, stream, p);
    else if (bm == 96 && bn == 64)
        DUQ_LAUNCH_HEAD((gemm_s4_prefill_kernel<3, 2, 1, 1, 8, 256, EPI, BIAS>), grid, dim3(512), 0, stream, p);
    else if (bm == 64 && bn == 128)
        DUQ_LAUNCH_HEAD((gemm_s4_prefill_kernel<2, 2, 1, 2, 4, 256, EPI, BIAS>), grid, dim3(512), 0, stream, p);
    else if (bm == 192 && bn == 128)
        DUQ_LAUNCH_HEAD((gemm_s4_prefill_kernel<3, 2, 2, 2, 2, 128, EPI, BIAS>), grid, dim3(512), 0, stream, p);
    else if (bm == 128 && bn == 128)
        DUQ_LAUNCH_HEAD((gemm_s4_prefill_kernel<2, 2, 2, 2, 2, 256, EPI, BIAS>), grid, dim3(512), 0, stream, p);
    else if (bm == 128 && bn == 256)
        DUQ_LAUNCH_HEAD((gemm_s4_prefill_kernel<2, 2, 2, 4, 1, 128, EPI, BIAS>), grid, dim3(512), 0, stream, p);
    else if constexpr (EPI != 5) {
        if (bm == 256 && bn == 256)
            DUQ_LAUNCH_HEAD((gemm_s4_prefill_kernel<4, 2, 2, 4, 1, 128, EPI, BIAS>), grid, dim3(512), 0, stream, p);
    }
    return (int)hipGetLastError();
}

int launch_prefill(GemmParams &p, StreamTile tile, bool fused, hipStream_t stream, uint32_t batch)
{
    if (!fused) return launch_prefill_epi<-1, false>(p, tile, stream, batch);
    const bool bias = p.epi.bias != nullptr;
    switch (p.epi.mode) {
#define DUQ_PREFILL(MODE)                                                                                              \
    case MODE:                                                                                                         \
        return bias ? launch_prefill_epi<MODE, true>(p, tile, stream, batch) : launch_prefill_epi<MODE, false>(p, tile, stream, batch);
        DUQ_PREFILL(0)
        DUQ_PREFILL(1)
        DUQ_PREFILL(2)
        DUQ_PREFILL(3)
        DUQ_PREFILL(4)
        DUQ_PREFILL(5)
#undef DUQ_PREFILL
    default: return (int)hipErrorInvalidValue;
    }
}

}  // namespace duq
