// The same int4 x int4 GEMM on the 6-bit floating point matrix path of gfx950.
//
// Every int4 value -8..7 is exactly an E3M2 ("bf6") number, every product of two of them is
// an integer of at most 7 bits, and the float32 accumulator of v_mfma_f32_16x16x128_f8f6f4
// holds every integer below 2^24 exactly.  |C| <= 64*K < 2^24 for K <= 131008 (the bound of
// the integer kernels), all partial sums are integers below 2^24 whatever the order, so the
// float32 result converted back to int32 is the integer result bit for bit.  The instruction
// runs at twice the rate of the i8 MFMA and the operands need no expansion in the loop.
//
// Operands are "shadows" of the packed-int4 tensors, made once (weights) or by the quantizer
// (activations).  A block is 32 consecutive k of one row: 32 codes x 6 bits = 24 bytes, as
// v_cvt_scalef32_pk32_bf6_f16 writes them; it is kept as a 16-byte part and an 8-byte part
// so that every load is naturally aligned.
//   activation shadow  [M][K/32 x 16 B | K/32 x 8 B]      (row-major, two planes per row)
//   weight shadow      [ceil(N/32)][K/128][3][64 lanes x 16 B]
//                      lane l of a (pair of 16-row tiles, 128-k step) holds the blocks of row l % 16,
//                      k-block l / 16 of either tile: 12 dwords [tile 2p | tile 2p+1], cut into three
//                      16-byte pieces; piece r of all lanes is one contiguous kilobyte.  Three 128-bit
//                      loads bring the two MFMA operands into twelve consecutive registers, which the
//                      kernel pins (mfma_pinned) so that the loads write them in place: three memory
//                      instructions per two fragments instead of four (a 128-bit and a 64-bit load per
//                      fragment), without a register move.  An odd last tile is paired with zeros.
// K % 128 == 0; parameter arrays as long as whole quads of columns, N % 16 == 0 where epilogue 5 reads its heads.
//
// Kernel: tile 128 (M) x 256 (N) per workgroup, 4 wavefronts side by side along N (128 x 64
// each: 8 x 4 MFMA tiles, 128 accumulator registers).  Weights go global -> registers (a ring
// of four 128-k steps), activations into LDS (three buffers of 256 k, one
// barrier per buffer) -> fragments read two MFMA groups ahead.  The weight operand is the
// MFMA "A" side, so a lane ends up with four consecutive output columns of one row.
// What bounds it is the bytes that a CU takes in, beside the MFMAs.  Loops of loads alone get 57 to 59 bytes a cycle from the L2
// in whole lines, 29 where the other half of a line is asked for later: the 80 KB of lines per 256 k of a 128-row tile (72 of
// operands; plane 1 comes in half lines) are 1410 cycles against 1024 of MFMAs, the 112 KB of a 256-row tile (96) 1980 against
// 2048.  The latter's activations used to be fetched 128 k at a time, half a
// cache line of plane 0 and a quarter of plane 1 per row, and the L2 delivers whole lines: 80.7 million of them where 44
// would do (4096 x 8192 x 28672), 176 KB per 256 k instead of 112.  Chunks of 256 k fit since they go to LDS without
// registers: 51.4 million lines, 549 -> 462 us with the quantizer (first 5 ms of a load; 491 -> 416 later), 4096 x 4096 x
// 4096 56.5 -> 50.2, 2048 x 8192 x 8192 93.5 -> 80.5.  LDS holds the pieces in swizzled order instead of padded rows: bank
// conflicts 44 -> 6 % of its cycles.  The smaller tiles are faster with their activations loaded to registers first and stored
// a body later (2048 x 4096 x 4096 31.5 against 32.6, 505 x 8960 x 4560 36.9 / 38.8): they are asked for a chunk earlier, and
// there the CU's intake is what is short.
#include <algorithm>

#include "duq_epilogue.h"
#include "duq_launch.h"
#include "duq_tiles.h"
#include <type_traits>

namespace duq {

typedef int v2i __attribute__((ext_vector_type(2)));
typedef int v6i __attribute__((ext_vector_type(6)));
typedef int v12i __attribute__((ext_vector_type(12)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v32h __attribute__((ext_vector_type(32)));

// ---------------------------------------------------------------------------------
// weight shadow
// ---------------------------------------------------------------------------------
// 32 signed nibbles (16 bytes, element 2j in the low nibble of byte j) -> one bf6 block.
// Position 8d + 2i + h of the block holds nibble i + 4h of word d (the order the quantizer
// kernels produce cheaply); both operands use it, and the sum over k does not care.
// A pair of positions (2i, 2i + 1) is one shift and one mask of the word: the nibbles' upper bits turned, they are the
// binary16 numbers 1024 + 8 + code, and a packed subtraction leaves the code.
__device__ __forceinline__ v6i bf6_block_from_nibbles(const v4u w)
{
    typedef uint32_t v16u __attribute__((ext_vector_type(16)));
    v16u f;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        const uint32_t u = w[d] ^ 0x88888888u;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            f[4 * d + i] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(v2h, ((u >> (4 * i)) & 0x000F000Fu) | 0x64006400u) - v2h{(f16)1032.0f, (f16)1032.0f});
    }
    return __builtin_bit_cast(v6i, __builtin_amdgcn_cvt_scalef32_pk32_bf6_f16(__builtin_bit_cast(v32h, f), 1.0f));
}

// Layout: for every pair of 16-row tiles and every 128-k step, 3072 bytes.  Lane l = (row l % 16, k-block l / 16) owns
// one block (24 bytes = 6 dwords) of either tile; its 12 dwords [tile 2p | tile 2p+1] are cut into three 16-byte
// pieces, and piece r of all 64 lanes forms run r (1 KB): three 128-bit loads bring two MFMA operands into twelve
// consecutive registers.  An odd last tile is paired with zeros.
__global__ __launch_bounds__(256) void weight_shadow_kernel(const uint8_t *w, uint32_t N, uint32_t K, uint8_t *out)
{
    const uint32_t ksteps = K / 128, tiles = N / 16;
    const uint64_t total = (uint64_t)((tiles + 1) / 2) * ksteps * 64;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t lane = (uint32_t)(i & 63u);
        const uint64_t ps = i >> 6;  // pair * ksteps + step
        const uint32_t step = (uint32_t)(ps % ksteps), pair = (uint32_t)(ps / ksteps);
        const uint32_t kb = step * 4 + (lane >> 4);
        v6i f[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t tile = pair * 2 + h, n = tile * 16 + (lane & 15u);
            f[h] = v6i{0, 0, 0, 0, 0, 0};
            if (tile < tiles) f[h] = bf6_block_from_nibbles(*reinterpret_cast<const v4u *>(w + (uint64_t)n * (K / 2) + kb * 16));
        }
        uint8_t *dst = out + ps * 3072 + lane * 16;
        *reinterpret_cast<v4i *>(dst) = v4i{f[0][0], f[0][1], f[0][2], f[0][3]};
        *reinterpret_cast<v4i *>(dst + 1024) = v4i{f[0][4], f[0][5], f[1][0], f[1][1]};
        *reinterpret_cast<v4i *>(dst + 2048) = v4i{f[1][2], f[1][3], f[1][4], f[1][5]};
    }
}

int launch_weight_shadow_bf6(const uint8_t *w, uint32_t N, uint32_t K, uint8_t *out, hipStream_t stream)
{
    const uint64_t total = (uint64_t)((N / 16 + 1) / 2) * (K / 128) * 64;
    if (total == 0) return 0;
    const uint32_t blocks = (uint32_t)std::min<uint64_t>((total + 255) / 256, 1u << 16);
    hipLaunchKernelGGL(weight_shadow_kernel, dim3(blocks), dim3(256), 0, stream, w, N, K, out);
    return (int)hipGetLastError();
}

// activation shadow from packed nibbles (the quantizers write it directly; this is the
// stand-alone conversion for tensors quantized elsewhere)
__global__ __launch_bounds__(256) void activation_shadow_kernel(const uint8_t *q, uint32_t M, uint32_t K, uint8_t *out)
{
    const uint32_t nblk = K / 32;
    const uint64_t total = (uint64_t)M * nblk;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t b = (uint32_t)(i % nblk);
        const uint64_t m = i / nblk;
        const v4u raw = *reinterpret_cast<const v4u *>(q + m * (K / 2) + b * 16);
        const v6i f = bf6_block_from_nibbles(raw);
        uint8_t *row = out + m * (uint64_t)nblk * 24;
        *reinterpret_cast<v4i *>(row + b * 16) = v4i{f[0], f[1], f[2], f[3]};
        *reinterpret_cast<v2i *>(row + (uint64_t)nblk * 16 + b * 8) = v2i{f[4], f[5]};
    }
}

int launch_activation_shadow_bf6(const uint8_t *q, uint32_t M, uint32_t K, uint8_t *out, hipStream_t stream)
{
    const uint64_t total = (uint64_t)M * (K / 32);
    if (total == 0) return 0;
    const uint32_t blocks = (uint32_t)std::min<uint64_t>((total + 255) / 256, 1u << 16);
    hipLaunchKernelGGL(activation_shadow_kernel, dim3(blocks), dim3(256), 0, stream, q, M, K, out);
    return (int)hipGetLastError();
}

// Shadows of both operands of one product in one launch, for a call that comes without any (launch_gemm_via_shadows): a thread a
// block of 32 codes of an activation row, or the two blocks of a lane of the weight shadow.  Columns past K (up to a multiple of 128)
// and weight rows past N are zeros.  Behind them the column parameters, padded to a multiple of 16, where the GEMM cannot read them
// in place.  Bound by memory, half a byte in and three quarters out per code: 4096 x 28672 x 8192 some 50 us at 6.7 TB/s of both.
struct ShadowsParams {
    const uint8_t *x, *w;
    uint8_t *X, *W;
    uint32_t M, N, K;
    uint32_t blocks_w, blocks_x;    // workgroups of either part; the rest copies parameters
    const uint16_t *par[5];         // s1, z1, s2, z2, bias (nullptr: not used), and the sums of epilogue 4
    const int32_t *sums;
    uint16_t *par_out;              // [5][N up to a multiple of 16], sums behind them
};

__global__ __launch_bounds__(256) void shadows_kernel(ShadowsParams p)
{
    const uint32_t ksteps = (p.K + 127) / 128, kblocks = p.K / 32, kbytes = p.K / 2;
    const v4u none = v4u{0u, 0u, 0u, 0u};
    if (blockIdx.x < p.blocks_w) {
        const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x, ps = i >> 6;  // pair * ksteps + step
        const uint32_t lane = (uint32_t)(i & 63u), step = (uint32_t)(ps % ksteps), pair = (uint32_t)(ps / ksteps);
        const uint32_t kb = step * 4 + (lane >> 4), n = pair * 32 + (lane & 15u);
        if (pair * 32 >= p.N) return;
        v4u raw[2];
#pragma unroll
        for (int h = 0; h < 2; ++h)
            raw[h] = n + 16 * h < p.N && kb < kblocks ? *reinterpret_cast<const v4u *>(p.w + (uint64_t)(n + 16 * h) * kbytes + kb * 16) : none;
        const v6i f0 = bf6_block_from_nibbles(raw[0]), f1 = bf6_block_from_nibbles(raw[1]);
        uint8_t *dst = p.W + ps * 3072 + lane * 16;
        *reinterpret_cast<v4i *>(dst) = v4i{f0[0], f0[1], f0[2], f0[3]};
        *reinterpret_cast<v4i *>(dst + 1024) = v4i{f0[4], f0[5], f1[0], f1[1]};
        *reinterpret_cast<v4i *>(dst + 2048) = v4i{f1[2], f1[3], f1[4], f1[5]};
    } else if (blockIdx.x < p.blocks_w + p.blocks_x) {
        const uint64_t i = (uint64_t)(blockIdx.x - p.blocks_w) * 256 + threadIdx.x;
        const uint32_t nblk = ksteps * 4, kb = (uint32_t)(i % nblk);
        const uint64_t m = i / nblk;
        if (m >= p.M) return;
        const v6i f = bf6_block_from_nibbles(kb < kblocks ? *reinterpret_cast<const v4u *>(p.x + m * kbytes + kb * 16) : none);
        uint8_t *row = p.X + m * nblk * 24;
        *reinterpret_cast<v4i *>(row + kb * 16) = v4i{f[0], f[1], f[2], f[3]};
        *reinterpret_cast<v2i *>(row + (uint64_t)nblk * 16 + kb * 8) = v2i{f[4], f[5]};
    } else {
        const uint32_t n = (blockIdx.x - p.blocks_w - p.blocks_x) * 256 + threadIdx.x, padded = (p.N + 15) & ~15u;
        if (n >= padded) return;
#pragma unroll
        for (int k = 0; k < 5; ++k)
            if (p.par[k]) p.par_out[k * (uint64_t)padded + n] = n < p.N ? p.par[k][n] : (uint16_t)0;
        if (p.sums) reinterpret_cast<int32_t *>(p.par_out + 5 * (uint64_t)padded)[n] = n < p.N ? p.sums[n] : 0;
    }
}

// ---------------------------------------------------------------------------------
// GEMM
// ---------------------------------------------------------------------------------

// One MFMA on half h (0: registers 0..5, 1: registers 6..11) of weight pair tuple t, which lives in the twelve
// registers v[128 + 12*t .. 139 + 12*t].  Naming the registers pins the tuple, so that the three 128-bit loads that
// fill it write them in place and the two operands are its halves: no register moves, which an opaque MFMA would
// need wait states behind (a "v" operand cannot name half of a tuple).  t and h are constants after unrolling; the
// switch folds to one statement.
#define DUQ_PIN(T, A0, A1, B0, B1)                                                                                     \
    case 2 * T:                                                                                                       \
        asm volatile("v_mfma_f32_16x16x128_f8f6f4 %0, v[" #A0 ":" #A1 "], %1, %0 cbsz:3 blgp:3"                        \
                     : "+a"(acc)                                                                                       \
                     : "v"(x), "{v[" #A0 ":" #B1 "]}"(w));                                                             \
        break;                                                                                                        \
    case 2 * T + 1:                                                                                                   \
        asm volatile("v_mfma_f32_16x16x128_f8f6f4 %0, v[" #B0 ":" #B1 "], %1, %0 cbsz:3 blgp:3"                        \
                     : "+a"(acc)                                                                                       \
                     : "v"(x), "{v[" #A0 ":" #B1 "]}"(w));                                                             \
        break;
// BASE: first register of the ring (chosen per kernel variant so that the ring ends where the variant's register
// count ends: the tuples are pinned, everything else is the compiler's).
template <int BASE>
__device__ __forceinline__ void mfma_pinned(int t, int h, v4f &acc, const v12i &w, const v6i &x)
{
    static_assert(BASE == 64 || BASE == 96 || BASE == 128 || BASE == 160, "ring base registers with a table below");
    if (BASE == 64) {  // 4 tuples (64 x 128 tiles)
        switch (2 * t + h) {
        DUQ_PIN(0, 64, 69, 70, 75)
        DUQ_PIN(1, 76, 81, 82, 87)
        DUQ_PIN(2, 88, 93, 94, 99)
        DUQ_PIN(3, 100, 105, 106, 111)
        default: __builtin_unreachable();
        }
    } else if (BASE == 96) {
        switch (2 * t + h) {
        DUQ_PIN(0, 96, 101, 102, 107)
        DUQ_PIN(1, 108, 113, 114, 119)
        DUQ_PIN(2, 120, 125, 126, 131)
        DUQ_PIN(3, 132, 137, 138, 143)
        DUQ_PIN(4, 144, 149, 150, 155)
        DUQ_PIN(5, 156, 161, 162, 167)
        DUQ_PIN(6, 168, 173, 174, 179)
        DUQ_PIN(7, 180, 185, 186, 191)
        default: __builtin_unreachable();
        }
    } else if (BASE == 128) {
        switch (2 * t + h) {
        DUQ_PIN(0, 128, 133, 134, 139)
        DUQ_PIN(1, 140, 145, 146, 151)
        DUQ_PIN(2, 152, 157, 158, 163)
        DUQ_PIN(3, 164, 169, 170, 175)
        DUQ_PIN(4, 176, 181, 182, 187)
        DUQ_PIN(5, 188, 193, 194, 199)
        DUQ_PIN(6, 200, 205, 206, 211)
        DUQ_PIN(7, 212, 217, 218, 223)
        default: __builtin_unreachable();
        }
    } else {
        switch (2 * t + h) {
        DUQ_PIN(0, 160, 165, 166, 171)
        DUQ_PIN(1, 172, 177, 178, 183)
        DUQ_PIN(2, 184, 189, 190, 195)
        DUQ_PIN(3, 196, 201, 202, 207)
        DUQ_PIN(4, 208, 213, 214, 219)
        DUQ_PIN(5, 220, 225, 226, 231)
        DUQ_PIN(6, 232, 237, 238, 243)
        DUQ_PIN(7, 244, 249, 250, 255)
        default: __builtin_unreachable();
        }
    }
}
#undef DUQ_PIN

// The first 56 bytes (through epi.mode) reach the kernel in registers (DUQ_HEAD_DECL / with_head).
struct Bf6Params {
    const uint8_t *X;  // activation shadow
    const uint8_t *W;  // weight shadow
    uint32_t M, N, K;
    uint32_t tiles_m;
    uint16_t *y;
    uint32_t tiles_n;
    Epilogue epi;
    // epilogue mode 5 only: the packed-int4 operands the shadows were made from (the first eight bytes of every row
    // are read: the codes of input columns 0..9)
    const uint8_t *xq;
    const uint8_t *wq;
};
static_assert(offsetof(Bf6Params, epi) + 8 == kHeadBytes, "the fields delivered in registers");

// TMI = 8: 128-row tiles (6: 96).  TMI = 4: 64-row tiles for problems that would leave most CUs without a 128-row tile
// (half the MFMAs for the same weight traffic, but twice the workgroups).  TMI = 16: 256-row tiles for problems
// with at least one such tile per CU: the same weight traffic feeds twice the MFMAs, which takes the kernel off
// the L2 -> CU limit that bounds the smaller tiles; all 256 AGPRs hold accumulators, its three buffers of 256 k take 144 KB
// of LDS, and the epilogue parameters are fetched after the loop.
template <int TMI, int TNI, int EPI>
struct Bf6Tile {
    static constexpr int BM = 16 * TMI, BN = 64 * TNI;
    static constexpr uint32_t kBuf = BM * 128 + (BM + 63) / 64 * 4096;  // a chunk of 256 k: BM rows of 128 bytes (plane 0), then of 64 (plane 1), in loads of 64 rows
    static constexpr uint32_t kYStride = 32 * TNI + 16;    // bytes per staged output row: 16*TNI binary16 + pad
    static constexpr uint32_t kLds = 3 * kBuf > 4 * BM * kYStride ? 3 * kBuf : 4 * BM * kYStride;
};

// The tile of rows m0 .. and columns n0 ...  lds: Bf6Tile::kLds bytes; dpar, dwide: staged parameters of EPI 5.
template <int TMI, int TNI, int EPI, bool BIAS>
__device__ __forceinline__ void bf6_tile(const Bf6Params &p, uint8_t *lds, uint32_t *dpar, uint32_t &dwide, const uint32_t m0, const uint32_t n0)
{
    static_assert(TMI == 16 || TMI == 8 || TMI == 6 || TMI == 4, "16-row MFMA tiles per wavefront along M");
    // TNI = 16 x 16 MFMA tiles per wavefront along N: BM rows x 64 columns (TNI = 4), or BM x 32 (TNI = 2, with
    // 64-row tiles only: twice the workgroups for problems that leave CUs without a 64 x 256 tile)
    static_assert(TNI == 4 || (TNI == 2 && TMI == 4), "column tiles per wavefront");
    using Tile = Bf6Tile<TMI, TNI, EPI>;
    constexpr int BM = Tile::BM, BN = Tile::BN;
    constexpr int CH = 2;                                   // 128-k steps per activation chunk
    constexpr int NXA = TMI / 2, NXB = (TMI + 3) / 4, NXP = NXA + NXB;  // activation loads per wavefront and chunk, a kilobyte each
    constexpr uint32_t kP1Base = BM * 128, kBuf = Tile::kBuf, kYStride = Tile::kYStride;
    // The 256-row tile's activations go to LDS directly, those of the others through registers (see the kernel's head).
    constexpr bool STAGED = TMI != 16;
    constexpr bool LATE_PARAMS = TMI == 16;
    constexpr int MODE = EPI;

    // dual-uniform row-sum epilogue (EPI 5): its parameters in dpar, eight words per column of the tile and per row, fetched
    // by the first BN / BM threads before the loop and read back from here after it (the records of the integer
    // kernel's epilogue, gemm_s4_stream_kernel)
    //   column: wlo, whi (first eight bytes of the packed weight row), s1 | s2 << 16, z1, z2, adj1, adj2, bias
    //   row   : xlo, xhi & 0xFF (first ten codes of the packed activation row), float(s), z, rx - rxl, rxl
    // dwide: non-zero when a factor of the corrections leaves the signed 24-bit range
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63u, wave = tid >> 6;
    const uint32_t l16 = lane & 15u, kb = lane >> 4;
    if constexpr (EPI == 5) {
        const uint32_t kbytes = p.K >> 1;
        if (tid == 0) dwide = 0;
        __syncthreads();
        bool wide = false;
        for (uint32_t i = tid; i < (uint32_t)BN; i += 256) {
            const uint32_t n = min(n0 + i, p.N - 1);
            const v2u head = *reinterpret_cast<const v2u *>(p.wq + (uint64_t)n * kbytes);
            uint32_t *d = dpar + i * 8;
            d[0] = head[0];
            d[1] = head[1];
            d[2] = (uint32_t)p.epi.s_col_1[n] | ((uint32_t)p.epi.s_col_2[n] << 16);
            d[3] = (uint32_t)rint_i32((float)bits_to_f16(p.epi.z_col_1[n]));
            d[4] = (uint32_t)rint_i32((float)bits_to_f16(p.epi.z_col_2[n]));
            d[5] = (uint32_t)p.epi.rs_col[n];
            d[6] = (uint32_t)p.epi.rs_col_2[n];
            d[7] = BIAS ? (uint32_t)p.epi.bias[n] : 0u;
            wide = wide || !(fits_i24(d[3]) && fits_i24(d[4]) && fits_i24(d[5]) && fits_i24(d[6]));
        }
        for (uint32_t i = tid; i < (uint32_t)BM; i += 256) {
            const uint32_t m = min(m0 + i, p.M - 1);
            const v2u head = *reinterpret_cast<const v2u *>(p.xq + (uint64_t)m * kbytes);
            const uint32_t xlo = head[0], xhi = head[1] & 0xFFu;  // input columns 0..7 and 8, 9
            const uint32_t rxl = dual_head_sum(xlo, xhi);
            uint32_t *d = dpar + (BN + i) * 8;
            d[0] = xlo;
            d[1] = xhi;
            d[2] = __builtin_bit_cast(uint32_t, (float)bits_to_f16(p.epi.s_row[m]));
            d[3] = (uint32_t)rint_i32((float)bits_to_f16(p.epi.z_row[m]));
            d[4] = (uint32_t)p.epi.rs_row[m] - rxl;
            d[5] = rxl;
            wide = wide || !(fits_i24(d[3]) && fits_i24(d[4]));
        }
        if (wide) dwide = 1;  // (same value from every writer)
        // (the barriers of the main loop order these writes before the epilogue's reads)
    }
    const uint32_t nblk = p.K / 32;
    const uint32_t row_bytes = nblk * 24, p1off = nblk * 16;
    const uint32_t ksteps = p.K / 128;
    const uint32_t nchunks = (ksteps + CH - 1) / CH;

    const uint32_t last_quad = ((p.N + 3) & ~3u) - 4;  // (parameter arrays are as long as whole quads of columns)
    const uint32_t wpairs = (min(p.N - n0, (uint32_t)BN) + 31) / 32;  // pairs of 16-row weight tiles in this tile
    const __amdgpu_buffer_rsrc_t rW =
        make_rsrc(p.W + (uint64_t)(n0 / 32) * ksteps * 3072, wpairs * ksteps * 3072);
    const __amdgpu_buffer_rsrc_t rNone = make_rsrc(p.X, 0);  // every read returns zero

    // weight fragments (2*pi, 2*pi + 1) of step g: 3072 bytes at ((wave*NP + pi) * ksteps + g) * 3072, three 16-byte
    // parts per lane (12 consecutive registers: two MFMA operands).  The scalar offset is not part of the hardware
    // range check: pairs past N sit in the vector offset, steps past K switch to the empty descriptor.
    constexpr int NP = TNI / 2;
    constexpr int kRingBase = TNI == 2 ? 64 : (TMI == 16 ? 160 : (TMI == 4 ? 96 : 128));
    uint32_t wv[NP];
#pragma unroll
    for (int pi = 0; pi < NP; ++pi)
        wv[pi] = wave * NP + pi < wpairs ? (wave * NP + pi) * ksteps * 3072 + lane * 16 : kOobOffset;
    // part 0..2 of the pair's twelve registers
    auto load_w = [&](v12i &dst, int pi, int part, uint32_t g, __amdgpu_buffer_rsrc_t r) {
        const v4i a = __builtin_bit_cast(
            v4i, __builtin_amdgcn_raw_buffer_load_b128(r, (int)(wv[pi] == kOobOffset ? kOobOffset : wv[pi] + part * 1024),
                                                       (int)(g * 3072), 0));
        dst[4 * part + 0] = a[0], dst[4 * part + 1] = a[1], dst[4 * part + 2] = a[2], dst[4 * part + 3] = a[3];
    };

    // activations: load j of this wavefront brings eight whole lines of plane 0 (j < NXA; rows 32 * j + 8 * wave ..) or sixteen
    // half lines of plane 1 (rows 64 * (j - NXA) + 16 * wave ..).  Lane l's 16 bytes go to 16 * l behind the load's base in LDS, so the
    // lane's source swizzles: piece q of row r lies at position q ^ ((r / 2) % 8) of the row's 128 bytes, q ^ ((r / 4) % 4) of its 64.
    const uint32_t uwave = (uint32_t)__builtin_amdgcn_readfirstlane((int)wave);
    const uint32_t xrow0 = wave * 8 + (lane >> 3), xrow1 = wave * 16 + (lane >> 2);
    const uint32_t xoff0 = xrow0 * row_bytes + ((lane & 7u) ^ ((xrow0 >> 1) & 7u)) * 16,
                   xoff1 = xrow1 * row_bytes + p1off + ((lane & 3u) ^ ((xrow1 >> 2) & 3u)) * 16;
    // (the chunk's offset is part of the vector offset, which the range check sees: with an odd number of steps the last chunk's
    // second half reads on in its row's next plane or the next row, or past the descriptor (zeros), and meets weights of zero)
    auto x_off = [&](int j, uint32_t c) {
        return j < NXA ? xoff0 + (j * 32 * row_bytes + c * 128) : xoff1 + ((j - NXA) * 64 * row_bytes + c * 64);
    };
    auto x_lds = [&](int j) { return j < NXA ? j * 4096 : kP1Base + (j - NXA) * 4096; };  // + 1024 * wave
    auto desc = [](const uint8_t *base, uint32_t bytes) {
        const uint64_t a = reinterpret_cast<uint64_t>(base);
        return v4u{(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a), (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)(a >> 32) & 0xFFFFu)),
                   (uint32_t)__builtin_amdgcn_readfirstlane((int)bytes), 0x00020000u};
    };
    const v4u dX = desc(p.X + (uint64_t)m0 * row_bytes, min(p.M - m0, (uint32_t)BM) * row_bytes);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds + uwave * 1024;
    auto chunk_desc = [&](uint32_t c) {
        v4u d = dX;
        d[2] = c < nchunks ? d[2] : 0u;  // chunks past the end: every lane out of range, zeros
        return d;
    };
    // load j of chunk c (d: chunk_desc(c)) to buffer buf
    auto load_x = [&](int j, uint32_t c, const v4u d, uint32_t buf) {
        asm volatile("s_add_u32 m0, %0, %1\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %3, 0 offen lds" ::"s"(lds0 + buf), "n"(x_lds(j)), "v"(x_off(j, c)), "s"(d)
                     : "memory", "m0", "scc");
    };
    // the same through registers: load j of chunk c, and its way to buffer buf
    v4u xreg[NXP];
    const __amdgpu_buffer_rsrc_t rX = make_rsrc(p.X + (uint64_t)m0 * row_bytes, min(p.M - m0, (uint32_t)BM) * row_bytes);
    auto fetch_x = [&](v4u &dst, int j, uint32_t c) { dst = buf_load16(c < nchunks ? rX : rNone, x_off(j, c), 0); };
    auto store_x = [&](const v4u &src, int j, uint32_t buf) { *reinterpret_cast<v4u *>(lds + buf + tid * 16 + x_lds(j)) = src; };

    // fragment of rows mi*16 + l16, k-step s of a chunk
    uint32_t frag0[CH], frag1[CH];
#pragma unroll
    for (int s = 0; s < CH; ++s) {
        frag0[s] = l16 * 128 + (((s * 4 + kb) ^ ((l16 >> 1) & 7u)) * 16);
        frag1[s] = kP1Base + l16 * 64 + (((s * 2 + (kb >> 1)) ^ ((l16 >> 2) & 3u)) * 16) + (kb & 1u) * 8;
    }

    v12i wf[4][NP];   // weight fragment pairs [ring slot][pair of column tiles], pinned to v[kRingBase + 12 * (slot * NP + pi) ..]
    v6i xf[4];        // activation fragments, ring over mi
    v4f acc[TMI][TNI];
#pragma unroll
    for (int a = 0; a < TMI; ++a)
#pragma unroll
        for (int b = 0; b < TNI; ++b) acc[a][b] = v4f{0.f, 0.f, 0.f, 0.f};

    auto read_x0 = [&](v6i &dst, uint32_t buf, int mi, int s) {
        const v4i a = *reinterpret_cast<const v4i *>(lds + buf + frag0[s] + mi * 2048);
        dst[0] = a[0], dst[1] = a[1], dst[2] = a[2], dst[3] = a[3];
    };
    auto read_x1 = [&](v6i &dst, uint32_t buf, int mi, int s) {
        const v2i b = *reinterpret_cast<const v2i *>(lds + buf + frag1[s] + mi * 1024);
        dst[4] = b[0], dst[5] = b[1];
    };

    // ---- prologue: activations of chunks 0 and 1 -> LDS (chunk 2 -> registers), weights of steps 0..2 (0..3), in the order of
    // first use, so that the wait for the activations leaves the weights of later steps in flight: all 256 workgroups start
    // together and their first ~170 KB each are bound by the L2 -> CU rate, not by latency.  (Weights of step 3: the direct
    // form's loop fetches them in its first step.)
    v4u x1[NXP];
#pragma unroll
    for (int j = 0; j < NXP; ++j)
        if constexpr (STAGED)
            fetch_x(xreg[j], j, 0);
        else
            load_x(j, 0, dX, 0);
#pragma unroll
    for (int pi = 0; pi < NP; ++pi)
#pragma unroll
        for (int part = 0; part < 3; ++part) load_w(wf[0][pi], pi, part, 0, rW);
#pragma unroll
    for (int j = 0; j < NXP; ++j)
        if constexpr (STAGED)
            fetch_x(x1[j], j, 1);
        else
            load_x(j, 1, chunk_desc(1), kBuf);
#pragma unroll
    for (int g = 1; g < (STAGED ? 4 : 3); ++g)
#pragma unroll
        for (int pi = 0; pi < NP; ++pi)
#pragma unroll
            for (int part = 0; part < 3; ++part) load_w(wf[g][pi], pi, part, g, (uint32_t)g < ksteps ? rW : rNone);
    if constexpr (STAGED) {
#pragma unroll
        for (int j = 0; j < NXP; ++j) store_x(xreg[j], j, 0);
#pragma unroll
        for (int j = 0; j < NXP; ++j) store_x(x1[j], j, kBuf);
#pragma unroll
        for (int j = 0; j < NXP; ++j) fetch_x(xreg[j], j, 2);
        lds_barrier();
    } else {
        // (counts what is certain to be issued behind chunk 0, see kBehind)
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(NXP) : "memory");
    }
#pragma unroll
    for (int mi = 0; mi < 2; ++mi) {
        read_x0(xf[mi], 0, mi, 0);
        read_x1(xf[mi], 0, mi, 0);
    }

    // ---- epilogue parameters: fetched now so that their latency hides behind the main loop (after the loop for
    // the 256-row tile, whose loop has no registers to spare)
    const Epilogue &e = p.epi;
    v2u raw_s1[TNI], raw_z1[TNI], raw_s2[TNI], raw_z2[TNI], raw_bias[TNI];
    v4i raw_rs[TNI];
    RowEpi rowp[TMI];
    auto load_params = [&]() {
        if constexpr (EPI == 5) return;  // staged in LDS above
#pragma unroll
        for (int mi = 0; mi < TMI; ++mi) rowp[mi] = load_row<MODE == 5 ? 0 : MODE>(e, min(m0 + mi * 16 + l16, p.M - 1));
#pragma unroll
        for (int ni = 0; ni < TNI; ++ni) {
            const uint32_t nq = min(n0 + wave * (16 * TNI) + ni * 16 + kb * 4, last_quad);
            raw_s1[ni] = *reinterpret_cast<const v2u *>(e.s_col_1 + nq);
            if (MODE == 1 || MODE == 3 || MODE == 4) raw_z1[ni] = *reinterpret_cast<const v2u *>(e.z_col_1 + nq);
            if (MODE == 4) raw_rs[ni] = *reinterpret_cast<const v4i *>(e.rs_col + nq);
            if (MODE >= 2 && MODE != 4) raw_s2[ni] = *reinterpret_cast<const v2u *>(e.s_col_2 + nq);
            if (MODE == 3) raw_z2[ni] = *reinterpret_cast<const v2u *>(e.z_col_2 + nq);
            if (BIAS) raw_bias[ni] = *reinterpret_cast<const v2u *>(e.bias + nq);
        }
    };
    if (!LATE_PARAMS) load_params();

    // One chunk = CH 128-k steps.  PH = position of the chunk in a turn of the weight ring: its steps use ring
    // slots CH*PH ..; a slot is refilled (with the step four ahead) during the step after its use.
    uint32_t cur = 0, nxt = kBuf, nx2 = 2 * kBuf;  // buffers of chunks c, c + 1, c + 2
    auto chunk = [&](auto ph, uint32_t c) {
        constexpr int PH = decltype(ph)::value;
        const v4u dXc = chunk_desc(c + 2);
        // Direct form: the loads that the body's barrier waits for have at least this many vector memory instructions behind them,
        // its own activation loads.  The weight loads between those are ordinary ones, which a compiler may leave out where nothing
        // reads them (after the loop it does): a wait that counted them would be too weak then.  Counting them, as the generated code
        // would allow, gains nothing: 4096 x 4096 x 1152 19.4 us either way, 4096 x 28672 x 8192 421 / 422.
        constexpr int kBehind = NXP;
        static_assert(STAGED || NXP == 6 * CH, "six activation loads in every step of a body, all in front of its barrier");
        // Side work is spread one instruction per MFMA: the loop is bound by the issue rate of its single
        // wavefront per SIMD, and a slot that holds more than about 12 cycles of other work stalls the matrix pipe.
#pragma unroll
        for (int s = 0; s < CH; ++s) {
            const int slot = CH * PH + s;
            const int prev = (slot + 3) & 3;          // slot of the step before this one
            const uint32_t gprev = CH * c + s - 1 + 4;  // the step that slot receives now
            const __amdgpu_buffer_rsrc_t rG = gprev < ksteps ? rW : rNone;
#pragma unroll
            for (int mi = 0; mi < TMI; ++mi) {
#pragma unroll
                for (int ni = 0; ni < TNI; ++ni) {
                    // The operands are written by loads only (the compiler waits for those).  A register move
                    // placed right in front of this opaque statement would need wait states the compiler
                    // cannot know of; the generated loop has none, and the bit-exact parity tests would show one.
                    mfma_pinned<kRingBase>(slot * NP + ni / 2, ni & 1, acc[mi][ni], wf[slot][ni / 2], xf[(s * TMI + mi) & 3]);
                    __builtin_amdgcn_sched_barrier(0);
                    if (!STAGED && s == CH - 1 && mi == TMI - 2 && ni == 0) {
                        // The next chunk is read from here on: its loads, issued before those of this body, have to be there.
                        // Every read of this chunk is done, so that the next body's loads may overwrite it.
                        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kBehind) : "memory");
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    // ---- side work in the shadow of this MFMA
                    if (ni < 2) {  // activation fragment two groups ahead
                        const int nm = (mi + 2) % TMI, ns = mi + 2 < TMI ? s : s + 1, nf = (s * TMI + mi + 2) & 3;  // (CH * TMI is a multiple of 4)
                        const uint32_t buf = ns < CH ? cur : nxt;
                        if (ni == 0)
                            read_x0(xf[nf], buf, nm, ns % CH);
                        else
                            read_x1(xf[nf], buf, nm, ns % CH);
                    }
                    // refill the previous step's slot: 3 * NP loads over the step
                    {
                        int widx = -1;  // which of the 3 * NP loads rides with this MFMA
                        if (TNI == 2) widx = mi < 2 ? mi * 2 + ni : -1;
                        if (TNI == 4 && (TMI == 8 || TMI == 6)) widx = ni == 2 ? mi : -1;
                        if (TNI == 4 && TMI == 4) widx = ni >= 2 ? mi * 2 + (ni - 2) : -1;
                        if (TNI == 4 && TMI == 16) widx = (ni == 2 && (mi & 1) == 0) ? mi / 2 : -1;
                        if (widx >= 0 && widx < 3 * NP) load_w(wf[prev][widx / 3], widx / 3, widx % 3, gprev, rG);
                    }
                    if constexpr (STAGED) {  // chunk c + 2 -> its buffer and, one group later, chunk c + 3 into the freed register
                        const int slot2 = TNI == 2 ? (mi - 2) * 2 + ni : ni == (TMI >= 6 ? 3 : 0) ? mi : -1, next2 = TNI == 2 ? slot2 : ni == 1 ? mi : 0;
                        if (s == 1 && slot2 >= 0 && slot2 < NXP) store_x(xreg[slot2], slot2, nx2);
                        if (s == 1 && next2 >= 1 && next2 <= NXP) fetch_x(xreg[next2 - 1], next2 - 1, c + 3);
                    } else {  // chunk c + 2 -> its buffer
                        if (ni == 2 && (mi & 1) == 1 && mi < 12) load_x(s * 6 + mi / 2, c + 2, dXc, nx2);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
        // the MFMAs are opaque to the compiler's hazard tracking: any accumulator copy it places
        // at a control-flow join must find them retired
        asm volatile("s_nop 15" ::: "memory");
        if (STAGED) lds_barrier();  // (a body's stores are for the next body but one, which begins to read them in the next)
        const uint32_t t = cur;
        cur = nxt;
        nxt = nx2;
        nx2 = t;
    };

    using P0 = std::integral_constant<int, 0>;
    using P1 = std::integral_constant<int, 1>;
    uint32_t c = 0;
    // (no branch inside the loop: a path that skips a chunk would make the compiler count only that
    // path's loads when it waits for a fragment, and drain the prefetch ring every iteration)
    for (; c + 1 < nchunks; c += 2) {
        chunk(P0{}, c);
        chunk(P1{}, c + 1);
    }
    if (c < nchunks) chunk(P0{}, c);
    // (every wavefront's loads and reads are done: the epilogue stages its outputs over the buffers)
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (LATE_PARAMS) load_params();
    // the MFMAs above are opaque to the compiler's hazard tracking: let the last ones retire
    asm volatile("s_nop 15\n\ts_nop 15\n\ts_nop 15" ::: "memory");

    // ---- epilogue: lane holds acc[mi][ni][r] = C[m = mi*16 + l16][n = ni*16 + 4*kb + r].  The
    // 128 x 64 fp16 tile of the wavefront goes through LDS so that global stores are whole
    // 128-byte lines.
    uint8_t *stage = lds + wave * (BM * kYStride);
    if constexpr (EPI == 5) {
        // every wavefront has passed the loop's last barrier: dpar is complete.  The staging area overlaps the
        // activation buffers that other wavefronts may still read in their last chunk: wait for them.
        __syncthreads();
        const bool wide = dwide != 0;
#pragma unroll
        for (int ni = 0; ni < TNI; ++ni) {
            const uint32_t ncol = ni * 16 + kb * 4;
            v4u c0[4], c1[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t *d = dpar + (wave * (16 * TNI) + ncol + r) * 8;
                c0[r] = *reinterpret_cast<const v4u *>(d);
                c1[r] = *reinterpret_cast<const v4u *>(d + 4);
            }
#pragma unroll
            for (int mi = 0; mi < TMI; ++mi) {
                const uint32_t *d = dpar + (BN + mi * 16 + l16) * 8;
                const v4u r0 = *reinterpret_cast<const v4u *>(d);
                const v2u r1 = *reinterpret_cast<const v2u *>(d + 4);
                const uint32_t s_bits = r0[2];  // (a copy: a bit cast of a vector element would read element 0)
                const float sx = __builtin_bit_cast(float, s_bits);
                uint16_t out[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float s1 = (float)bits_to_f16((uint16_t)(c0[r][2] & 0xFFFFu)), s2 = (float)bits_to_f16((uint16_t)(c0[r][2] >> 16));
                    const f16 b = bits_to_f16((uint16_t)c1[r][3]);
                    const int a = (int)acc[mi][ni][r];
                    out[r] = wide ? dual_rowsum_one<false>(a, r0[0], r0[1], r0[3], r1[1], r1[0], sx, c0[r][0], c0[r][1], s1, s2,
                                                           c0[r][3], c1[r][0], c1[r][1], c1[r][2], BIAS, b)
                                  : dual_rowsum_one<true>(a, r0[0], r0[1], r0[3], r1[1], r1[0], sx, c0[r][0], c0[r][1], s1, s2,
                                                          c0[r][3], c1[r][0], c1[r][1], c1[r][2], BIAS, b);
                }
                *reinterpret_cast<v2u *>(stage + (mi * 16 + l16) * kYStride + ncol * 2) =
                    v2u{(uint32_t)out[0] | ((uint32_t)out[1] << 16), (uint32_t)out[2] | ((uint32_t)out[3] << 16)};
            }
        }
    } else {
#pragma unroll
    for (int ni = 0; ni < TNI; ++ni) {
        const uint32_t ncol = ni * 16 + kb * 4;
        const uint32_t nq = min(n0 + wave * (16 * TNI) + ncol, last_quad);
        PairCols<MODE, BIAS> cols[2];
#pragma unroll
        for (int k = 0; k < 2; ++k)
            cols[k] = pair_cols_from_raw<MODE, BIAS>(raw_s1[ni], raw_z1[ni], raw_s2[ni], raw_z2[ni], raw_bias[ni], nq, k, raw_rs[ni]);
#pragma unroll
        for (int mi = 0; mi < TMI; ++mi) {
            *reinterpret_cast<v2u *>(stage + (mi * 16 + l16) * kYStride + ncol * 2) =
                v2u{dequant_pair<MODE, BIAS>(acc[mi][ni][0], acc[mi][ni][1], rowp[mi], cols[0]),
                    dequant_pair<MODE, BIAS>(acc[mi][ni][2], acc[mi][ni][3], rowp[mi], cols[1])};
        }
    }
    }
    const uint32_t rows_here = min(p.M - m0, (uint32_t)BM);
    const __amdgpu_buffer_rsrc_t rY = make_rsrc(p.y + (uint64_t)m0 * p.N, rows_here * p.N * 2);
    constexpr uint32_t PPR = 2 * TNI, RPI = 64 / PPR;  // 16-byte pieces per staged row, rows per store instruction
    const uint32_t piece = lane % PPR, rsub = lane / PPR;
    const uint32_t ncol0 = n0 + wave * (16 * TNI) + piece * 8;
    auto store_rows = [&](auto streamed) {
#pragma unroll
        for (int it = 0; it < BM / (int)RPI; ++it) {
            const uint32_t row = it * RPI + rsub;
            const v4u v = *reinterpret_cast<const v4u *>(stage + row * kYStride + piece * 16);
            const uint32_t off = (row < rows_here && ncol0 < p.N) ? (row * p.N + ncol0) * 2 : kOobOffset;
            __builtin_amdgcn_raw_buffer_store_b128(v, rY, (int)off, 0, decltype(streamed)::value ? 2 : 0);
        }
    };
    // (rows that are not 16-byte aligned: the same pieces at whatever alignment they have, the last one element by element)
    if (p.N % 8 != 0 || reinterpret_cast<uintptr_t>(p.y) % 16 != 0) {
        for (uint32_t row = rsub; row < rows_here; row += RPI) {
            const v4u v = *reinterpret_cast<const v4u *>(stage + row * kYStride + piece * 16);
            store_row_piece(p.y + (uint64_t)(m0 + row) * p.N + ncol0, v, p.N - min(ncol0, p.N));
        }
        return;
    }
    // (rows that begin at half lines are streamed too.  75 shapes of 17 to 110 Mi outputs, 640 to 4096 elements: 1 % ahead in the
    // geometric mean with one weight and one output, 2 % with three weights, 7 % with three of both in turn; 4096 x 28640 x 4096 267
    // against 288 us, 2000 x 28320 x 1280 27 % with three of both; the most lost 6 %, 1000 x 28320 x 640 and 3000 x 9056 x 1280)
    if (p.N % 32 == 0 || streams_outputs(p.M, p.N, 1, 100u << 20)) store_rows(std::true_type{});
    else store_rows(std::false_type{});
}

template <int TMI, int TNI, int EPI, bool BIAS>
__global__ __launch_bounds__(256) void gemm_bf6_kernel(DUQ_HEAD_DECL, Bf6Params tail)
{
    using Tile = Bf6Tile<TMI, TNI, EPI>;
    Bf6Params p = with_head(tail, DUQ_HEAD_USE);
    to_global(p.X);
    to_global(p.W);
    to_global(p.y);
    __shared__ __attribute__((aligned(16))) uint8_t lds[Tile::kLds];
    __shared__ __attribute__((aligned(16))) uint32_t dpar[EPI == 5 ? (Tile::BN + Tile::BM) * 8 : 4];
    __shared__ uint32_t dwide;
    uint32_t tile_m, tile_n;
    tile_of_block(blockIdx.x, p.tiles_m, p.tiles_n, tile_m, tile_n);
    bf6_tile<TMI, TNI, EPI, BIAS>(p, lds, dpar, dwide, tile_m * Tile::BM, tile_n * Tile::BN);
}

// Rounds that do not come out even: p.tiles_m x p.tiles_n tiles of 256 rows, as many as fill whole rounds of 256 workgroups, and
// behind them the columns that are left in tiles of REST * 16 rows (256 columns either way).
template <int REST, int EPI, bool BIAS>
__global__ __launch_bounds__(256) void gemm_bf6_mixed_kernel(DUQ_HEAD_DECL, Bf6Params tail)
{
    using Tile = Bf6Tile<16, 4, EPI>;
    using Rest = Bf6Tile<REST, 4, EPI>;
    Bf6Params p = with_head(tail, DUQ_HEAD_USE);
    to_global(p.X);
    to_global(p.W);
    to_global(p.y);
    __shared__ __attribute__((aligned(16))) uint8_t lds[Tile::kLds];
    uint32_t none = 0, tile_m, tile_n;
    const uint32_t whole = p.tiles_m * p.tiles_n;
    if (blockIdx.x < whole) {
        tile_of_block(blockIdx.x, p.tiles_m, p.tiles_n, tile_m, tile_n);
        bf6_tile<16, 4, EPI, BIAS>(p, lds, &none, none, tile_m * Tile::BM, tile_n * 256);
    } else {
        const uint32_t n1 = p.tiles_n * 256;
        tile_of_block(blockIdx.x - whole, (p.M + Rest::BM - 1) / Rest::BM, (p.N - n1 + 255) / 256, tile_m, tile_n);
        bf6_tile<REST, 4, EPI, BIAS>(p, lds, &none, none, tile_m * Rest::BM, n1 + tile_n * 256);
    }
}

template <int TMI, int TNI, int EPI>
static void launch_tile(const Bf6Params &p, hipStream_t stream)
{
    const dim3 grid(p.tiles_m * p.tiles_n);
    if (p.epi.bias)
        DUQ_LAUNCH_HEAD((gemm_bf6_kernel<TMI, TNI, EPI, true>), grid, dim3(256), 0, stream, p);
    else
        DUQ_LAUNCH_HEAD((gemm_bf6_kernel<TMI, TNI, EPI, false>), grid, dim3(256), 0, stream, p);
}

template <int REST, int EPI>
static void launch_mixed(const Bf6Params &p, hipStream_t stream)
{
    const dim3 grid(p.tiles_m * p.tiles_n + ((p.M + 16 * REST - 1) / (16 * REST)) * ((p.N + 255) / 256 - p.tiles_n));
    if (p.epi.bias)
        DUQ_LAUNCH_HEAD((gemm_bf6_mixed_kernel<REST, EPI, true>), grid, dim3(256), 0, stream, p);
    else
        DUQ_LAUNCH_HEAD((gemm_bf6_mixed_kernel<REST, EPI, false>), grid, dim3(256), 0, stream, p);
}

// Tile height: a round of 256 workgroups lasts about f + c * (K / 256) microseconds, measured (one round, K = 1024 / 4096 / 8192):
// 64 x 256 8.0 / 17.5 / 30.5, 96 x 256 9.7 / 20.2 / 35.7, 128 x 256 10.9 / 24 / 40.6, 256 x 256 18 / 38 / 65.5 (1.4 of it once per launch); the cheapest of uniform
// tiles and, where the model has them 4 % ahead, whole rounds of 256 rows with the columns that are left in one round of smaller
// tiles behind them, in the same launch (with the quantizer, first 5 ms of a load: 2048 x 11008 x 4096 70.7 -> 66.5 us, 1743 x
// 9520 x 6528 104 -> 91.6, 1000 x 22016 x 4096 68.3 -> 62.6, 1500 x 13824 x 4096 68.2 -> 62.2).  The 96-row tile is for what needs a
// round and a bit of 64-row tiles and leaves half the CUs without a 128-row one (GEMM alone: 2894 x 1536 x 3840 22.8 -> 20.1, 1957 x
// 2256 x 19968 87.5 -> 78.9, 3000 x 2048 x 2048 14.0 -> 12.4; with epilogue 5 1536 x 4096 x 4096 32.1 -> 27.8).
Bf6Plan plan_bf6(uint32_t M, uint32_t N, uint32_t K, bool mode5)
{
    const float n = (float)((K + 255) / 256);
    const uint32_t rows[4] = {64, 96, 128, 256}, tn = (N + 255) / 256;
    const float cost[4] = {n * 0.79f + 3.6f, n * 0.93f + 4.4f, n * 1.06f + 5.1f, n * 1.69f + 9.9f};
    auto tiles = [&](int k, uint32_t cols) { return (uint64_t)((M + rows[k] - 1) / rows[k]) * cols; };
    auto rounds = [](uint64_t t) { return (float)((t + 255) / 256); };
    Bf6Plan best{128};
    float least = rounds(tiles(2, tn)) * cost[2];
    const int order[3] = {0, 1, 3};
    for (int k : order) {
        if (k == 3 && mode5) continue;  // (the 256-row tile leaves no LDS for the staged parameters of epilogue 5)
        // (several rounds of short rows are their outputs, and the model's differences are small: 1410 x 10928 x 768 18.8 us with
        // 64 rows, 21.1 with 96)
        if (k == 1 && n < 6.0f && tiles(1, tn) > 256) continue;
        // (as many tiles of 96 rows as of 128, and weights beyond the last-level cache, whose rate decides: 185 x 24464 x 26496 147
        // us with 128 rows, 157 with 96, 180 x 28672 x 20480 110 / 115; but 185 x 24464 x 12800 63.8 / 49.0)
        if (k == 1 && tiles(1, tn) == tiles(2, tn) && (uint64_t)N * K * 3 / 4 > (256u << 20)) continue;
        const float c = rounds(tiles(k, tn)) * cost[k];
        if (c < least) best.rows = rows[k], least = c;
    }
    // CUs left without a 64 x 256 tile: 64 x 128 tiles, twice as many, as long as they still run in one round
    // (measured: 23-35 % faster up to 128 tiles of 64 x 256, slower from 160 on)
    if (best.rows == 64 && tiles(0, tn) <= 128) best.width = 128;
    best.us = least;
    if (mode5) return best;
    least *= 0.96f;
    // (whole rounds of 256 rows only: a round of 128-row tiles and one of 64-row tiles take longer than a round of 256-row ones;
    // not for rows so short that the outputs are most of a tile's time: 2242 x 9872 x 640 31.9 -> 33.4 us)
    const uint32_t whole = (uint32_t)(tiles(3, tn) / 256), cols = whole * 256 / ((M + 255) / 256);
    if (whole == 0 || cols >= tn || n < 6.0f) return best;
    for (int r = 0; r < 3; ++r) {
        const float c = (float)whole * cost[3] + cost[r];
        if (tiles(r, tn - cols) <= 256 && c < least) least = c, best = Bf6Plan{256, 256, cols, rows[r], c};
    }
    return best;
}

template <int EPI>
static void launch_mode(Bf6Params &p, hipStream_t stream)
{
    const Bf6Plan plan = plan_bf6(p.M, p.N, p.K, EPI == 5);
    p.tiles_m = (p.M + plan.rows - 1) / plan.rows;
    if constexpr (EPI != 5) {
        if (plan.cols) {
            p.tiles_n = plan.cols;
            if (plan.rest == 128) return launch_mixed<8, EPI>(p, stream);
            if (plan.rest == 96) return launch_mixed<6, EPI>(p, stream);
            return launch_mixed<4, EPI>(p, stream);
        }
        if (plan.rows == 256) return launch_tile<16, 4, EPI>(p, stream);
    }
    if (plan.rows == 128) return launch_tile<8, 4, EPI>(p, stream);
    if (plan.rows == 96) return launch_tile<6, 4, EPI>(p, stream);
    if (plan.width == 256) return launch_tile<4, 4, EPI>(p, stream);
    p.tiles_n = (p.N + 127) / 128;
    launch_tile<4, 2, EPI>(p, stream);
}

int launch_gemm_bf6(const uint8_t *X, const uint8_t *W, uint32_t M, uint32_t N, uint32_t K, const Epilogue &epi,
                    uint16_t *y, hipStream_t stream, const uint8_t *xq, const uint8_t *wq)
{
    if (M == 0 || N == 0) return 0;
    Bf6Params p{X, W, M, N, K, (M + 127) / 128, y, (N + 255) / 256, epi, xq, wq};
    switch (epi.mode) {
    case 0: launch_mode<0>(p, stream); break;
    case 1: launch_mode<1>(p, stream); break;
    case 2: launch_mode<2>(p, stream); break;
    case 3: launch_mode<3>(p, stream); break;
    case 4: launch_mode<4>(p, stream); break;
    case 5:
        if (!xq || !wq) return (int)hipErrorInvalidValue;
        launch_mode<5>(p, stream);
        break;
    default: return (int)hipErrorInvalidValue;
    }
    return (int)hipGetLastError();
}

static uint64_t up256(uint64_t bytes) { return (bytes + 255) & ~(uint64_t)255; }
static uint32_t padded_k(uint32_t K) { return (K + 127) & ~127u; }

// [activation shadow | weight shadow | parameters], each from a multiple of 256 bytes on
uint64_t shadows_bytes(uint32_t M, uint32_t N, uint32_t K)
{
    const uint64_t row = padded_k(K) / 4 * 3;
    return up256(M * row) + up256((N + 31ull) / 32 * 32 * row) + (N + 15ull) / 16 * 16 * 14;
}

// Whether a product that comes without shadows is faster by the 6-bit float kernel with the time to make them, by the two kernels'
// models.  Up to 1024 rows the pass takes what the kernel gains (1024 x 11008 x 4096 42.1 us integer, 28.6 and 11 of the pass).  Integer / by
// shadows, us: 4096 x 28672 x 8192 662 / 493, 1999 x 11008 x 4096 76 / 68, 3072 x 4096 x 4096 49.6 / 40.4, 3679 x 3712 x 10240 110.7 / 87.0, 1827 x
// 7352 x 13824 142 / 119; of 70 shapes (700..4096 rows, 256..28672 columns, 512..28672 elements) the 18 that it takes are 1.16 times as
// fast in the geometric mean and 1.03 at least, of those that it leaves five would be 1.05 to 1.13 times as fast (3181 x 2959 x 23872
// 198 / 176), 2048 x 4096 x 4096 31.6 / 32.9.
bool pays_shadows(uint32_t M, uint32_t N, uint32_t K)
{
    if (M <= 1024 || K < 512 || (uint64_t)M * N < (1u << 22)) return false;
    const float pass = 2.0f + 1.25f * (float)(((double)M + N) * K * 1.7e-7);
    return plan_bf6(M, N, K, false).us + pass < 0.96f * select_stream_tile(M, N, K, 1, false).us;
}

// That rule's 0.96 holds for rows of 2600 elements and more, and for weights that the last-level cache holds beside the rest: on shorter rows the
// 6-bit float kernel's model leaves out more of its end than the integer kernel's (measured over model 1.19 against 1.07 at 800 to 1800
// elements), and a larger shadow comes from memory a second time.  Integer / by shadows, us: 3285 x 5068 x 1152 36.6 / 48.2, 2671 x 3584 x 1664 22.9 /
// 29.1, 2304 x 14616 x 640 48.6 / 60.5, 2238 x 21032 x 576 53.2 / 56.2, 1489 x 25479 x 11840 325 / 373, 1253 x 23636 x 16448 348 / 410, but 5652 x 14176 x 1664
// 167 / 130, 1663 x 10675 x 1728 53 / 42, 3882 x 21744 x 14784 931 / 688.  Of 580 shapes that the rule above takes 97 were behind by more than 2 %, by
// this one 5 of the 394 that it leaves, 1.16 times as fast in the geometric mean (the most lost 2034 x 39106 x 6976 432 / 473); of those
// that it gives back the most would have been 3130 x 26112 x 704 111 / 89.
bool shadows_are_ahead(uint32_t M, uint32_t N, uint32_t K)
{
    if (!pays_shadows(M, N, K)) return false;
    float margin = 1.04f;
    if (K < 2600) margin += 0.12f * std::min(1.0f, (float)(2600 - K) / 1000.0f);
    if ((uint64_t)N * K > 200000000ull) margin = std::max(margin, 1.12f);
    const float pass = 2.0f + 1.25f * (float)(((double)M + N) * K * 1.7e-7);
    return (plan_bf6(M, N, K, false).us + pass) * margin < select_stream_tile(M, N, K, 1, false).us;
}

int launch_gemm_via_shadows(const uint8_t *xq, const uint8_t *w, uint32_t M, uint32_t N, uint32_t K, const Epilogue &epi, uint16_t *y,
                            uint8_t *room, hipStream_t stream)
{
    if (M == 0 || N == 0 || K == 0) return (int)hipErrorInvalidValue;
    const uint32_t kpad = padded_k(K), npad = (N + 15) & ~15u;
    ShadowsParams s{};
    s.x = xq;
    s.w = w;
    s.X = room;
    s.W = room + up256((uint64_t)M * (kpad / 4 * 3));
    s.M = M;
    s.N = N;
    s.K = K;
    s.par_out = reinterpret_cast<uint16_t *>(s.W + up256((N + 31ull) / 32 * 32 * (kpad / 4 * 3)));
    const uint64_t bw = ((N + 31ull) / 32 * (kpad / 128) * 64 + 255) / 256, bx = ((uint64_t)M * (kpad / 32) + 255) / 256;
    s.blocks_w = (uint32_t)bw;
    s.blocks_x = (uint32_t)bx;
    Epilogue e = epi;
    // (the GEMM reads four columns' parameters at a time)
    auto in_place = [](const void *p, uintptr_t to) { return reinterpret_cast<uintptr_t>(p) % to == 0; };
    uint32_t bp = 0;
    if (N % 16 != 0 || !in_place(e.s_col_1, 8) || !in_place(e.z_col_1, 8) || !in_place(e.s_col_2, 8) || !in_place(e.z_col_2, 8) ||
        !in_place(e.bias, 8) || !in_place(e.rs_col, 16)) {
        const uint16_t **const at[5] = {&e.s_col_1, &e.z_col_1, &e.s_col_2, &e.z_col_2, &e.bias};
        for (int k = 0; k < 5; ++k) {
            s.par[k] = *at[k];
            if (*at[k]) *at[k] = s.par_out + (uint64_t)k * npad;
        }
        s.sums = e.rs_col;
        if (e.rs_col) e.rs_col = reinterpret_cast<int32_t *>(s.par_out + 5ull * npad);
        bp = (npad + 255) / 256;
    }
    if (bw + bx + bp > 0x7FFFFFFFull) return (int)hipErrorInvalidValue;
    hipLaunchKernelGGL(shadows_kernel, dim3((uint32_t)(bw + bx) + bp), dim3(256), 0, stream, s);
    if (const int st = (int)hipGetLastError()) return st;
    return launch_gemm_bf6(s.X, s.W, M, N, kpad, e, y, stream);
}

}  // namespace duq
