// What the kernels of the packed-int4 GEMM share: their parameter block, the nibble expansion and the store of four
// neighbouring outputs (duq_gemm.hip, duq_prefill.hip).
#pragma once
#include "duq_epilogue.h"
#include "duq_launch.h"
#include "duq_tiles.h"

namespace duq {

constexpr uint32_t kNibbleMask = 0xF0F0F0F0u;

// The first 56 bytes (through tiles_n) reach the kernels in registers (DUQ_HEAD_DECL / with_head).
struct GemmParams {
    const uint8_t *A;  // activations [M, K/2]
    const uint8_t *B;  // weights     [N, K/2]
    uint32_t M, N, K;
    uint32_t tiles_m;
    int32_t *C;        // int32 out (EPI < 0)
    uint16_t *y;       // fp16 out  (EPI >= 0)
    uint32_t tiles_n;
    uint32_t problems; // in the launch, see batch_shift
    Epilogue epi;
};
static_assert(offsetof(GemmParams, epi) == kHeadBytes, "the fields delivered in registers");

// Batched launch: problem blockIdx.z of a batch whose tensors are contiguous ([batch, M, K/2], [batch, N, K/2],
// [batch, M, N], per-row arrays [batch, M], per-column arrays [batch, N]).
__device__ __forceinline__ void batch_shift(GemmParams &p, uint32_t b)
{
    p.A += (uint64_t)b * p.M * (p.K >> 1);
    p.B += (uint64_t)b * p.N * (p.K >> 1);
    if (p.C) p.C += (uint64_t)b * p.M * p.N;
    if (p.y) p.y += (uint64_t)b * p.M * p.N;
    batch_shift(p.epi, b, p.M, p.N);
}

__device__ __forceinline__ void expand_nibbles(const v4u w, v4u &even, v4u &odd)
{
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        even[i] = (w[i] << 4) & kNibbleMask;
        odd[i] = w[i] & kNibbleMask;
    }
}


// Store four consecutive output columns of one row.
template <int EPI, bool BIAS>
__device__ __forceinline__ void store_quad(const GemmParams &p, uint32_t m, uint32_t n0, v4i acc, bool vec_ok)
{
    if (m >= p.M || n0 >= p.N) return;
    if (EPI < 0) {
        int32_t *dst = p.C + (uint64_t)m * p.N + n0;
        if (vec_ok && n0 + 3 < p.N) {
            *reinterpret_cast<v4i *>(dst) = acc;
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (n0 + r < p.N) dst[r] = acc[r];
        }
    } else {
        constexpr int MODE = EPI < 0 ? 0 : EPI;
        const RowEpi rp = load_row<MODE>(p.epi, m);
        uint16_t out[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t n = min(n0 + r, p.N - 1);
            const ColParams c = load_col<MODE, BIAS>(p.epi.s_col_1, p.epi.z_col_1, p.epi.s_col_2, p.epi.z_col_2,
                                                     p.epi.bias, n, p.epi.rs_col);
            out[r] = dequant_one<MODE, BIAS>(acc[r], rp, c);
        }
        uint16_t *dst = p.y + (uint64_t)m * p.N + n0;
        if (vec_ok && n0 + 3 < p.N) {
            *reinterpret_cast<v2u *>(dst) = v2u{(uint32_t)out[0] | ((uint32_t)out[1] << 16),
                                                (uint32_t)out[2] | ((uint32_t)out[3] << 16)};
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (n0 + r < p.N) dst[r] = out[r];
        }
    }
}

typedef int v16i __attribute__((ext_vector_type(16)));

// Prefill kernel (duq_prefill.hip) on a tile that select_stream_tile picked; `fused`: p.epi into p.y, else int32 into p.C.
int launch_prefill(GemmParams &p, StreamTile tile, bool fused, hipStream_t stream, uint32_t batch);

}  // namespace duq
