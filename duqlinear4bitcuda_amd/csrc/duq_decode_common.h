// What the kernels for few rows share (duq_decode.hip, duq_quant_gemm.hip): their parameter block, the quantization step over
// several units, sums over groups of lanes, and the epilogue of one output per thread.
#pragma once
#include <cstddef>

#include "duq_epilogue.h"
#include "duq_launch.h"
#include "duq_rowquant.h"
#include "duq_tiles.h"

namespace duq {

constexpr uint32_t kNibbleMaskD = 0xF0F0F0F0u;

// The first 56 bytes (through `y`) reach the kernels in registers (DUQ_HEAD_DECL / with_head).
struct DecodeParams {
    const uint8_t *A;    // packed activations [M, K/2] (pre-quantized input)
    const uint16_t *X;   // binary16 activations [M, K] (FUSEQ)
    const uint8_t *B;    // packed weights [N, K/2]
    uint32_t M, N, K;
    uint32_t tiles_per_wg;
    int32_t *C;          // int32 out (EPI < 0)
    uint16_t *y;         // binary16 out (EPI >= 0)
    Epilogue epi;        // FUSEQ: s_row is not read, the kernel computes it
    float clip;          // FUSEQ
    int qmax;            // FUSEQ
    uint8_t *q_out;      // FUSEQ, optional: the packed codes [M, K/2] (written by workgroup 0)
    uint16_t *s_out;     // FUSEQ, optional: the per-token scales [M]
    uint16_t *z_out;     // FUSEQ with an asymmetric epilogue, optional: the per-token zero points [M]
    int32_t *rs_out;     // FUSEQ with the row-sum epilogue, optional: the per-token sums of the shifted codes [M]
};
static_assert(offsetof(DecodeParams, y) + sizeof(uint16_t *) == kHeadBytes, "the fields delivered in registers");

// The quantization step over N units, G at a time (RowQuant::quant_units: the path is chosen once per group and the
// group's chains interleave; a group holds 4 G more registers than a single unit).
template <int G, int S = 0, bool ASYM, bool UNIFORM, int N>
__device__ __forceinline__ void quant_in_groups(const RowQuant<ASYM, UNIFORM> &rq, const v4u (&raw)[N], uint32_t (&out)[N])
{
    if constexpr (S < N) {
        constexpr int L = N - S < G ? N - S : G;
        v4u in[L];
        uint32_t w[L];
#pragma unroll
        for (int j = 0; j < L; ++j) in[j] = raw[S + j];
        rq.quant_units(in, w);
#pragma unroll
        for (int j = 0; j < L; ++j) out[S + j] = w[j];
        quant_in_groups<G, S + L>(rq, raw, out);
    }
}

template <int CTRL>
__device__ __forceinline__ int dpp_add(int v)
{
    return v + __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, true);
}
// Sum over groups of G consecutive lanes (G = 2, 4, 8 or 16, inside one DPP row): every lane of a group
// ends with the group's total.
template <int G>
__device__ __forceinline__ int group_sum(int v)
{
    v = dpp_add<0xB1>(v);               // quad_perm [1,0,3,2]
    if (G >= 4) v = dpp_add<0x4E>(v);   // quad_perm [2,3,0,1]
    if (G >= 8) v = dpp_add<0x141>(v);  // row_half_mirror: lane i <- lane 7 - i
    if (G >= 16) v = dpp_add<0x140>(v); // row_mirror: lane i <- lane 15 - i
    return v;
}

__device__ __forceinline__ v4u load16(const void *p) { return *reinterpret_cast<const v4u *>(p); }

// Epilogue records of one output row / one output column, by mode: modes 0..4 the shared ColParams / RowEpi,
// mode 5 (row-sum epilogue of the dual-uniform layer) the records that also carry the codes of input columns 0..9.
template <int MODE>
struct EpiRec {
    using Col = ColParams;
    using Row = RowEpi;
};
template <>
struct EpiRec<5> {
    using Col = DualCol;
    using Row = DualRow;
};

// B / A: the packed operands (mode 5 reads the first eight bytes of the row)
template <int MODE>
__device__ __forceinline__ typename EpiRec<MODE>::Col load_col_rt(const Epilogue &e, uint32_t col, bool bias, const uint8_t *B,
                                                                  uint32_t kbytes)
{
    if constexpr (MODE == 5)
        return load_dual_col(e, B, kbytes, col, bias);
    else
        return bias ? load_col<MODE, true>(e.s_col_1, e.z_col_1, e.s_col_2, e.z_col_2, e.bias, col, e.rs_col)
                    : load_col<MODE, false>(e.s_col_1, e.z_col_1, e.s_col_2, e.z_col_2, e.bias, col, e.rs_col);
}
template <int MODE>
__device__ __forceinline__ typename EpiRec<MODE>::Row load_row_rt(const Epilogue &e, uint32_t row, const uint8_t *A, uint32_t kbytes)
{
    if constexpr (MODE == 5)
        return load_dual_row(e, A, kbytes, row);
    else
        return load_row<MODE>(e, row);
}
template <int MODE>
__device__ __forceinline__ uint16_t dequant_rt(int acc, const typename EpiRec<MODE>::Row &r, const typename EpiRec<MODE>::Col &c,
                                               bool bias)
{
    if constexpr (MODE == 5)
        return dual_finish(acc, r, c, bias);
    else
        return bias ? dequant_one<MODE, true>(acc, r, c) : dequant_one<MODE, false>(acc, r, c);
}

}  // namespace duq
