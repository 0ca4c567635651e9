// Host-side launchers implemented by the .hip files; the extern "C" layer in
// duq_abi.hip validates arguments and forwards here.  All return a hipError_t as int.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <algorithm>

namespace duq {

int launch_sym_quant(const uint16_t *x, const uint16_t *scale, uint32_t rows, uint32_t colsSrc, uint32_t colsDst,
                     int qmax, uint8_t *q, hipStream_t stream);
int launch_sym_dual_quant(const uint16_t *x, const uint16_t *s1, const uint16_t *s2, uint32_t rows,
                          uint32_t colsSrc, uint32_t colsDst, int qmax, uint8_t *q, hipStream_t stream);
int launch_asym_quant(const uint16_t *x, const uint16_t *scale, const uint16_t *zeros, uint32_t rows,
                      uint32_t colsSrc, uint32_t colsDst, uint8_t *q, hipStream_t stream);
int launch_asym_dual_quant(const uint16_t *x, const uint16_t *s1, const uint16_t *z1, const uint16_t *s2,
                           const uint16_t *z2, uint32_t rows, uint32_t colsSrc, uint32_t colsDst, uint8_t *q,
                           hipStream_t stream);
// bf6 != nullptr (cols % 128 == 0): also write the E3M2 shadow of the codes; q may then be nullptr.
int launch_quantize_rows_sym(const uint16_t *x, uint32_t rows, uint32_t cols, float clip, int qmax, uint8_t *q,
                             uint16_t *scale, uint8_t *bf6, hipStream_t stream);
// rowsum == nullptr: unsigned codes and zero points as the reference stores them; otherwise the
// signed-shifted form (code - 8, zero - 8) plus the per-row sum of the shifted codes.
int launch_quantize_rows_asym(const uint16_t *x, uint32_t rows, uint32_t cols, uint8_t *q, uint16_t *scale,
                              uint16_t *zeros, int32_t *rowsum, uint8_t *bf6, hipStream_t stream);
// The rows of two tensors of one width in one launch, without the shadow: codes, scales (and zero points) of x2's rows
// follow those of x's.
int launch_quantize_two(const uint16_t *x, uint32_t rows, const uint16_t *x2, uint32_t rows2, uint32_t cols, bool asym, float clip,
                        int qmax, uint8_t *q, uint16_t *scale, uint16_t *zeros, hipStream_t stream);
// A product with one row of A per problem in one launch, without packed operands: the shapes of product_row_takes.  N > 0, K > 0.
bool product_row_takes(uint32_t M, uint32_t N, uint32_t K);
int launch_product_row(bool asym, const uint16_t *a, const uint16_t *b, uint32_t batch, uint32_t N, uint32_t K, float clip_a,
                       int qmax_a, float clip_b, int qmax_b, uint16_t *y, hipStream_t stream);
// Products of short rows, K = 64, 128, 192 or 256, in the same form (duq_product.hip); eager_only: not in a recording.
bool product_tiles_takes(bool asym, uint32_t batch, uint32_t M, uint32_t N, uint32_t K);
bool product_tiles_eager_only(uint32_t batch, uint32_t M, uint32_t N, uint32_t K);
int launch_product_tiles(bool asym, const uint16_t *a, const uint16_t *b, uint32_t batch, uint32_t M, uint32_t N, uint32_t K, float clip_a,
                         int qmax_a, float clip_b, int qmax_b, uint16_t *y, hipStream_t stream);

// Products of long rows with few columns (duq_product_long.hip); q: room for the codes of B, whole tiles of 32 rows; s, z [batch, N].
bool product_long_takes(uint32_t batch, uint32_t M, uint32_t N, uint32_t K);
uint32_t product_long_reads(uint32_t N, uint32_t K);
int launch_product_long(bool asym, const uint16_t *a, const uint16_t *b, uint32_t batch, uint32_t M, uint32_t N, uint32_t K, float clip_a,
                        int qmax_a, float clip_b, int qmax_b, uint16_t *y, uint8_t *q, uint16_t *s, uint16_t *z, hipStream_t stream);

// What runs a product of activations (duq_quantize_product).  Several kernels may take a shape: the first of these that does.  *recorded: what
// runs it where the call is being recorded into a graph.
enum ProductPath { kProductRow = 1, kProductTiles, kProductLong, kProductTwoLaunches };
inline ProductPath product_path(bool asym, uint32_t batch, uint32_t M, uint32_t N, uint32_t K, ProductPath *recorded)
{
    const ProductPath separate = product_long_takes(batch, M, N, K) ? kProductLong : kProductTwoLaunches;
    const ProductPath path = product_row_takes(M, N, K)                    ? kProductRow
                             : product_tiles_takes(asym, batch, M, N, K) ? kProductTiles
                                                                         : separate;
    *recorded = path == kProductTiles && product_tiles_eager_only(batch, M, N, K) ? separate : path;
    return path;
}

// Epilogue description shared by the stand-alone dequant kernels and the fused GEMM.
// mode: 0 sym, 1 asym, 2 sym-dual, 3 asym-dual, 4 asym with row-sum zero-point correction, 5 the same for the
// dual-uniform layer (fused GEMM only, shapes of gemm_fuses_dual_rowsum) (DUQ_EPI_* of the public header).
struct Epilogue {
    int mode;
    const uint16_t *s_row;   // [rows]
    const uint16_t *z_row;   // [rows]  asym modes
    const uint16_t *s_col_1; // [cols]
    const uint16_t *z_col_1; // [cols]  asym modes
    const uint16_t *s_col_2; // [cols]  dual modes
    const uint16_t *z_col_2; // [cols]  asym-dual
    const uint16_t *bias;    // [cols] or nullptr
    const int32_t *rs_row;   // [rows]  mode 4: sum over k of the row's shifted codes
    const int32_t *rs_col;   // [cols]  mode 4: sum over k of the column's shifted codes minus K * zero (mode 5: of
                             //         input columns 0..9)
    const int32_t *rs_col_2; // [cols]  mode 5: the same over the other input columns
};

int launch_dequant(const int32_t *acc, const Epilogue &epi, uint32_t rows, uint32_t cols, uint16_t *y,
                   hipStream_t stream);
// the same over `batches` accumulator matrices [batches, rows, cols] in one launch, every batch entry with its
// own per-row [batches, rows] and per-column [batches, cols] parameters.  batches <= 65535.
int launch_dequant_batched(const int32_t *acc, const Epilogue &epi, uint32_t batches, uint32_t rows, uint32_t cols,
                           uint16_t *y, hipStream_t stream);

// Row-sum epilogue of the dual-uniform layer on int32 accumulators (definition: include/duq_hip.h,
// duq_asym_dual_rowsum_dequant_host).  xq / w are the packed operands of the GEMM that made `acc`: the kernel reads
// the first eight bytes of every row of both (the codes of input columns 0..9).
struct DualRowsumParams {
    const int32_t *acc;      // [rows, cols]
    const uint8_t *xq;       // [rows, kbytes]
    const uint8_t *w;        // [cols, kbytes]
    uint32_t kbytes;
    const uint16_t *s_row, *z_row;   // [rows]
    const int32_t *rs_row;           // [rows]
    const uint16_t *s_col_1, *z_col_1, *s_col_2, *z_col_2;  // [cols]
    const int32_t *adj_col_1, *adj_col_2;                   // [cols]
    const uint16_t *bias;            // [cols] or nullptr
    uint32_t rows, cols;
    uint16_t *y;             // [rows, cols]
};
int launch_dual_rowsum_dequant(const DualRowsumParams &p, hipStream_t stream);

// Kernels of the int4 GEMM and the host-side rule that picks one (gemm_kernel_for: host arithmetic only, exported as
// duq_gemm_kernel_for so that the rule can be tested without a GPU): takes_wide_kernel and takes_lds_kernel are asked first, what
// they leave goes by size (select_gemm_kernel, whose answers for the shapes that they take only the question of who
// asks for room for accumulators still goes by: gemm_fuses_dual_rowsum).
enum GemmKernelId {
    kKernelDecodeRows = 1,  // duq_decode.hip, v_dot8_i32_i4, M <= 4
    kKernelDecodeMfma = 2,  // duq_decode.hip, MFMA, activations in registers: 5 <= M <= 64, K <= 8192 (more than 32 rows: 4096)
    kKernelDot = 3,         // duq_gemm.hip, M <= 4 with rows longer than 16384 elements
    kKernelLds = 4,         // duq_decode.hip, both operands through LDS: 5 <= M <= 64 on up to 8192 columns, narrow problems
    kKernelSkinny = 5,      // duq_gemm.hip, 9 <= M <= 16 with 1536 or more column tiles, K <= 4096
    kKernelStream = 6,      // duq_prefill.hip (duq_gemm.hip for short rows), prefill
    kKernelTile = 7,        // the same kernels on problems of few tiles or rows too long for the others
    kKernelWide = 8,        // duq_decode.hip, 5 <= M <= 64 on more than 8192 columns, weights through LDS
};
int select_gemm_kernel(uint32_t M, uint32_t N, uint32_t K);
int gemm_kernel_for(uint32_t M, uint32_t N, uint32_t K);
// Tile of the LDS kernel in 16 x 16 units: the first of these, in the order of their time (64 x 4096 x 4096, one round of 256
// workgroups: 4.0, 4.4, 4.5, 5.2, 5.4, 5.9, 6.1, 6.8 us), whose workgroups, a column range and a group of rows each, are one
// round.  More row groups read the weights again, from their XCD's cache: 64 x 1024 x 8192 6.6 us with four row tiles each,
// 4.4 with one; 128 x 1024 x 16384 9.1 with two row tiles, 17.2 on tiles of the prefill kernel.  rows = 0: none.
struct LdsShape {
    uint32_t rows, cols;
};
inline LdsShape lds_shape(uint32_t M, uint32_t N)
{
    const LdsShape order[8] = {{1, 1}, {2, 1}, {1, 2}, {3, 1}, {2, 2}, {4, 1}, {3, 2}, {4, 2}};
    const uint64_t rows = (M + 15) / 16, cols = (N + 15) / 16;
    for (const LdsShape &t : order)
        if ((rows + t.rows - 1) / t.rows * ((cols + t.cols - 1) / t.cols) <= 256) return t;
    return rows <= 4 ? LdsShape{(uint32_t)rows, 2} : LdsShape{0, 0};
}
// Shapes of the LDS kernel (duq_decode.hip), asked next and before select_gemm_kernel.  Measured against what would run otherwise (or
// ran before it) on 2500 shapes, every weight out of the caches (a pool of 720 MB, 640 MB of other data read before each run), us:
//  - 5..64 rows: up to 4096 columns (up to 60 % less; 16 x 512 x 1024 3.1 -> 2.9, 64 x 1024 x 8192 8.1 -> 4.7, 16 x 512 x 28672 26.4
//    -> 10.3) but for up to 16 rows of 2049 to 4095 elements that begin inside a cache line, whose lines are fetched twice (5 x 1434 x
//    3136 3.2 -> 3.4, 16 x 1024 x 2624 0.92 times as fast; 3072 and 3584 1.0 - 1.06 times, 2048 and 4096 1.1 and 1.05).  Up to 8192
//    columns where the rows are many or long (64 x 5120 x 5120 11.1 -> 8.5, 16 x 8192 x 8192 10.8 -> 9.2, but 16 x 8192 x 4096 5.3 ->
//    5.6 and 24 x 8192 x 4096 6.1 -> 6.3, and where rows begin inside a cache line, 19 x 5332 x 3648 5.55 -> 5.95: the MFMA kernel
//    keeps its activations in registers over several column tiles, one fetch of them per CU).  More columns: lengths that the MFMA
//    kernel does not hold (16 x 12288 x 14336 27.1 -> 20.8, 32 x 16384 x 11008 28.0 -> 23.1; 48 x 11008 x 11008 20.1 -> 22.8).
//  - more rows while one round of its workgroups covers them (lds_shape), from 512 elements on, in its largest tile from
//    1024 elements on and up to 1024 rows (128 x 1024 x 512 4.9 -> 3.5, x 28672 33.9 -> 13.5; 200 x 2048 x 1024 6.8 -> 5.0; 128 x 4000 x
//    512 level).
//  - up to 4 rows longer than the rows kernel's 16384 (the dot kernel, one weight row per wavefront pair, or beyond 30720 a
//    prefill tile): up to 4096 columns (4 x 2606 x 28672 13.2 -> 9.6, 1 x 1024 x 40000 37.6 -> 11.6; one row of up to 30720 from 2048
//    columns on, 1 x 2600 x 28672 10.6 -> 9.3, but 1 x 1024 x 28672 7.4 -> 8.0: the dot kernel has twice the workgroups; the
//    dual-uniform row-sum epilogue, `mode5`, which that one does not have and which would be a launch more, stays here), above
//    for 3 and 4 rows (4 x 8192 x 28672 31.0 -> 22.9, but 4 x 8192 x 16448 18.4 -> 20.2) and beyond 30720 (1 x 8192 x 40000 46.6 ->
//    32.0; 1 x 8192 x 28672 22.2 against 22.6).  Behind and left: one and two rows of 16448 on 4096 columns, 0.90 and 0.93.
inline bool takes_lds_kernel(uint32_t M, uint32_t N, uint32_t K, bool mode5 = false)
{
    if (M == 0 || K == 0 || K > 65536 || (uint64_t)N * (K / 2) >= 0xFFFFFF00ull) return false;
    if (M > 64) {
        const LdsShape t = lds_shape(M, N);
        return t.rows > 0 && (t.rows * t.cols < 8 ? K >= 512 : K >= 1024 && M <= 1024);
    }
    if (M <= 4) return K > 16384 && (N <= 4096 ? M > 1 || N >= 2048 || K > 30720 || mode5 : N <= 16384 && K > (M > 2 ? 18432 : 30720));
    if (N <= 4096) return M > 16 || K <= 2048 || K >= 4096 || K % 256 == 0;
    if (N <= 8192) return M > 32 || K > 4096 || (M > 16 && (K <= 2048 || (N <= 6144 && K % 256 == 0)));
    return K > 8192 && (M <= 16 ? K <= 16384 : M <= 32 && K <= 12288);
}
// Shapes of the wide kernel (duq_decode.hip), asked first.  Measured against the MFMA kernel, us, (c) out of the caches as above, the
// others with a few copies of the weight, which decided the lines: up to 16 rows longer than 6144 elements, from 5120 on above
// 16384 columns ((c) 16 x 28672 x 5120 19.8 -> 17.5, 8 x 20000 x 8192 20.3 -> 17.7; 8 x 16384 x 6144 10.2 -> 10.8, (c) level, and up to
// 4096 elements it is level or behind, 16 x 16384 x 4096 7.8 -> 8.3); 17..32 rows of up to 4096 elements on up to 14336 columns
// ((c) 24 x 9000 x 4096 7.8 -> 7.1; 24 x 20000 x 3072 9.6 -> 10.0, (c) 10.6 -> 10.1), of more than 6144 above 16384 ((c) 32 x 28672 x 8192
// 31.0 -> 27.7; 18 x 33087 x 4160 20.6 -> 22.3, half of whose steps are padding, (c) level; of fewer columns, tiles of the prefill
// kernel, 32 x 11008 x 8192 12.3 against 12.9, (c) 15.0 against 14.0); 33 and more rows of up to 2048 elements ((c) 48 x 28672 x 1024
// 11.1 -> 10.0; longer ones 48 x 13824 x 3072 9.5 -> 10.3), from 49 on above 16384 columns ((c) 64 x 28672 x 2048 14.8 -> 12.9, 64 x
// 13824 x 2048 8.5 -> 8.6).
inline bool takes_wide_kernel(uint32_t M, uint32_t N, uint32_t K)
{
    if (M < 5 || M > 64 || N <= 8192 || K == 0 || K > 8192 || (uint64_t)N * (K / 2) >= 0xFFFFFF00ull) return false;
    if (M <= 16) return K > 6144 || (K >= 5120 && N > 16384);
    if (M <= 32) return K <= 4096 ? N <= 14336 : K > 6144 && N > 16384;
    return K <= 2048 && (M <= 48 || N > 16384);
}
// Shapes whose GEMM can apply the dual-uniform row-sum epilogue itself (mode 5): those of the decode kernels, and those
// of the stream and prefill kernels with rows longer than 256 elements (512 where output rows are not 16-byte aligned:
// there the accumulators' detour through memory, 8 bytes per output, is what a launch takes); the others run the GEMM into
// int32 and launch_dual_rowsum_dequant.
inline bool gemm_fuses_dual_rowsum(uint32_t M, uint32_t N, uint32_t K)
{
    const int kernel = select_gemm_kernel(M, N, K);
    if (kernel == kKernelDecodeRows || kernel == kKernelDecodeMfma) return true;
    return (kernel == kKernelStream || kernel == kKernelTile) && (N % 8 == 0 ? K > 256 : K >= 512);
}
// (the entry points ask callers for room for the accumulators by that rule; the LDS and wide kernels apply the epilogue
// themselves all the same)
inline bool gemm_applies_dual_rowsum(uint32_t M, uint32_t N, uint32_t K)
{
    return takes_wide_kernel(M, N, K) || takes_lds_kernel(M, N, K, true) || gemm_fuses_dual_rowsum(M, N, K);
}
// Tile for a problem gemm_kernel_for gives to the prefill kernel (duq_prefill.hip) or, `stream`, to the stream kernel's
// 64 x 128 tiles (duq_gemm.hip).  Whole rounds of 256 workgroups (one per CU) cost about f + c * (K / 256) microseconds
// each, measured per tile shape (N = 4096, one round, K = 1024 / 4096 / 16384): 64 x 128 6.6 / 11.9 / 33, 128 x 128 8.9 /
// 17.5 / 55, 128 x 256 12.5 / 30 / 100, 256 x 256 21 / 52.7 / 178 (1.3 of it once per launch); the cheapest wins.  192 x 128
// tiles (11.5 / 25.4 / 80) in one round only, where larger ones would leave CUs without any (1536 x 4096 x 4096 28.4 -> 25.4 us,
// x 16384 95 -> 80) and the walk over K is long enough for their end, stores of 64 bytes a row (2422 x 2312 x 1088 13.9 / 17.2).
// 64 x 64 and
// 96 x 64 tiles (128 rows; 65 rows) 5.9 / 8.7 / 22 and - / 10 / 22.6: in one round only, where they halve the walk over K;
// two rounds of them are behind (512 x 4096 x 4096 17 against 12.4, 96 x 28672 x 8192 38 against 34.7).  96 x 64 against the
// next best on 65..96 rows, 8200..16384 columns of 4096..8192 elements: 1 - 11 % ahead on 47 of 48 shapes, level on one (65 x
// 8200 x 4096 10.9 / 11.5, 65 x 13824 x 8192 19.3 / 21.1, 96 x 16384 x 5120 16.7 / 17.6, 96 x 11008 x 4096 11.9 / 12.1).  The
// stream kernel has the longer loop but starts and ends faster (512 x 4096 x 512 4.8 against 5.9 us, x 1024 5.8 / 6.6, x
// 2048 8.1 / 8.3, x 4096 13.3 / 11.9; 32 products of 1216 x 64 x 1216, 608 tiles: 12.8 us; 250 x 11008 x 4096, 344 tiles:
// 24.8 against 17.7 on 128 x 128: two or three of its workgroups share a CU, but a round begun takes a round's time).  The dual-uniform row-sum epilogue (`mode5`) has no 256 x 256 tile
// (its staged parameters do not fit in LDS beside the operands).
struct StreamTile {
    uint32_t rows, cols;
    bool stream;
    // main_cols > 0: binary16 outputs in tiles of main_rows x 256 up to that column and of rest_rows x rest_cols from there on;
    // rows x cols (stream) is the tile for int32 outputs, the cheapest for the whole problem (int32 outputs in 128 x 256 tiles
    // against it, us: 4160 x 3924 x 5888 114 -> 104, 897 x 8688 x 4544 60.3 -> 49.3, 2355 x 3344 x 2496 40.7 -> 32.0, 2614 x 3424 x 15360
    // 168 -> 145; of 26 shapes two behind by more than 2 %, 2048 x 6100 x 4096 56.9 -> 59.6 and 1203 x 15441 x 2176 103 -> 107)
    uint32_t main_cols = 0, rest_rows = 0, main_rows = 0, rest_cols = 0;
    float us = 0.f;  // what the model gives it
};
// Rounds that do not come out even: tiles of 128 x 256 or 256 x 256 over as many columns as fill whole rounds, and the columns
// that are left in one round of smaller tiles, 192 x 128, 128 x 128, 64 x 128 or (behind 256 x 256) 128 x 256, in the same launch
// (a launch of their own would start when the last large tile has ended).  Taken where the model above has it 4 % ahead of every uniform choice; measured, in
// turn, against uniform tiles: 2048 x 6144 x 4096 50.9 -> 46.4 us, 4000 x 8200 x 4160 150 -> 137.  One round of 256 x 256 costs
// 2.62 per 256 k where two of 128 x 256 cost 2.94 (a CU takes in a third less for the same outputs), and one end instead of two;
// against whole rounds of 128 x 256, with the quantizer, in the first 5 ms of a load: 1999 x 11008 x 4096 96.5 -> 87.1, 1188 x
// 14615 x 3136 73.5 -> 64.0, 2195 x 14547 x 4800 172 -> 149, 3806 x 4832 x 2048 52.9 -> 49.1; of 17 shapes the least 1.03, the mean 1.12.
// Rows of less than 2048 elements lose by it (1234 x 6658 x 832 0.87).  Before the rounds of 256 x 256 it and the 192 x 128 tiles
// changed fifteen of 75 shapes drawn at random (128..4096 rows, 700..20000 columns), by 1.02 to 1.34 (147 x 24961 x 14464).
inline StreamTile with_rest(StreamTile best, float best_cost, uint32_t M, uint32_t N, float nch)
{
    best.us = best_cost;
    if (nch < 8.0f) return best;
    best_cost *= 0.96f;
    const uint32_t main_rows[2] = {128, 256};
    const float main_c[2] = {1.47f, 2.62f}, main_f[2] = {5.5f, 9.5f};
    const uint32_t rm[4] = {192, 128, 64, 128}, rn[4] = {128, 128, 128, 256};
    const float c_us[4] = {1.146f, 0.76f, 0.44f, 1.47f}, f_us[4] = {7.1f, 4.3f, 3.6f, 5.5f};
    for (int i = 0; i < 2; ++i) {
        const uint32_t tm = (M + main_rows[i] - 1) / main_rows[i], rounds = (uint32_t)((uint64_t)tm * ((N + 255) / 256) / 256);
        const uint32_t cols = rounds * 256 / tm * 256;
        if (rounds == 0 || cols >= N) continue;
        for (int k = 0; k < 4; ++k) {
            if ((i == 0 && k == 3) || (uint64_t)((M + rm[k] - 1) / rm[k]) * ((N - cols + rn[k] - 1) / rn[k]) > 256) continue;
            const float cost = (float)rounds * (nch * main_c[i] + main_f[i]) + nch * c_us[k] + f_us[k];
            if (cost < best_cost) {
                best_cost = cost;
                best = StreamTile{best.rows, best.cols, best.stream, cols, rm[k], main_rows[i], rn[k], cost};
            }
        }
    }
    return best;
}
inline StreamTile select_stream_tile(uint32_t M, uint32_t N, uint32_t K, uint32_t batch, bool mode5)
{
    const float nch = (float)((K + 255) / 256);
    const uint32_t bm[7] = {64, 64, 96, 192, 128, 128, 256}, bn[7] = {128, 64, 64, 128, 128, 256, 256};
    const float c_us[7] = {0.44f, 0.2f, 0.258f, 1.146f, 0.76f, 1.47f, 2.62f}, f_us[7] = {3.6f, 5.5f, 6.1f, 7.1f, 4.3f, 5.5f, 9.5f};
    auto tiles = [&](int k) { return (uint64_t)((M + bm[k] - 1) / bm[k]) * ((N + bn[k] - 1) / bn[k]) * batch; };
    StreamTile best{64, 128, true};
    float best_cost = (float)((tiles(0) + 255) / 256) * (nch * 0.62f + 0.9f) + 1.3f;
    for (int k = 0; k < (mode5 ? 6 : 7); ++k) {
        if ((bn[k] == 64 || bm[k] == 192) && tiles(k) > 256) continue;
        if (bm[k] == 192 && nch < 8.0f) continue;
        const float cost = (float)((tiles(k) + 255) / 256) * (nch * c_us[k] + f_us[k]);
        if (cost < best_cost) {
            best_cost = cost;
            best = StreamTile{bm[k], bn[k], false};
        }
    }
    return batch == 1 && !mode5 ? with_rest(best, best_cost, M, N, nch) : best;
}
inline bool decode_uses_rows_kernel(uint32_t M) { return M <= 4; }
// MFMA decode kernel: one round of at most 256 workgroups, each with its share of the 16-column tiles.  The
// activations enter a CU once, and a workgroup has two tiles' weights in flight whatever their number; measured
// against one tile per workgroup (16 rows, K = 4096): N = 4800 4.96 against 6.54 us, N = 8192 5.67 against 6.89,
// N = 11008 7.05 against 8.78; 64 rows, N = 11008: 10.95 against 15.7.
inline uint32_t decode_tiles_per_workgroup(uint32_t ntiles) { return (ntiles + 255) / 256; }
// quantize + GEMM + dequant from binary16 activations in one launch: shapes of the rows kernel, and 5..8 rows
// of at most 4096 elements, or 8192 on at most 4096 columns (the rows kernel with eight rows, one wavefront
// quantizing each; measured against quantizer + MFMA decode kernel at 8 rows: N = K = 4096 4.7 against 6.5 us,
// N = 11008 7.2 against 9.3, N = 28672 13.0 against 16.0, N = 65536 K = 2048 18.7 against 21.5; K = 8192: N = 8192
// 15.3 against 13.0, N = 11008 21.0 against 15.0).  Two to four rows longer than 8192 elements only up to 16384
// output columns: every workgroup quantizes the rows again (4 rows: N = 28672 K = 8192 20.5 - 21.9 against 23.4 us,
// N = 32000 K = 4096 12.6 against 14.1, N = 128256 K = 4096 41.3 against 42.4, but N = 20000 K = 16384 45.2 against
// 36.3).
// 9..16 rows: while the rows together hold at most 32768 elements, 40960 on at most 4096 columns (quant_gemm_shape).
// This is the rule of the entry points that ask for no room for codes; quant_gemm_shape makes more shapes one launch, and takes
// most of these from the rows kernel.
inline bool decode_fp16in_one_launch(uint32_t M, uint32_t N, uint32_t K)
{
    const int kernel = select_gemm_kernel(M, N, K);
    if (kernel == kKernelDecodeRows) return M == 1 || N <= 16384 || K <= 8192;
    if (M > 8) return M <= 16 && K <= 4096 && M * K <= (N <= 4096 ? 40960u : 32768u) && N <= 16384 && kernel == kKernelDecodeMfma;
    return M <= 8 && (K <= 4096 || (K <= 8192 && N <= 4096)) && kernel == kKernelDecodeMfma;
}
// decode kernels (duq_decode.hip); the shape must be one select_gemm_kernel gives to them
int launch_decode_s4(const uint8_t *A, const uint8_t *B, uint32_t M, uint32_t N, uint32_t K, int32_t *out_acc,
                     const Epilogue *epi, uint16_t *y, hipStream_t stream);
// the same with binary16 activations in: the per-token quantizer runs inside the launch, SymQuantizer for the
// symmetric epilogues (scale = h(h(max|x| / 7) * clip), codes clamp(rint(h(x / scale)), -8, qmax)), AsymQuantizer for
// modes 1 and 3 (unsigned codes, as the reference stores them) and its signed-shifted form for modes 4 and 5 (codes and
// zero points minus 8, plus the per-token sums of the shifted codes); epi.s_row / z_row / rs_row are ignored.
// q_out / s_out / z_out / rs_out (optional) receive the codes, scales, zero points and sums.  Shapes of
// decode_fp16in_one_launch only.
int launch_decode_fp16in(const uint16_t *x, float clip, int qmax, const uint8_t *B, uint32_t M, uint32_t N, uint32_t K,
                         const Epilogue &epi, uint16_t *y, uint8_t *q_out, uint16_t *s_out, uint16_t *z_out,
                         int32_t *rs_out, hipStream_t stream);

// The same in workgroups that quantize the rows of their tile (duq_quant_gemm.hip): `rows` rows (8 of up to 8192 elements, 16 of 4096 or
// 32 of 1024) and `chunks` times `cols` tiles of 16 columns.  rows = 0: not a shape of that kernel.
struct QuantGemmShape {
    uint32_t rows, cols, chunks;
    bool eager_only = false;  // in a recording, where a launch costs the host nothing, two launches are level or ahead
};
// The cheapest of the tiles whose workgroups are one round of 256, by time fitted to one launch of each in a graph (base + per
// 1024 elements of a row, us; mode 0, three tiles of columns 0.5 more than one), against quantizer launch and GEMM launch: a step of
// two launches takes 8.2 us of host time and 4.7 of a graph's at least, and this kernel is 3.0 to 6.8.  Measured (N x K, graph, us):
// 128 rows 1024 x 1024 5.5 -> 3.7, 512 x 1024 x 512 6.9 -> 4.0, 1000 x 1000 x 1024 9.8 -> 6.7, 32 x 4096 x 2048 5.8 -> 4.6, 16 x 28672 x
// 2048 11.7 -> 8.0, 100 x 300 x 4096 5.5 -> 4.6, 128 x 4096 x 2048 8.0 -> 6.2.  Against the decode kernels' own quantizers: 8 x 4096 x
// 4096 5.9 -> 4.8, 8 x 12000 x 1024 7.1 -> 4.5, 4 x 8192 x 2048 5.1 -> 4.1, 3 x 4096 x 4096 4.6 -> 4.1, but 2 x 4096 x 4096 3.7 against 4.1.
// Sixteen rows of more than 2048 elements take two sets of registers one after the other, and groups of eight rows of more than 4096
// twice as many registers: level in a graph, or behind (28 x 3136 x 3136 6.65 / 6.6, 75 x 1270 x 2560 6.1 / 6.6, 36 x 604 x 7680 7.7 / 7.9), so
// that only the launch less decides (`eager_only`).  More than four chunks are behind (300 x 8000 x 512 8.7 against
// 9.4 with five, 64 x 28672 x 512 12.7 against 8.2 with four).
inline QuantGemmShape quant_gemm_shape(uint32_t M, uint32_t N, uint32_t K)
{
    QuantGemmShape best{0, 0, 0};
    if (M < 3 || M > 2048 || N == 0 || N > 65536 || K == 0 || K > 8192) return best;
    float best_us = 1e9f;
    const float k = (float)K / 1024.0f;
    auto offer = [&](uint32_t rows, uint32_t cols, uint32_t most_chunks, float us, float more_us) {
        const uint32_t groups = (M + rows - 1) / rows, tiles = (N + 16 * cols - 1) / (16 * cols);
        if (groups > 64 || groups * ((tiles + most_chunks - 1) / most_chunks) > 256) return;
        const uint32_t per = 256 / groups, chunks = (tiles + per - 1) / per;  // (at most that many workgroups a group of rows)
        if (chunks > most_chunks || (rows == 16 && cols == 1 && K > 2048 && chunks == 1)) return;  // (that tile has two buffers of weights)
        us += more_us * (float)(chunks - 1);
        if (us < best_us) {
            best_us = us;
            best = QuantGemmShape{rows, cols, chunks, (rows == 16 && K > 2048) || (K > 4096 && M > 8)};
        }
    };
    const float three[3] = {0.f, 0.12f, 0.6f};
    for (uint32_t c = 1; c <= 3; ++c) {
        if (K <= 4096) offer(8, c, 1, 3.0f + 0.45f * k + three[c - 1], 0.f);
        if (K <= 2048) offer(16, c, 1, 3.0f + 0.6f * k + three[c - 1], 0.f);
        else if (K <= 4096 && c > 1) offer(16, c, 1, 4.0f + 0.62f * k + three[c - 1], 0.f);
    }
    if (K > 4096) offer(8, 1, 1, 0.f, 0.f);
    if (K <= 2048) offer(16, 8, 1, 3.4f + 1.25f * k, 0.f);
    if (K <= 1024) offer(32, 4, 4, 3.2f + 1.6f * k, 0.9f + 1.1f * k);
    if (K > 2048 && K <= 4096) offer(16, 1, 4, 4.0f + 0.62f * k, 1.0f);
    return best;
}
// Three and four rows of more than 2048 elements: the rows kernel, which splits a row's quantization over all its wavefronts, is ahead of the
// tile where that quantization counts for more than the products, and where the tile is one of sixteen rows for a few.  Up to 4096 elements
// without row sums 4096 x 3072 3.88 / 4.12 us (rows kernel / tile, three rows, symmetric, in a graph), 4096 x 4096 3.96 / 4.37, asymmetric, four
// rows 4.37 / 4.49.  Its time over the tile's, three rows and four:
//  symmetric, 3000 columns: 4160 elements 1.02, 1.05; 5120 0.99, 1.04; 5632 0.94, 0.98; 6144 0.95, 0.98
//  asymmetric, 3000 columns: 4160 0.99, 1.02; 5120 0.97, 1.01; 5632 0.96, 0.99; 6144 0.94, 0.98; 7168 0.88, 0.92
//  row sums, 1000 columns: 5120 1.00, 1.05; 5632 0.96, 1.03; 6208 0.92, 0.97; 8192 0.93, 0.97 (four rows, 3000 columns 1.01); 13000 columns: 2560
//   0.94, 3840 0.95, 4032 1.09, 4096 0.98 (called eagerly 0.91); 12288 columns: 3072 1.14
//  dual row sums, 1500 columns: 3072 1.00, 3456 0.98, 4096 0.95 (4200 columns: 4032 1.23); 300 columns: 6208 0.96, 1.01; 3000 columns: 8192 1.05, 1.08
inline bool leaves_few_rows(uint32_t M, uint32_t N, uint32_t K, int mode)
{
    if (M > 4 || K <= 2048 || !decode_fp16in_one_launch(M, N, K)) return false;
    if (mode < 4) return K <= 4096 || M <= 3 || K > 5632;
    if (mode == 4) {
        if (K <= 4096) return N > 12288 && (K <= 3840 || K % 2048 == 0);
        return M <= 3 ? K > 5120 : K > 6144 && N <= 2048;
    }
    return K <= 4096 ? K > 3264 && N <= 4096 : M <= 3 && K > 6144 && N <= 2048;
}
// The tile of a call from binary16 rows (rows = 0: the rows kernel, or two launches).  A call that brings no room for codes is one launch in a
// recording too.
inline QuantGemmShape quant_gemm_tile(uint32_t M, uint32_t N, uint32_t K)
{
    QuantGemmShape s = quant_gemm_shape(M, N, K);
    if (decode_fp16in_one_launch(M, N, K)) s.eager_only = false;
    return s;
}
// Tiles of several chunks of columns that two launches are ahead of, for calls that bring room for the codes.  Sixteen rows of more than 2048 elements
// (not in a recording anyway), two launches / this kernel called eagerly, us: 62 x 3467 x 2368 asymmetric 0.87 of its time, 41 x 4107 x 2304 dual row
// sums 9.07 / 10.42, 64 x 3906 x 3200 symmetric 0.93.  Thirty-two rows, more than two groups of them and more than 256 elements (shorter ones have
// another kernel behind the quantizer, 651 x 2334 x 192 asymmetric 9.29 / 8.02; so have up to 64 rows, 51 x 29730 x 832 13.85 / 10.13): four chunks
// are behind where the GEMM's tiles come out even, 363 x 5035 x 576 asymmetric 9.18 / 10.33, 974 x 1824 x 640 symmetric 8.74 / 9.92, 276 x 6397 x 640 row
// sums 9.96 / 11.14, and ahead where they do not, 143 x 12886 x 960 12.15 / 10.40; the lines are fits of both, by the model of the GEMM's tiles.  The
// epilogue of the dual row sums takes this kernel twice as long: three chunks 498 x 2093 x 832 11.05 / 11.99, four 313 x 4875 x 640 10.59 / 13.90, but
// where no GEMM applies it 604 x 2231 x 448 22.68 / 11.16.
inline bool leaves_chunks(const QuantGemmShape &s, uint32_t M, uint32_t N, uint32_t K, int mode)
{
    if (s.chunks < 2 || decode_fp16in_one_launch(M, N, K)) return false;
    if (s.rows == 16) return true;
    if (s.chunks < (mode == 5 ? 3 : 4) || M <= 64 || K <= 256 || gemm_kernel_for(M, N, K) != kKernelStream ||
        (mode == 5 && !gemm_applies_dual_rowsum(M, N, K)))
        return false;
    const float us = select_stream_tile(M, N, K, 1, false).us, k = (float)K / 1024.0f;
    return us < (mode != 5 ? 2.7f : s.chunks == 3 ? 2.9f : 5.1f) + (mode != 5 ? 3.0f : 3.2f) * k;
}
// The same for an epilogue mode.
inline QuantGemmShape quant_gemm_tile(uint32_t M, uint32_t N, uint32_t K, int mode)
{
    const QuantGemmShape s = quant_gemm_tile(M, N, K);
    return leaves_few_rows(M, N, K, mode) || leaves_chunks(s, M, N, K, mode) ? QuantGemmShape{0, 0, 0} : s;
}
// q_out / s_out / z_out / rs_out as above.
int launch_quant_gemm(QuantGemmShape s, const uint16_t *x, float clip, int qmax, const uint8_t *B, uint32_t M, uint32_t N, uint32_t K,
                      const Epilogue &epi, uint16_t *y, uint8_t *q_out, uint16_t *s_out, uint16_t *z_out, int32_t *rs_out,
                      hipStream_t stream);

// measurement aid: read `bytes` (< 4 GiB) with the decode kernels' access pattern and discard them
int launch_probe_read(const void *src, uint64_t bytes, uint32_t *sink, hipStream_t stream);

// GEMM: out_acc != nullptr -> int32 accumulators [M,N]; else fused epilogue into y.
int launch_gemm_s4(const uint8_t *A, const uint8_t *B, uint32_t M, uint32_t N, uint32_t K, int32_t *out_acc,
                   const Epilogue *epi, uint16_t *y, hipStream_t stream);
// `batch` problems of one shape in one launch: A [batch, M, K/2], B [batch, N, K/2], out [batch, M, N], the
// epilogue's per-row arrays [batch, M] and per-column arrays [batch, N], all contiguous.  batch <= 65535.
int launch_gemm_s4_batched(const uint8_t *A, const uint8_t *B, uint32_t M, uint32_t N, uint32_t K, uint32_t batch,
                           int32_t *out_acc, const Epilogue *epi, uint16_t *y, hipStream_t stream);


// 6-bit float (E3M2) shadows of packed-int4 tensors and the GEMM that multiplies them
// (duq_bf6.hip).  K % 128 == 0, N % 16 == 0.
int launch_weight_shadow_bf6(const uint8_t *w, uint32_t N, uint32_t K, uint8_t *out, hipStream_t stream);
int launch_activation_shadow_bf6(const uint8_t *q, uint32_t M, uint32_t K, uint8_t *out, hipStream_t stream);
// Tiles of a launch: rows x width; cols > 0: that many columns of them, the others in tiles of `rest` rows.
struct Bf6Plan {
    uint32_t rows, width = 256, cols = 0, rest = 0;
    float us = 0.f;  // what the model gives it
};
Bf6Plan plan_bf6(uint32_t M, uint32_t N, uint32_t K, bool mode5);
// epi.mode 5 (row-sum epilogue of the dual-uniform layer) also needs the packed-int4 operands the shadows were made
// from, xq [M, K/2] and wq [N, K/2]: the first eight bytes of every row are read.
int launch_gemm_bf6(const uint8_t *X, const uint8_t *W, uint32_t M, uint32_t N, uint32_t K, const Epilogue &epi,
                    uint16_t *y, hipStream_t stream, const uint8_t *xq = nullptr, const uint8_t *wq = nullptr);
// The same product from packed operands that come without shadows (epilogue modes 0 - 4): both are made first, in `room` of
// shadows_bytes(M, N, K) bytes, 16-byte aligned.  Any N, K % 64 == 0, y at any address.
uint64_t shadows_bytes(uint32_t M, uint32_t N, uint32_t K);
bool pays_shadows(uint32_t M, uint32_t N, uint32_t K);       // by the kernels' models alone
bool shadows_are_ahead(uint32_t M, uint32_t N, uint32_t K);  // and with what these leave out
int launch_gemm_via_shadows(const uint8_t *xq, const uint8_t *w, uint32_t M, uint32_t N, uint32_t K, const Epilogue &epi, uint16_t *y,
                            uint8_t *room, hipStream_t stream);

// 8-bit asymmetric layer (duq_int8.hip): float32 activations, int8 codes, int32 accumulators, float32 results.
int launch_asym_quant8(const float *x, const float *scale, const float *zeros, uint32_t rows, uint32_t cols, int8_t *q,
                       hipStream_t stream);
int launch_quantize_rows_asym8(const float *x, uint32_t rows, uint32_t cols, int8_t *q, float *scale, float *zeros,
                               hipStream_t stream);
// up to eight rows: the same and the GEMM in one launch (duq_int8.hip)
bool quantize_gemm8_fuses(uint32_t M, uint32_t N, uint32_t K);
int launch_quantize_gemm_s8(const float *x, const int8_t *B, bool b_tiled, uint32_t M, uint32_t N, uint32_t K, const float *s_col,
                            const float *z_col, const float *bias, float *y, hipStream_t stream);
// the same in workgroups that quantize the rows of their tile (duq_quant_gemm8.hip): `rows` rows (8 of up to 4096 elements, 16 of 2048, 32
// of 1024) and `chunks` times `cols` tiles of 16 columns.  The cheapest tile whose workgroups are one round, by times fitted to
// launches of each in a graph, as quant_gemm_shape; against two launches (5.0 us of a graph at least, 8.2 of host time) or, up to
// eight rows, the decode kernel's own quantizer (N x K, tiled copy, us): 64 rows 1024 x 1024 5.1 -> 3.7, 512 x 1024 x 512 7.1 -> 4.3, 73 x
// 4359 x 896 10.0 -> 5.6, 16 x 11008 x 1024 7.9 -> 4.7, 32 x 4096 x 2048 7.2 -> 5.5, 78 x 310 x 3296 6.3 -> 5.2, 256 x 2048 x 1024 7.6 -> 5.9, 1000 x
// 1000 x 512 8.7 -> 6.4; 8 x 4096 x 4096 6.8 -> 5.6, 4 rows 6.2 -> 5.7, but two 5.67 against 5.80.
inline QuantGemmShape quant_gemm8_shape(uint32_t M, uint32_t N, uint32_t K)
{
    QuantGemmShape best{0, 0, 0};
    if (M < 3 || M > 2048 || N == 0 || N > 65536 || K == 0 || K > 4096) return best;
    float best_us = 1e9f;
    const float k = (float)K / 1024.0f;
    auto offer = [&](uint32_t rows, uint32_t cols, uint32_t most_chunks, float us) {
        const uint32_t groups = (M + rows - 1) / rows, tiles = (N + 16 * cols - 1) / (16 * cols);
        if (groups > 64 || groups * ((tiles + most_chunks - 1) / most_chunks) > 256) return;
        const uint32_t per = 256 / groups, chunks = (tiles + per - 1) / per;  // (at most that many workgroups a group of rows)
        if (chunks > most_chunks) return;
        us += 2.1f * (float)(chunks - 1);
        if (us < best_us) {
            best_us = us;
            best = QuantGemmShape{rows, cols, chunks};
        }
    };
    offer(8, 1, 1, 2.8f + 0.7f * k);
    if (K <= 2048) {
        offer(8, 2, 1, 3.4f + 0.7f * k);
        offer(8, 3, 1, 4.3f + 0.7f * k);
        offer(16, 1, 1, 2.5f + 1.2f * k);
        offer(16, 2, 1, 2.6f + 1.2f * k);
        offer(16, 3, 1, 2.7f + 1.7f * k);
    }
    if (K <= 1024) {
        offer(16, 8, 1, 3.3f + 3.4f * k);
        offer(32, 4, K <= 512 ? 2 : 1, 3.2f + 2.7f * k);
    }
    return best;
}
int launch_quant_gemm8(QuantGemmShape s, const float *x, const int8_t *B, bool b_tiled, uint32_t M, uint32_t N, uint32_t K, const float *s_col,
                       const float *z_col, const float *bias, float *y, hipStream_t stream);
int launch_dequant_hprec(const int32_t *acc, const float *s_row, const float *z_row, const float *s_col,
                         const float *z_col, const float *bias, uint32_t rows, uint32_t cols, float *x,
                         hipStream_t stream);
// C != nullptr -> int32 accumulators [M,N]; else the float32 dequant (+ bias) fused into y.
// b_tiled: B is the output of launch_weight_tile8 (fused form only).
int launch_gemm_s8(const int8_t *A, const int8_t *B, bool b_tiled, uint32_t M, uint32_t N, uint32_t K, int32_t *C,
                   const float *s_row, const float *z_row, const float *s_col, const float *z_col, const float *bias,
                   float *y, hipStream_t stream);
int launch_weight_tile8(const int8_t *w, uint32_t N, uint32_t K, int8_t *out, hipStream_t stream);
// The kernel it runs, by shape and weight layout (host arithmetic only; exported as duq_gemm8_kernel_for).
enum Gemm8KernelId {
    kKernel8Rows = 1,    // up to four rows on the weight as stored
    kKernel8Decode = 2,  // up to 64 rows of at most 4096 elements, activations in registers
    kKernel8Lds = 3,     // few rows, and more on narrow problems, through LDS
    kKernel8Skinny = 4,  // up to 32 longer rows
    kKernel8Split = 5,   // one round of 64 x 64 tiles, wavefronts side by side along K
    kKernel8Tile = 6,    // prefill tiles
};
int select_gemm8_kernel(uint32_t M, uint32_t N, uint32_t K, bool tiled);

// Weight preparation (duq_weight.hip).  kind 0: asymmetric over |w|, 1: signed-shifted, 2: symmetric with given scales s1,
// s2.  split: first column of the second range (0: one range, parameters s1, z1, r1).  cols % 8 == 0.
int launch_weight_rows(int kind, const uint16_t *w, uint32_t rows, uint32_t cols, uint32_t split, uint8_t *q, uint16_t *s1,
                       uint16_t *z1, int32_t *r1, uint16_t *s2, uint16_t *z2, int32_t *r2, int32_t *bad, hipStream_t stream);
int launch_weight_rows8(const float *w, uint32_t rows, uint32_t cols, int8_t *q, float *scale, float *zero, hipStream_t stream);

}  // namespace duq
