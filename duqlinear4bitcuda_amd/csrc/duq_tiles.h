// Helpers shared by the GEMM kernels: workgroup -> tile mapping for the eight XCDs and raw
// buffer descriptors (out-of-range reads return zero without a branch).
#pragma once
#include "duq_device.h"

namespace duq {

// Workgroup id -> tile id.  Consecutive workgroup ids land on consecutive XCDs (8 of them,
// each with its own L2), so ids are regrouped to give every XCD one contiguous range of
// tiles; tiles inside a range walk down a band of 8 tile-rows first, which keeps the A and
// B panels an XCD touches compact.
__device__ __forceinline__ void tile_of_block(uint32_t bid, uint32_t tiles_m, uint32_t tiles_n, uint32_t &tm,
                                              uint32_t &tn)
{
    const uint32_t ntiles = tiles_m * tiles_n;
    const uint32_t per = ntiles / 8, rem = ntiles % 8;
    const uint32_t xcd = bid % 8, local = bid / 8;
    const uint32_t logical = xcd < rem ? xcd * (per + 1) + local : rem * (per + 1) + (xcd - rem) * per + local;
    constexpr uint32_t GM = 8;
    const uint32_t per_band = GM * tiles_n;
    const uint32_t band = logical / per_band;
    const uint32_t first_m = band * GM;
    const uint32_t band_h = min(tiles_m - first_m, GM);
    const uint32_t in_band = logical % per_band;
    tm = first_m + in_band % band_h;
    tn = in_band / band_h;
}

constexpr uint32_t kOobOffset = 0xFFFFFF00u;  // beyond any descriptor: the load returns 0

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void *base, uint32_t bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ v4u buf_load16(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff)
{
    return __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff, (int)soff, 0));
}
// The same with a cache policy (2 = non-temporal: for bytes that are read once, in whole cache lines).
template <int AUX>
__device__ __forceinline__ v4u buf_load16_aux(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff)
{
    return __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff, (int)soff, AUX));
}

// Eight neighbouring outputs (`left` of them inside the row) to a place of any alignment.
__device__ __forceinline__ void store_row_piece(uint16_t *dst, const v4u v, uint32_t left)
{
    typedef v4u v4u_any __attribute__((aligned(2)));
    if (left >= 8) {
        *reinterpret_cast<v4u_any *>(dst) = v;
    } else {
#pragma unroll
        for (int r = 0; r < 8; ++r)
            if ((uint32_t)r < left) dst[r] = (uint16_t)((r & 1) ? (v[r >> 1] >> 16) : (v[r >> 1] & 0xFFFFu));
    }
}

// Workgroup barrier that waits for this wavefront's LDS traffic only.  __syncthreads() also
// drains the vector memory counter, which would wait for loads requested ahead
// (a full memory latency) and for stores on their way.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Binary16 outputs of prefill-sized launches (rows of y 16-byte aligned): stored past the L2 (non-temporal) or into it.  What fits
// in the eight L2s, 32 MB, is still there when the last workgroup ends and would be written back only then, and rows that are whole
// cache lines leave as whole lines either way: streamed (integer kernel 2048 x 4096 x 4096 30.5 us against 31.5, 2048 x 4096 x 1024
// 12.6 / 14.0, 2461 x 28288 x 768 75.6 / 77.2; 6-bit floats 23.8 / 25.6, 10.3 / 12.0, 62.6 / 66.2).  Larger outputs of other widths:
// the pieces of a line that come from different workgroups meet in the L2, if they stop there (integer kernel 2461 x 28336 x 768 92.2
// -> 78.4, 4078 x 13360 x 832 91.7 -> 82.2, 1999 x 11024 x 4096 80.0 -> 74.0; 6-bit floats 80.3 -> 67.8, 61.6 -> 53.9, 59.2 -> 56.2).  The output
// is that of all problems of a launch (8 of 2000 x 2008 x 512 43.3 -> 35.1, 16 of 1000 x 1992 x 640 48.2 -> 39.6, 32 of 1000 x 1000 x 1024 51.6
// -> 43.9, 8 of 2048 x 2056 x 2048 83.1 -> 80.9; the least 5 of 2000 x 2008 x 512 23.0 -> 23.4).
__host__ __device__ __forceinline__ bool few_or_whole_lines(uint32_t M, uint32_t N, uint32_t problems = 1)
{
    return N % 64 == 0 || (uint64_t)M * N * problems <= (16u << 20);
}
// And streamed again above `most` outputs, where the last-level cache (256 MB) does not hold them beside what else is in it.  Past the L2 /
// into it, us, into one output and into four in turn.  One problem, integer kernel: 4608 x 25072 x 1024 145 / 128 and 144 / 139, 8192 x
// 16400 x 1024 172 / 170 and 169 / 194, 8192 x 28688 x 1024 284 / 328 and 280 / 328.  6-bit floats: 3600 x 28656 x 1024 123 / 113 and 121 / 120,
// 4608 x 25072 x 1024 130 / 131 and 129 / 133, 8192 x 28688 x 1024 256 / 308 and 253 / 309.  Batches of small problems: 16 of 2000 x 2008 x 512
// 70 / 59 and 69 / 70, 24 of them 96 / 84 and 97 / 110, 32 128 / 148 and 124 / 147; 64 of 1000 x 1000 x 1024 97 / 87 and 99 / 98, 96 136 / 138
// and 136 / 141 (the most lost below the line: 200 of 500 x 504 x 640 83 / 84 and 82 / 90); of large ones 4 of 4090 x 4104 x 2048 158 / 142 and
// 156 / 147, 6 of 4090 x 4104 x 512 107 / 91 and 107 / 110.
__device__ __forceinline__ bool streams_outputs(uint32_t M, uint32_t N, uint32_t problems, uint32_t most)
{
    return few_or_whole_lines(M, N, problems) || (uint64_t)M * N * problems > most;
}

// Products of short rows (K up to 256), whose instructions store 512 bytes of a row, two parts of cache lines at most.  Batches: into the L2 only
// where rows do not begin at half lines and are of 192 elements at most.  Asymmetric, past the L2 / into it, us: 32 x 2000 x
// 1992 x 64 74.7 / 42.4, x 128 73.2 / 50.0, x 192 70.9 / 58.6, x 256 65.3 / 76.4; 32 x 2000 x 2016 x 128 48.8 / 52.1; the
// largest loss 10 x 4000 x 4040 x 192 89 / 93.
// One problem: past it only where rows of more than 128 elements begin at half lines, or the outputs of rows of more than 192
// are larger than the last-level cache (8192 x 28704 x 256 108 / 151, x 192 91 / 129, x 128 94 / 107, but 8192 x 14368 x 128 47 / 42; 8192 x
// 28680 x 256 152 / 169, but x 192 136 / 131 and 8192 x 14344 x 256 71 / 66; 8192 x 10248 x 128 49 / 29).
__host__ __device__ __forceinline__ bool streams_short_rows(uint32_t M, uint32_t N, uint32_t K, uint32_t problems)
{
    const bool past = problems > 1   ? N % 32 == 0 || K > 192
                      : N % 32 == 0 ? K > 128
                                    : K > 192 && (uint64_t)M * N > (128u << 20);
    return past || few_or_whole_lines(M, N, problems);
}

// Stages of the LDS kernels (duq_decode.hip, duq_int8.hip): MT row tiles and NT column tiles of 16 per workgroup of eight
// wavefronts.
template <int MT, int NT>
struct LdsTile {
    static constexpr int G = NT == 1 ? 1 : 8;            // wavefronts that share a stage
    static constexpr int RB = G == 1 ? 128 : 512;        // bytes of a row in it
    static constexpr int DEPTH = G == 1 ? 2 : 3;         // stages
    static constexpr int U = RB / (64 * G);              // a wavefront's 64-byte fragments of a row in a stage
    static constexpr int L = (MT + NT) * U;              // load instructions of a wavefront and stage, a kilobyte each
    static constexpr int kStage = G * L * 1024, kLds = 8 / G * DEPTH * kStage, kPart = NT * MT * 8 * 1024;
    static_assert(kLds <= 160 * 1024 && kPart <= kLds, "LDS");
};

}  // namespace duq
