// rules.h -- the conditions by which launches and epilogues choose a path, as
// plain functions of sizes (no HIP types: the CPU tests compile them alone).
#pragma once

#include <cstdint>

namespace lbt {

// Whether a wavefront block of `tokens` tokens from tok0 and `rows` rows of an
// m x ld matrix of 32-bit values can store through 32-bit byte offsets from
// its first element, with tokens past m dropped by the end of a buffer of
// m ld values.  The block's last token may lie past m: its offset has to stay
// below 2^32 too, or it wraps round to the first tokens' values.
constexpr bool lean_offsets_fit(int64_t m, int64_t ld, int64_t tok0, int64_t tokens, int64_t rows) {
    constexpr int64_t kMax = int64_t{1} << 30;  // 4-byte values
    return m * ld < kMax && (tok0 + tokens) * ld + rows < kMax;
}

// Whether the attention of m rows from position pos0 (head_dim 128) is faster
// in 16-row tiles (attention_tile_kernel) than in the kernels of one workgroup
// or wavefront per (row, KV head, split).  A tile wavefront runs its split's
// keys one after another (12 us at 64 keys, 30 at 220), so there has to be
// enough work to keep the other kernels busy for longer: theirs goes by the
// (query head, visible key) pairs and by the workgroups, of which the more
// heads share one the longer each lasts and the cheaper a pair is.  Fitted to
// both sides at 1872 sizes (2 to 512 rows at positions 0 to 3500, 13 groupings
// of 2 to 32 heads; the line is within 0.3 us of the faster side on the other
// kernels' and 0.8 us on the tiles').  us workgroup / tile: 20 / 5 heads, 100
// rows 10.5 / 12.6, 160 rows 14.9 / 13.1, 17 rows behind 3500 24.9 / 33; 8 / 8
// heads, 160 rows 9.3 / 12.9, 17 rows behind 2000 13.3 / 18.9, 50 rows there
// 35 / 21; 4 / 4 heads, 33 rows behind 700 7.4 / 12.1.
constexpr bool attn_tiles_pay(int64_t m, int64_t pos0, int64_t nh, int64_t kvh, int64_t splits, int64_t split_keys) {
    const int64_t gh = nh / kvh;  // heads per workgroup: 1, 2 or 4, other groups head by head
    const double groups = (double)(m * splits * (gh == 1 || gh == 2 || gh == 4 ? kvh : nh));
    const double pairs = (double)nh * ((double)m * (double)pos0 + 0.5 * (double)m * (double)(m + 1));
    const double other = gh == 4   ? 5.2e-6 * pairs + 3.15e-3 * groups
                         : gh == 2 ? 11.2e-6 * pairs + 1.42e-3 * groups
                                   : 13.4e-6 * pairs + 0.86e-3 * groups;
    return other > 1.9 + 0.059 * (double)split_keys;
}

// Whether the several-row head of a matrix runs as lmhead_tile_kernel rather
// than the older several-row kernels.  Every workgroup of it first stages its
// token rows (80 KB at 8 rows of 2560 columns), so matrices of fewer than two
// 16-row tiles a CU, four at 5 to 8 rows, stay on the older ones
// (lmhead_batch_kernel, 2560 x 4000: 12 against 13 us at 2 rows, 12 against 18
// at 8; 2560 x 9000: 23 against 18 at 2, 23 against 25 at 8; 2560 x 24000 at 8:
// 40 against 30; lmhead_stream_kernel, 16 rows, 2560 x 4000: 13 against 20, x
// 8500: 25 against 26, x 12300: 31 against 28; 24 rows, x 4000: 20 against 21,
// x 8500: 37 against 31).
constexpr bool head_tiled(int64_t rows, int64_t m, int64_t cus) {
    return (rows + 15) / 16 * ((m + 15) / 16) > (m > 4 && m <= 8 ? 4 : 2) * cus;
}

// Whether a linear of m >= 2 rows without a norm is faster with the one-row
// kernel run per row (the same bits) than with the several-row kernels.  Those
// read the weights once per 8 to 16 rows but stage the rows in LDS first
// (2560 columns: 9 to 15 us before the first product), the one-row kernel
// starts at once and reads them per row, from L2 where the matrix fits.
// Estimates in us fitted to both sides at 4760 sizes (8 to 2560 columns, 16 to
// 128256 rows, 2 to 64 tokens, bf16 and int8), one-row / several-row: bf16,
// 2560 x 1000, 2 rows 7.1 / 10.8, 16 rows 9.0 / 11.5, 32 rows 13.4 / 12.1; 2560
// x 4000, 2 rows 8.9 / 12.0, 4 rows 14.2 / 12.0; int8, 2560 x 1000, 16 rows 9.1
// / 15.6; 2560 x 16000, 2 rows 15.9 / 19.6, 3 rows 22.0 / 19.5.  The one-row
// kernel has the rows in its grid's y, which ends at 65535.
constexpr bool head_row_by_row(int64_t rows, int64_t cols, int64_t m, bool q8, int64_t cus) {
    const double mb = (double)rows * (double)cols * (q8 ? 1e-6 : 2e-6);  // the weights
    const double one = (rows <= 32 ? 4.4 : 6.2) + (mb <= 5.5 ? 0.067 : 0.085) * mb * (double)m;
    const bool big = m > 8;  // 16-token groups
    const double reads = mb * (double)(big ? (m + 15) / 16 : 1);
    const double several =
        head_tiled(rows, m, cus)
            ? 5.8 + 0.0012 * (double)cols + 0.146 * reads
            : (big && q8 ? 5.3 : 4.1) + (!big ? 0.00175 : q8 ? 0.00235 : 0.00275) * (double)cols + 0.13 * reads;
    return m <= 65535 && one <= several;
}

// Whether a prefill GEMM outside the one-workgroup-per-CU kernel takes 128 x
// 128 tiles (t128 of them) rather than 64 x 64 (t64).  A round of 64 x 64 costs
// 1.6 of their MFMA tiles (half the reuse of either operand), and 128 x 128
// tiles that leave each CU at most one workgroup, one wavefront per SIMD, 4.6
// instead of 4; 5.6 with an epilogue as long as that of q/k/v or of blocks
// that straddle two matrices (2B shape, o and down at 850 tokens, 140 tiles:
// 22.5 us against 26.6 on 560 of 64 x 64; at 768, 480 of them in two rounds:
// 22.4 against 18.7; q/k/v at 768: 27.5 against 25.1, at 850: 27.8 against 29.6;
// three matrices of 1000 rows, 700 tokens: 10.7 against 8.6 at 256 columns,
// 13.3 against 12.1 at 1000, 1000 tokens and 4096 columns: 27.6 against 24.7).
constexpr bool gemm_128_tiles(int64_t t128, int64_t t64, bool long_epilogue) {
    const int64_t c64 = (t64 + 255) / 256 * 16;
    const int64_t c128 = t128 > 256 ? (t128 + 255) / 256 * 40 : long_epilogue ? 56 : 46;
    return c128 <= c64;
}

}  // namespace lbt
