// Decode products for matrices of many columns (the output head, other stored products): blocks that walk runs of column
// tiles.  Part of the decode products of gemm_decode.hip; the gated product is built in gemm_decode_wide_gated.hip.
#include "gemm_decode_wide.h"

bool gd_wide_gated(const GdArgs& a, bool f32_out);

bool gd_wide_try(const GdArgs& a, int epi, bool scaled, bool f32_out) {
    // Plain rows with float32 results, the output head behind a norm kernel (several prompts in a step, a portion beside requests): with two column
    // tiles a block every block pulls X through L2 for 32 columns.  Us, what stood there / this: 151936 x 2048, 12 rows 123 / 118, 16 rows
    // 141 / 122, 21 rows 132 / 129, 32 rows 160 / 137, 48 rows 197 / 146, 64 rows 246 / 156; x 2560, 16 rows 188 / 148, 48 rows 255 / 179; x 4096, 64 rows
    // 405 / 283; 32768 x 4096, 16 rows 57.5 / 44.6.  With more than 16 column tiles a unit not where rows fill less than 0.65 of their row tiles, as the products
    // take as long for a row tile that is part empty (151936 x 2048, 9 rows 108 / 116, 11 rows 119 / 119, 17 rows 120 / 125, 20 rows 131 / 130, 22 rows
    // 138 / 131; 100352 x 2048, 11 rows 78 / 81, 19 rows 85 / 87, 21 rows 88 / 89, 24 rows 94 / 91); with fewer, there too (32768 x 2048, 9 rows 27 / 24, 17 rows
    // 29 / 27; 16384 x 2048, 9 rows 15 / 13).
    if (epi == EPI_STORE && !scaled && !a.xt && f32_out && a.N % 16 == 0 && a.K % GD_CHUNK == 0 && a.M >= GD_WIDE_MIN_ROWS && a.M <= 64) {
        if (a.N / 16 > 16 * gd_compute_units() && 20 * a.M < 13 * ((a.M + 15) / 16 * 16)) return false;
        if (a.M <= 16) return gd_launch_wide<EPI_STORE, false, float, 1, false, false>(a);
        if (a.M <= 32) return gd_launch_wide<EPI_STORE, false, float, 2, false, false>(a);
        if (a.M <= 48) return gd_launch_wide<EPI_STORE, false, float, 3, false, false>(a);
        return gd_launch_wide<EPI_STORE, false, float, 4, false, false>(a);
    }
    if (!scaled || !a.xt || a.M > 128 || a.N % 16 != 0 || a.K % GD_CHUNK != 0) return false;
    if (epi == EPI_STORE) return f32_out ? wide_rows<EPI_STORE, float, false>(a) : wide_rows<EPI_STORE, bf16_t, false>(a);
    if (epi == EPI_GATED) return gd_wide_gated(a, f32_out);
    return false;
}
