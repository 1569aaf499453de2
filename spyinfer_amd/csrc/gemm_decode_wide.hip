// Decode products for matrices of many columns (the output head, other stored products): blocks that walk runs of column
// tiles.  Part of the decode products of gemm_decode.hip; the gated product is built in gemm_decode_wide_gated.hip.
#include "gemm_decode_wide.h"

bool gd_wide_gated(const GdArgs& a, bool f32_out);

bool gd_wide_try(const GdArgs& a, int epi, bool scaled, bool f32_out) {
    // Plain rows with float32 results, the output head behind a norm kernel (several prompts in a step, a portion beside requests): with two column
    // tiles a block every block pulls X through L2 for 32 columns.  Us, what stood there / this: 151936 x 2048, 12 rows 123 / 118, 16 rows
    // 141 / 122, 21 rows 132 / 129, 32 rows 160 / 137, 48 rows 197 / 146, 64 rows 246 / 156; x 2560, 16 rows 188 / 148, 48 rows 255 / 179; x 4096, 64 rows
    // 405 / 283; 32768 x 4096, 16 rows 57.5 / 44.6.  Not at the lower end of one and two row tiles with many columns (9 rows 108 / 116, 17 rows
    // 120 / 125); with up to 16 column tiles a unit, there too (32768 x 2048, 9 rows 26.4 / 24.1, 17 rows 27.9 / 27.1).
    if (epi == EPI_STORE && !scaled && !a.xt && f32_out && a.N % 16 == 0 && a.K % GD_CHUNK == 0 && a.M >= GD_WIDE_MIN_ROWS && a.M <= 64) {
        if (a.N / 16 > 16 * gd_compute_units() && (a.M < 11 || a.M == 17 || a.M == 18)) return false;
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
