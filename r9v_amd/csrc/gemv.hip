/*
 * gemv.hip -- the decode GEMV's dispatch: how a launch's rows are cut into lanes
 * and K segments (r9vx_gemv.h has the kernels).
 */
#include "r9vx_gemv.h"

/* Lanes per row of `cpr` 16-byte chunks: 64, or the power of two at or above the
 * row's chunks when they are fewer than 33; lanes past the row's end idle.  A row
 * is then read in one wave-wide piece per segment whatever K is: with the largest
 * power of two that divides the row's chunks instead, K = 1792 or 6144 took 7 or 3
 * segments in series, one load latency each (Q4_K m = 6, n = 832, K = 6144: 9.8
 * us; K = 1792 gated, n = 1792, m = 1: 10.6).
 *
 * From enough weight rows to fill the SIMDs the latency is hidden, and what idle
 * lanes cost is their share of the dots: there a wave takes more rows of fewer
 * lanes, the most that idle on no more than a fifth.  A row of one segment keeps
 * its wave longer (its x is shared through LDS), and without a gate always; so
 * does a row of f32 activations up to K = 4096 (two chunks a lane at m = 1, 2:
 * IQ4_XS n = 16384, K = 2304, m = 2 13.3 / 21.4).  The line follows n, K and the
 * types alone, so that a row has the same bits in every bucket.
 * Us at 64 lanes / at fewer (in braces), and with the power of two that divides:
 *   n = 16384, K = 2304 {16}: Q4_K m = 1 9.1 / 9.5, 14.8; m = 8 31.1 / 29.7, 33.0
 *   n = 40000, K = 2304 {16}: Q8_0 m = 8 94 / 66, 59; K = 768 {8}: 29.4 / 17.8, 17.8 (IQ3_S)
 *   gated, n = 6000, K = 2304 {16}: Q4_K m = 1 9.0 / 8.3, 12.1; m = 8 34.2 / 24.1, 27.2
 *   gated, n = 16384, K = 4352 {32}: Q8_0 m = 1 37.0 / 33.4, 45.7; m = 8 117 / 84, 88 */
static uint32_t row_lanes(uint32_t cpr, uint32_t n, bool gated, bool xf32) {
    uint32_t lpr = 64;
    while (lpr > 8 && lpr / 2 >= cpr) lpr >>= 1;
    const uint64_t simds = 4u * r9vx_device_cus();
    const uint64_t line = cpr <= 32 ? (gated ? 24 : 32) * simds : cpr > 64 ? (gated ? 5 : 16) * simds : gated ? 10 * simds : ~0ull;
    if (n < line || (xf32 && cpr < 128)) return lpr;
    while (lpr > 8 && 4 * ((cpr + lpr - 1) / lpr * lpr) > 5 * cpr) lpr >>= 1;
    return lpr;
}

/* m <= 8 rows, K % 256 == 0.  Rows of x are x_row_stride elements apart. */
int r9vx_launch_gemv(const r9vx_gemv_problem &p, hipStream_t stream) {
    const uint32_t cpr = p.k / 32; /* 16-byte chunks per row, a multiple of 8 */
    const bool gated = p.epilogue == R9VX_EPILOGUE_SWIGLU;
    const uint32_t lpr = row_lanes(cpr, p.n, gated, p.x_dtype == R9VX_DTYPE_F32);
    /* Two chunks per lane when that fills whole segments (K a multiple of
     * 4096) or makes the row one segment (K in 2048..4096), and the activation
     * registers fit (M rows x 2 chunks); half-empty pairs in a row of several
     * segments are slower (Q4_K n = K = 5120, m = 2: 9.7 -> 11.4 us).  This
     * choice, the rows per lane group, the activation staging and the
     * streaming forms follow m, but none of them changes a row's arithmetic: a
     * lane always owns the chunks lir, lir + lpr, ... of every row and adds them
     * in that order (two per segment or one; ragged rows the last first), and
     * the cross-lane sum over the lanes is the same tree for every value, so a
     * row's outputs are the same bits for every m of a bucket <= 8. */
    const bool pairs = lpr == 64 && (cpr % 128 == 0 || (cpr > 64 && cpr < 128));
    const int spl = (pairs && p.m <= (p.x_dtype == R9VX_DTYPE_F32 ? 2u : 4u)) ? 2 : 1;
    uint32_t lpr_log2 = 0;
    while ((1u << lpr_log2) < lpr) ++lpr_log2;
    GemvArgs a;
    a.w = p.w;
    a.ws = p.w_scales;
    a.ws_row = p.scheme == R9VX_SCHEME_Q8_0 ? p.k / 32 : p.k / 256;
    a.x = p.x;
    a.bias = p.bias;
    a.residual = p.residual;
    a.y = p.y;
    a.w_row_stride = p.w_row_stride;
    a.x_row_stride = p.x_row_stride;
    a.n = p.n;
    a.k = p.k;
    a.lpr_log2 = lpr_log2;
    a.cpr = cpr;
    a.nseg = (cpr + lpr * spl - 1) / (lpr * spl);
    a.ragged = cpr != a.nseg * lpr * spl;
    a.y_bf16 = p.y_dtype == R9VX_DTYPE_BF16;
    a.epilogue = p.epilogue;
    const uint32_t groups = 64 / lpr;
    const bool xf32 = p.x_dtype == R9VX_DTYPE_F32;
    switch (p.scheme) {
    case R9VX_SCHEME_Q4_K: return r9vx_gemv_q4k(a, p.m, xf32, gated, spl, groups, stream);
    case R9VX_SCHEME_IQ4_XS: return r9vx_gemv_iq4xs(a, p.m, xf32, gated, spl, groups, stream);
    case R9VX_SCHEME_Q6_K: return r9vx_gemv_q6k(a, p.m, xf32, gated, spl, groups, stream);
    case R9VX_SCHEME_IQ3_S: return r9vx_gemv_iq3s(a, p.m, xf32, gated, spl, groups, stream);
    default: return r9vx_gemv_q80(a, p.m, xf32, gated, spl, groups, stream);
    }
}
