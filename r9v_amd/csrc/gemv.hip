/*
 * gemv.hip -- the decode GEMV's dispatch: how a launch's rows are cut into lanes
 * and K segments (r9vx_gemv.h has the kernels).
 */
#include "r9vx_gemv.h"

/* m <= 8 rows, K % 256 == 0.  Rows of x are x_row_stride elements apart. */
int r9vx_launch_gemv(const r9vx_gemv_problem &p, hipStream_t stream) {
    const uint32_t cpr = p.k / 32; /* 16-byte chunks per row, a multiple of 8 */
    /* 64 lanes per row, or the power of two at or above the row's chunks when
     * they are fewer than 33; lanes past the row's end idle.  A row is
     * then read in one wave-wide piece per segment whatever K is: with the
     * largest power of two that divides the row's chunks instead, K = 1792 or
     * 6144 took 7 or 3 segments in series, one load latency each (Q4_K m = 6,
     * n = 832, K = 6144: 9.8 us; K = 1792 gated, n = 1792, m = 1: 10.6).
     * Two chunks per lane when that fills whole segments (K a multiple of
     * 4096) or makes the row one segment (K in 2048..4096), and the activation
     * registers fit (M rows x 2 chunks); half-empty pairs in a row of several
     * segments are slower (Q4_K n = K = 5120, m = 2: 9.7 -> 11.4 us).  This
     * choice, the rows per lane group, the activation staging and the
     * streaming forms follow m, but none of them changes a row's arithmetic: a
     * lane always owns the chunks lir, lir + 64, ... of every row and adds them
     * in that order (two per segment or one; ragged rows the last first), and the cross-lane sum over the
     * 64 lanes is the same tree for every value, so a row's outputs are the
     * same bits for every m of a bucket <= 8. */
    const bool pairs = cpr % 128 == 0 || (cpr > 64 && cpr < 128);
    const int spl = (pairs && p.m <= (p.x_dtype == R9VX_DTYPE_F32 ? 2u : 4u)) ? 2 : 1;
    uint32_t lpr = 64;
    while (lpr > 8 && lpr / 2 >= cpr) lpr >>= 1;
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
    const bool gated = p.epilogue == R9VX_EPILOGUE_SWIGLU;
    switch (p.scheme) {
    case R9VX_SCHEME_Q4_K: return r9vx_gemv_q4k(a, p.m, xf32, gated, spl, groups, stream);
    case R9VX_SCHEME_IQ4_XS: return r9vx_gemv_iq4xs(a, p.m, xf32, gated, spl, groups, stream);
    case R9VX_SCHEME_Q6_K: return r9vx_gemv_q6k(a, p.m, xf32, gated, spl, groups, stream);
    case R9VX_SCHEME_IQ3_S: return r9vx_gemv_iq3s(a, p.m, xf32, gated, spl, groups, stream);
    default: return r9vx_gemv_q80(a, p.m, xf32, gated, spl, groups, stream);
    }
}
