/* gemv_q80.hip -- the decode GEMV (r9vx_gemv.h) over Q8_0 weights. */
#include "r9vx_gemv.h"

int r9vx_gemv_q80(const GemvArgs &a, uint32_t m, bool xf32, bool gated, int spl, uint32_t g, hipStream_t s) {
    return launch_gemv_scheme<R9VX_SCHEME_Q8_0>(a, m, xf32, gated, spl, g, s);
}
