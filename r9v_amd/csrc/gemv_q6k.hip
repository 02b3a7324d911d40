/* gemv_q6k.hip -- the decode GEMV (r9vx_gemv.h) over Q6_K weights. */
#include "r9vx_gemv.h"

int r9vx_gemv_q6k(const GemvArgs &a, uint32_t m, bool xf32, bool gated, int spl, uint32_t g, hipStream_t s) {
    return launch_gemv_scheme<R9VX_SCHEME_Q6_K>(a, m, xf32, gated, spl, g, s);
}
