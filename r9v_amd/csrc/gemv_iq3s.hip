/* gemv_iq3s.hip -- the decode GEMV (r9vx_gemv.h) over IQ3_S weights. */
#include "r9vx_gemv.h"

int r9vx_gemv_iq3s(const GemvArgs &a, uint32_t m, bool xf32, bool gated, int spl, uint32_t g, hipStream_t s) {
    return launch_gemv_scheme<R9VX_SCHEME_IQ3_S>(a, m, xf32, gated, spl, g, s);
}
