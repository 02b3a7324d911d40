/*
 * gemm_thin.hip -- dequant-GEMM for the buckets above the decode GEMV's whose
 * rows do not fill the 256-row tiles of gemm.hip: y[m, n] = sum_k x[m, k] *
 * w[n, k] for bf16 activations, every weight scheme, every n.
 *
 * T0 meaning: crates/r9v-t0/src/matmul.rs:1940-2414 (Branch D), epilogue
 * matmul.rs:2421-2446.
 *
 * What bounds it: with few activation rows the weights' decode does, and the
 * chain of dependent MFMAs over K.  The chain is part of the results: an
 * output is the same bits in every bucket above the decode GEMV's, so K is
 * summed by one wave in the 256-row loop's order (v_mfma_f32_32x32x16_f16 over
 * each 64-K step's slices, 13.5 ns each) and cannot be split.  So a workgroup
 * is a narrow column strip (32 NC columns) and its waves have two roles: NR
 * waves each run the chain of one 32-row tile, eight waves decode the strip's
 * weights for them, a super-block (256 K) ahead, into LDS tiles; one barrier
 * per super-block.  The chain then waits for no decode, and the strips are
 * narrow enough to spread over the chip at the n of a projection: the 256-row
 * loop pays its whole step (about 1 us) for a tile of 32 rows, on n / 256 of
 * the CUs.  Measured (Q4_K, k = 4096, MI355X, both launches, graph-replayed):
 * m = 32, n = 4096 61 -> 16.0 us, n = 14336 62 -> 24.5; Q6_K m = 57, n = 4096,
 * k = 14336 252 -> 46.  A super-block costs 0.5 us (32 rows x 32 columns)
 * against 0.22 us of MFMAs: its decode is 32 fma_mix (8 cycles each) and about
 * 75 other instructions a thread, and neither hides all of the other's waits.
 * A wave that decoded its own operands, without the LDS tiles, took 1.0 us;
 * four decode waves instead of eight cost 5 to 20% more at 64 columns.  Eight
 * chains a workgroup (against four) halve the decode and the weights' reads of
 * prompt chunks: n = 4096, k = 4096 m = 777 55 -> 48 us, m = 1024 65 -> 54; they
 * then wait on the activations, 128 KB a super-block from the L2.
 */
#include <type_traits>

#include "r9vx_thin.h"

using namespace r9vx;

namespace {

struct ThinArgs {
    const _Float16 *x16; /* x_to_f16_thin_kernel's order */
    const float *scale;
    const uint8_t *w;
    const uint16_t *ws;
    const float *bias;
    const float *residual;
    void *y;
    uint64_t w_row_stride;
    uint32_t m, n, k;
    uint32_t y_bf16, epilogue;
    uint32_t ws_row;
};

/* One workgroup per activation row (a wave per row, x_to_f16_kernel, leaves a
 * bucket of 32 rows on 8 CUs: 6.7 -> 4.5 us at k = 4096): its max picks the power-of-two scale
 * (row_shift), and the row is written as fp16 in the weight scheme's K order,
 * so that an MFMA operand is one contiguous load: 32-row tile t's 8-element
 * group c / 8 of row r is at x16 + 32 t k + ((c / 8) R + r) 8, R the tile's
 * rows (32, or what m leaves in the last: whole tiles there would take up to
 * 31 rows more of the workspace than the rows themselves).  The bits are those of x16_row.  K <= 8192 stays in registers
 * between the max and the conversion. */
template <int PERM>
__global__ __launch_bounds__(256) void x_to_f16_thin_kernel(const uint16_t *__restrict__ x, uint32_t m, uint32_t k,
                                                            _Float16 *__restrict__ x16, float *__restrict__ scale) {
    __shared__ float wmax[4];
    const uint32_t row = blockIdx.x, tid = threadIdx.x;
    const uint16_t *const xr = x + (uint64_t)row * k;
    auto load_chunk = [&](uint32_t c, uint32_t (&w)[4]) {
        const r9vx_u32x2 lo = *reinterpret_cast<const r9vx_u32x2 *>(xr + order_pos<PERM>(c, 0));
        const r9vx_u32x2 hi = *reinterpret_cast<const r9vx_u32x2 *>(xr + order_pos<PERM>(c, 4));
        w[0] = lo.x, w[1] = lo.y, w[2] = hi.x, w[3] = hi.y;
    };
    auto max_chunk = [&](const uint32_t (&w)[4], float mx) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            mx = fmaxf(mx, fabsf(__builtin_bit_cast(float, w[j] << 16)));
            mx = fmaxf(mx, fabsf(__builtin_bit_cast(float, w[j] & 0xFFFF0000u)));
        }
        return mx;
    };
    constexpr int kHold = 4;
    const bool hold = k <= 2048u * kHold;
    uint32_t w[kHold][4];
    float mx = 0.f;
    if (hold) {
#pragma unroll
        for (int i = 0; i < kHold; ++i) {
            const uint32_t c = 8 * tid + 2048u * i;
            if (c < k) {
                load_chunk(c, w[i]);
                mx = max_chunk(w[i], mx);
            }
        }
    } else {
        for (uint32_t c = 8 * tid; c < k; c += 2048) {
            load_chunk(c, w[0]);
            mx = max_chunk(w[0], mx);
        }
    }
    for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
    if ((tid & 63) == 0) wmax[tid >> 6] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
    const int e = row_shift(mx);
    const float inv = ldexpf(1.0f, -e);
    if (tid == 0) scale[row] = ldexpf(1.0f, e);
    _Float16 *const out = x16 + (uint64_t)(row & ~31u) * k + 8 * (row & 31u);
    const uint32_t tile = row & ~31u, rows = m - tile < 32 ? m - tile : 32;
    auto put = [&](uint32_t c, const uint32_t (&v)[4]) {
        uint32_t o[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
            o[j] = pack_h2(__builtin_bit_cast(float, v[j] << 16) * inv, __builtin_bit_cast(float, v[j] & 0xFFFF0000u) * inv);
        *reinterpret_cast<r9vx_u32x4 *>(out + (uint64_t)rows * c) = r9vx_u32x4{o[0], o[1], o[2], o[3]};
    };
    if (hold) {
#pragma unroll
        for (int i = 0; i < kHold; ++i) {
            const uint32_t c = 8 * tid + 2048u * i;
            if (c < k) put(c, w[i]);
        }
    } else {
        for (uint32_t c = 8 * tid; c < k; c += 2048) {
            load_chunk(c, w[0]);
            put(c, w[0]);
        }
    }
}

/* Eight decode waves: in groups of 4 NC, each group a whole super-block. */
constexpr int kThinDec = 8;
constexpr int kThinAhead = 3; /* of its own super-blocks whose payload a decode thread holds */
constexpr int thin_groups(int nc) { return kThinDec / (4 * nc); }
/* LDS tiles: one being multiplied, the next whole, one being decoded by each group */
constexpr int thin_tiles(int nc) { return 2 + thin_groups(nc); }
/* 64-K steps of activations a chain holds, all but one in flight (a divisor of
 * 12: the chain's loop is unrolled over three super-blocks), and slices of B
 * (of 16).  Eight chains make four waves a SIMD, 128 registers each: they hold
 * less (127 used, none spilled) and cover each other's waits instead, two
 * chains a SIMD. */
constexpr int thin_a_ring(int nr, int nc) { return nr == 8 ? 3 : nc == 1 ? 6 : 4; }
constexpr int thin_b_ring(int nr) { return nr == 8 ? 2 : 4; }

template <int SCHEME, int NR, int NC>
__global__ __launch_bounds__(64 * (NR + kThinDec)) void gemm_thin_kernel(ThinArgs a) {
    /* B tile of one super-block: slice 4 ks + s of column tile ct is 64
     * 16-byte slots, lane (h, r)'s operand at slot 32 h + (r ^ (2 ks + h)):
     * the eight decode threads of a weight row write eight units at once, to
     * distinct banks */
    constexpr int TILES = thin_tiles(NC), G = thin_groups(NC);
    constexpr uint32_t kTile = NC * 16 * 64;
    __shared__ r9vx_u32x4 bt[TILES * kTile];
    __shared__ uint32_t lut[SCHEME == R9VX_SCHEME_IQ4_XS ? 256 : SCHEME == R9VX_SCHEME_IQ3_S ? kM3Iq3Words : 1];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t n0 = blockIdx.x * (32 * NC), nb = a.k / 256;
    if constexpr (SCHEME == R9VX_SCHEME_IQ4_XS) m3_init_iq4_lut(lut, tid, 64 * (NR + kThinDec));
    if constexpr (SCHEME == R9VX_SCHEME_IQ3_S) m3_init_iq3s_lut(lut, tid, 64 * (NR + kThinDec));
    if constexpr (m3_table(SCHEME)) __syncthreads();

    if (wave >= NR) {
        /* decode: thread (ct, r, u) owns unit u of every super-block of
         * weight row n0 + 32 ct + r (past n: row n - 1 again, not stored) */
        constexpr int P = kThinAhead;
        const uint32_t t = tid - 64 * NR, u = t & 7, r = (t >> 3) & 31, ct = (t >> 8) & (NC - 1);
        const uint32_t g = G == 1 ? 0u : (uint32_t)__builtin_amdgcn_readfirstlane(t >> 8);
        const uint8_t *const base = a.w + (uint64_t)n0 * a.w_row_stride;
        const uint8_t *const sbase = reinterpret_cast<const uint8_t *>(a.ws + (uint64_t)n0 * a.ws_row);
        const uint32_t row = n0 + 32 * ct + r < a.n ? 32 * ct + r : a.n - 1 - n0;
        const uint32_t off = row * (uint32_t)a.w_row_stride, soff = row * a.ws_row * 2u;
        const uint32_t ni = nb > g ? (nb - g + G - 1) / G : 0; /* its super-blocks: g + G i */
        ThinUnit<SCHEME> ring[P];
#pragma unroll
        for (int j = 0; j < P; ++j) thin_load<SCHEME>(base, off, sbase, soff, g + G * j < nb ? g + G * j : nb - 1, u, ring[j]);
        r9vx_u32x4 *const dst = bt + ct * 16 * 64 + (4 * (u >> 1)) * 64 + 32 * (u & 1) + (r ^ u);
        /* Barrier b, of nb, comes before the chain steps of super-block b and
         * says that super-block b + 1 is whole; a group has G periods between
         * barriers for a super-block.  Super-block d's tile was last read for
         * d - TILES, before barrier d - 1 - G.  Its loads are unconditional: a
         * load under a condition would make every wait a wait for all of them. */
        uint32_t tile = g, bar = 0;
        auto decode = [&](uint32_t i, int j, bool mid) {
            thin_decode<SCHEME>(ring[j], u, lut, dst + tile * kTile, [&]() {
                if (G == 2 && mid) {
                    lds_barrier();
                    ++bar;
                }
            });
            const uint32_t d = g + G * (i + P);
            thin_load<SCHEME>(base, off, sbase, soff, d < nb ? d : nb - 1, u, ring[j]);
            tile = tile + G < TILES ? tile + G : tile + G - TILES;
        };
        auto own = [&](uint32_t i, int j) { /* i >= 1 */
            if (G == 1 ? i > 1 : (i > 1 || g == 1)) {
                lds_barrier();
                ++bar;
            }
            decode(i, j, true);
        };
        if (ni > 0) decode(0, 0, false);
        uint32_t i0 = 1;
        for (; i0 + P <= ni; i0 += P) {
#pragma unroll
            for (int j = 0; j < P; ++j) own(i0 + j, (1 + j) % P);
        }
#pragma unroll
        for (int j = 0; j < P - 1; ++j)
            if (i0 + j < ni) own(i0 + j, (1 + j) % P);
        for (; bar < nb; ++bar) lds_barrier();
        return;
    }

    /* the chain of row tile mt */
    const uint32_t mt = blockIdx.y * NR + wave, h = lane >> 5;
    const uint32_t rows = a.m > 32 * mt ? (a.m - 32 * mt < 32 ? a.m - 32 * mt : 32) : 0; /* uniform */
    if (rows == 0) {
        for (uint32_t c = 0; c < nb; ++c) lds_barrier();
        return;
    }
    /* lanes past the last tile's rows read its last row again and store nothing */
    const uint32_t nk = a.k / 64, ar = (lane & 31) < rows ? (lane & 31) : rows - 1;
    const uint32_t aoff = (4 * h * rows + ar) * 16; /* slice s: group 4 h + s of a step's eight */
    const uint8_t *const abase = reinterpret_cast<const uint8_t *>(a.x16 + (uint64_t)32 * mt * a.k);
    /* A operands, up to five steps ahead: x16 comes from the L2 or, on an XCD's
     * first touch, from the memory side cache, hundreds of nanoseconds away */
    constexpr int kARing = thin_a_ring(NR, NC);
    half8 af[kARing][4];
    auto load_a = [&](uint32_t step, int s, half8 &f) {
        f = thin_ld<half8>(abase + (uint64_t)(step < nk ? step : nk - 1) * (128u * rows) + 16u * s * rows, aoff, 0);
    };
    r9vx_f32x16 acc[NC];
#pragma unroll
    for (int ct = 0; ct < NC; ++ct)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[ct][i] = 0.f;
#pragma unroll
    for (int i = 0; i < kARing - 1; ++i) {
#pragma unroll
        for (int s = 0; s < 4; ++s) load_a(i, s, af[i][s]);
        __builtin_amdgcn_sched_barrier(0); /* in the order of their use */
    }
    constexpr int kBRing = thin_b_ring(NR);
    half8 bf[kBRing][NC]; /* B operands of this slice and the next ones */
    auto load_b = [&](uint32_t tile, int sl, half8 (&f)[NC]) { /* slice sl = 4 ks + s of a tile */
        const uint32_t at = tile * kTile + 64 * sl + 32 * h + ((lane & 31) ^ (2 * (sl >> 2) + h));
#pragma unroll
        for (int ct = 0; ct < NC; ++ct) f[ct] = __builtin_bit_cast(half8, bt[at + ct * 16 * 64]);
    };
    /* One wave runs the whole chain, so its issue slots count: a slice's MFMAs
     * (32 cycles each, the chain's accumulators forwarded at full rate) are
     * followed by the loads that fit in their shadow. */
    uint32_t tile = 0;
    auto chunk = [&](uint32_t c, int j) { /* j = c modulo 3 */
        const uint32_t next = tile + 1 < TILES ? tile + 1 : 0;
#pragma unroll
        for (int sl = 0; sl < 16; ++sl) {
            const int ks = sl >> 2, s = sl & 3;
#pragma unroll
            for (int ct = 0; ct < NC; ++ct)
                acc[ct] = __builtin_amdgcn_mfma_f32_32x32x16_f16(bf[sl % kBRing][ct], af[(4 * j + ks) % kARing][s], acc[ct], 0, 0, 0);
            constexpr int P = kBRing - 1;
            load_b(sl + P < 16 ? tile : next, (sl + P) & 15, bf[(sl + P) % kBRing]); /* B(c + 1) is whole */
            load_a(4 * c + ks + kARing - 1, s, af[(4 * j + ks + kARing - 1) % kARing][s]);
            __builtin_amdgcn_sched_barrier(0);
        }
        tile = next;
        if (c + 1 < nb) lds_barrier(); /* B(c + 2) whole; the tile of B(c) is free */
    };
    lds_barrier(); /* B(0) and B(1) whole */
#pragma unroll
    for (int sl = 0; sl < kBRing - 1; ++sl) load_b(0, sl, bf[sl]);
    uint32_t c0 = 0;
    for (; c0 + 3 <= nb; c0 += 3) {
#pragma unroll
        for (int j = 0; j < 3; ++j) chunk(c0 + j, j);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
        if (c0 + j < nb) chunk(c0 + j, j);

    /* lane: row 32 mt + (lane & 31); acc[ct][4 g + e]: column n0 + 32 ct +
     * 8 g + 4 h + e.  y = acc 2^e [+ bias | + residual] in f32, then the cast */
    if ((lane & 31) >= rows) return;
    const uint32_t row = 32 * mt + (lane & 31);
    const float sc = a.scale[row];
    const bool vec = (a.n & 3u) == 0;
#pragma unroll
    for (int ct = 0; ct < NC; ++ct)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const uint32_t c0 = n0 + 32 * ct + 8 * g + 4 * h;
            if (c0 >= a.n) continue;
            const uint64_t at = (uint64_t)row * a.n + c0;
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = acc[ct][4 * g + e] * sc;
            if (a.epilogue != R9VX_EPILOGUE_NONE) {
                const float *const add = a.epilogue == R9VX_EPILOGUE_BIAS ? a.bias + c0 : a.residual + at;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (vec || c0 + e < a.n) v[e] += add[e];
            }
            if (a.y_bf16) {
                uint16_t *const y = reinterpret_cast<uint16_t *>(a.y) + at;
                const uint16_t b[4] = {r9vx_f32_to_bf16(v[0]), r9vx_f32_to_bf16(v[1]), r9vx_f32_to_bf16(v[2]),
                                       r9vx_f32_to_bf16(v[3])};
                if (vec) {
                    *reinterpret_cast<r9vx_u32x2 *>(y) =
                        r9vx_u32x2{b[0] | ((uint32_t)b[1] << 16), b[2] | ((uint32_t)b[3] << 16)};
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (c0 + e < a.n) y[e] = b[e];
                }
            } else {
                float *const y = reinterpret_cast<float *>(a.y) + at;
                if (vec) {
                    *reinterpret_cast<r9vx_f32x4 *>(y) = r9vx_f32x4{v[0], v[1], v[2], v[3]};
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (c0 + e < a.n) y[e] = v[e];
                }
            }
        }
}

/* Rows of one launch: a multiple of every shape's row tiles whose grids stay
 * within HIP's limits (2^32 threads in x, one workgroup of 256 per row in the
 * conversion; 65535 workgroups in y, 32 rows each and more).  Which rows share a
 * launch changes no output bit. */
constexpr uint32_t kThinMaxRows = 1u << 20;

template <int SCHEME>
int launch_thin(const ThinArgs &a, uint32_t nr, uint32_t nc, hipStream_t s) {
    const dim3 grid((a.n + 32 * nc - 1) / (32 * nc), (a.m + 32 * nr - 1) / (32 * nr)), block(64 * (nr + kThinDec));
#define R9VX_THIN(NR, NC, NS, LOAD)                                                      \
    if (nr == NR && nc == NC) {                                                          \
        hipLaunchKernelGGL((gemm_thin_kernel<SCHEME, NR, NC>), grid, block, 0, s, a);    \
        return (int)hipGetLastError();                                                   \
    }
    R9VX_THIN_SHAPES(R9VX_THIN)
#undef R9VX_THIN
    return (int)hipErrorInvalidValue;
}

void launch_x16(uint32_t order, const uint16_t *x, uint32_t m, uint32_t k, _Float16 *x16, float *scale, hipStream_t s) {
    const dim3 grid(m), block(256);
    switch (order) {
    case R9VX_SCHEME_Q4_K: hipLaunchKernelGGL(x_to_f16_thin_kernel<R9VX_SCHEME_Q4_K>, grid, block, 0, s, x, m, k, x16, scale); break;
    case R9VX_SCHEME_IQ4_XS: hipLaunchKernelGGL(x_to_f16_thin_kernel<R9VX_SCHEME_IQ4_XS>, grid, block, 0, s, x, m, k, x16, scale); break;
    case R9VX_SCHEME_Q6_K: hipLaunchKernelGGL(x_to_f16_thin_kernel<R9VX_SCHEME_Q6_K>, grid, block, 0, s, x, m, k, x16, scale); break;
    default: hipLaunchKernelGGL(x_to_f16_thin_kernel<0>, grid, block, 0, s, x, m, k, x16, scale); break;
    }
}

}  // namespace

int r9vx_launch_gemm_thin(const r9vx_gemm_problem &p, uint32_t nr, uint32_t nc, hipStream_t stream) {
    if (nr == 0 || nc == 0) return (int)hipErrorInvalidValue;
    ThinArgs a{};
    _Float16 *x16 = reinterpret_cast<_Float16 *>(p.workspace);
    float *scale = reinterpret_cast<float *>(reinterpret_cast<uint8_t *>(p.workspace) +
                                             r9vx_gemm_x16_bytes(p.m, p.k));
    a.w = p.w;
    a.ws = p.w_scales;
    a.bias = p.bias;
    a.w_row_stride = r9vx_row_bytes(p.scheme, p.k);
    a.ws_row = r9vx_row_scales(p.scheme, p.k);
    a.n = p.n;
    a.k = p.k;
    a.y_bf16 = p.y_dtype == R9VX_DTYPE_BF16;
    a.epilogue = p.epilogue;
    for (uint32_t r0 = 0; r0 < p.m; r0 += kThinMaxRows) {
        a.m = p.m - r0 < kThinMaxRows ? p.m - r0 : kThinMaxRows;
        a.x16 = x16 + (size_t)r0 * p.k;
        a.scale = scale + r0;
        a.residual = p.residual ? p.residual + (size_t)r0 * p.n : nullptr;
        a.y = reinterpret_cast<uint8_t *>(p.y) + (size_t)r0 * p.n * (a.y_bf16 ? 2 : 4);
        launch_x16(r9vx_group_order(p.scheme), p.x + (size_t)r0 * p.k, a.m, p.k, x16 + (size_t)r0 * p.k, scale + r0, stream);
        int e = (int)hipGetLastError();
        if (e) return e;
        switch (p.scheme) {
        case R9VX_SCHEME_Q4_K: e = launch_thin<R9VX_SCHEME_Q4_K>(a, nr, nc, stream); break;
        case R9VX_SCHEME_IQ4_XS: e = launch_thin<R9VX_SCHEME_IQ4_XS>(a, nr, nc, stream); break;
        case R9VX_SCHEME_Q6_K: e = launch_thin<R9VX_SCHEME_Q6_K>(a, nr, nc, stream); break;
        case R9VX_SCHEME_Q8_0: e = launch_thin<R9VX_SCHEME_Q8_0>(a, nr, nc, stream); break;
        default: e = launch_thin<R9VX_SCHEME_IQ3_S>(a, nr, nc, stream); break;
        }
        if (e) return e;
    }
    return 0;
}
