// Decode path, the shared expert's down rows ahead of the routed experts' down kernel, for the row
// formats and widths that moe_decode_down_x does not fold in (src/engine.zig:644-653):
//   s[t][r] = sigmoid(g[t]) * (W_sd[r] . a[t]) (+ res[t][r])
// with a and g from moe_router_s; the routed down kernel then adds s as its residual. One launch for
// what took an SwiGLU, a matrix-vector, a gate dot and one or two elementwise launches; each wave reads two
// rows (shared_rows.h), all loads in flight at once, since a row of a few hundred columns is one
// or two loads a lane and the launch is bound by their latency. Measured with moe_router_s on the
// real model's layer (hidden 2560, Q8_0 shared expert of width 640), 2 tokens: 84.0 -> 46.5 us a layer
// against mv_q8 twice (15.1 us each), ew twice (4.6) and a one-row mv_f32 (9.6).
// Grid: x = ceil(E / 8); 256 threads.
// Constants: 0 a_uav 1 a_off (fp32 [n][SF]) 2 g_uav 3 g_off (fp32 [n]) 4 w_srv ([E] rows) 5 row bytes
// 6 row format (0 bf16, 1 Q8_0, 2 fp32) 7 SF (a multiple of 64) 8 E 9 n_tok (1 .. 8) 10 s_uav 11 s_off
// (fp32 [n][E]) 12 residual (0: none, 1: add) 13 res_uav 14 res_off (fp32 [n][E])
#include "shared_rows.h"

template <int KIND>
__device__ __forceinline__ void shared_down(const GdArgs &a, uint32_t r0) {
    const uint32_t lane = threadIdx.x & 63u, E = a.c[8], n_tok = min(a.c[9], (uint32_t)SHR_MAX_TOK);
    const uint8_t *W = gd_buf<const uint8_t>(a, a.c[4]);
    const uint8_t *const row[2] = {W + (size_t)r0 * a.c[5], W + (size_t)min(r0 + 1u, E - 1u) * a.c[5]};
    // Lane 8 i + t finishes row i of token t: its gate dot and residual, requested ahead of the rows.
    const uint32_t i = (lane >> 3) & 1u, t = lane & 7u;
    const bool mine = lane < 16u && t < n_tok && r0 + i < E;
    float g = 0.f, res = 0.f;
    if (mine) {
        g = gd_bits_f32(*gd_global(gd_buf<const uint32_t>(a, a.c[2]) + a.c[3] + t));
        if (a.c[12]) res = gd_bits_f32(*gd_global(gd_buf<const uint32_t>(a, a.c[13]) + a.c[14] + t * E + r0 + i));
    }
    float sum[2][SHR_MAX_TOK];
    shr_dots<KIND, 2>(row, a.c[7], gd_buf<const uint32_t>(a, a.c[0]) + a.c[1], a.c[7], n_tok, sum);
    float v = 0.f;
#pragma unroll
    for (int k = 0; k < SHR_MAX_TOK; ++k)
        if ((uint32_t)k < n_tok) v = t == (uint32_t)k ? (i ? sum[1][k] : sum[0][k]) : v;
    if (mine) {
        v = gd_sigmoid_accurate(g) * v;
        if (a.c[12]) v = res + v;
        gd_buf<float>(a, a.c[10])[a.c[11] + t * E + r0 + i] = v;
    }
}

GD_PIPELINE_NAMED(moe_decode_shared_down, 256) {
    const uint32_t r0 = __builtin_amdgcn_readfirstlane((blockIdx.x * 4u + (threadIdx.x >> 6)) * 2u);
    if (r0 >= a.c[8]) return;  // uniform per wave; no barrier follows
    switch (a.c[6]) {
        case SHR_Q8: shared_down<SHR_Q8>(a, r0); break;
        case SHR_F32: shared_down<SHR_F32>(a, r0); break;
        default: shared_down<SHR_BF16>(a, r0); break;
    }
}
