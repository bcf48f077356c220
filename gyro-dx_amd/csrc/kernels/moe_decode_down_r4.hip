// Decode path, step 3 for batches: the down-input rotation, the fused TQ2_T dequant-GEMV of the down
// rows, and the route-weighted combine, DN_R output rows per wave.
//
// moe_decode_down owns 8 rows per group, so 8 tokens at hidden 2048 are 2,048 groups in four rounds,
// each paying the id-to-row load chain, the codebook's staging, the eight rotated inputs and a read of
// them per block. Here a lane holds the 64 activations of its (expert, block, half) in registers and
// decodes DN_R rows against them (their words straight from HBM, six per half block), so 8 tokens
// are one round of groups. Inputs are silu(g) * u, formed by moe_decode_gu_r4 / _r2.
// The rotation, products and sums are moe_decode_down's, so the results are equal bit for bit.
// Measured, 8 tokens, hidden 2048, F 512: 13.3 us against 18.0 (moe_decode_down).
// Grid: x = E / (8 * DN_R), y = n_tok; 512 threads.
// Constants: those of moe_decode_down; 0, 1 name act[slot][F]; 19 is not read.
// Requires TQ2_T experts, n_used == 8, F == 512 and E a multiple of 8 * DN_R.
#include "gyro_fast.h"
#include "fwht.h"

#ifndef DN_R
#define DN_R 4
#define DN_PIPELINE moe_decode_down_r4
#endif
#define DN_DEFINE(NAME, WG) GD_PIPELINE_NAMED_OCC(NAME, WG, 4)
#define DN_U 8
#define DN_F 512
#define DN_NB (DN_F / 128)
#define DN_ROW_BYTES (DN_NB * 34)
#define DN_BLOCK_STRIDE 132  // floats per 128-block in LDS (bank spread)

DN_DEFINE(DN_PIPELINE, 512) {
    __shared__ uint4 book4[512];
    __shared__ float act[DN_U * DN_NB * DN_BLOCK_STRIDE];
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t E = a.c[15], NE = a.c[20], t = blockIdx.y;
    const uint32_t row0 = (gd_xcd_group(blockIdx.x, gridDim.x) * 8u + wave) * DN_R;  // this wave's first row
    const bool has_signs = a.c[11] != 0xffffffffu;

    // Unit (expert k, block bb, half hf) on lane 8 k + 2 bb + hf; its expert first: the rows wait for it.
    const uint32_t k = lane >> 3, bb = (lane >> 1) & 3u, hf = lane & 1u;
    const uint32_t id = gd_global(gd_buf<const uint32_t>(a, a.c[2]) + a.c[3] + t * DN_U)[k];
    cfloat *wtp = as_const(gd_buf<const float>(a, a.c[4]) + a.c[5] + t * DN_U);
    float wts[DN_U];  // read at the end; loaded now so that their latency overlaps the rows'
#pragma unroll
    for (int kx = 0; kx < DN_U; ++kx) wts[kx] = wtp[kx];

    // Down input of expert `wave`, block ib = lane / 16, values l16 * 8 .. l16 * 8 + 7 of the block.
    const uint32_t ib = lane >> 4, l16 = lane & 15u, i0 = ib * 128u + l16 * 8u;
    gd_gu32x4 *ip = gd_global4(gd_buf<const uint32_t>(a, a.c[0]) + a.c[1] + (size_t)(t * DN_U + wave) * DN_F + i0);
    const gd_u32x4 in[2] = {ip[0], ip[1]};
    gd_u32x4 s4[2] = {};
    if (has_signs) {
        gd_gu32x4 *S = gd_global4(gd_buf<const uint32_t>(a, a.c[11]) + a.c[12] + i0);
        s4[0] = S[0];
        s4[1] = S[1];
    }
    const gd_u32x4 cbv = gd_global4(gd_buf<const uint32_t>(a, a.c[10]))[tid];
    const bool residual = a.c[21] != 0u;
    const uint32_t orow = row0 + min(lane, DN_R - 1u);
    float res = 0.f;
    if (residual) res = gd_buf<const float>(a, a.c[22])[a.c[23] + t * E + orow];

    // The lane's half blocks: words 4 hf .. 4 hf + 4 of the nine from the block's 4-byte-aligned start,
    // and the word that holds the scale (half 1) or the stream's last byte (half 0).
    const uint64_t layer_base = (uint64_t)a.c[6] | ((uint64_t)a.c[7] << 32);
    const uint8_t *src = reinterpret_cast<const uint8_t *>(layer_base) + (uint64_t)min(id, NE - 1u) * a.c[8] + a.c[9] +
                         (size_t)row0 * DN_ROW_BYTES + ((bb * 34u) & ~3u);
    gd_guint *wp = gd_global(reinterpret_cast<const uint32_t *>(src));
    uint32_t w[DN_R][5], z[DN_R];
#pragma unroll
    for (int r = 0; r < DN_R; ++r) {
#pragma unroll
        for (int j = 0; j < 5; ++j) w[r][j] = wp[r * (DN_ROW_BYTES / 4) + 4 * hf + j];
        z[r] = wp[r * (DN_ROW_BYTES / 4) + (hf ? 0u : 8u)];
    }

    float v[8];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int c = 0; c < 4; ++c) v[4 * j + c] = gd_bits_f32(in[j][c]);
    if (has_signs) {
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] *= gd_bits_f32(s4[j >> 2][j & 3]);
        gd_fwht128_x8(v, l16);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] *= GD_INV_SQRT128;
    }
    float4 *dst = reinterpret_cast<float4 *>(act + (wave * DN_NB + ib) * DN_BLOCK_STRIDE + l16 * 8u);
    dst[0] = make_float4(v[0], v[1], v[2], v[3]);
    dst[1] = make_float4(v[4], v[5], v[6], v[7]);
    reinterpret_cast<gd_u32x4 *>(book4)[tid] = cbv;
    gd_lds_barrier();  // the rows stay in flight

    float x[64];
    const float4 *xp = reinterpret_cast<const float4 *>(act + (k * DN_NB + bb) * DN_BLOCK_STRIDE + 64u * hf);
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        const float4 q = xp[j];
        x[4 * j] = q.x;
        x[4 * j + 1] = q.y;
        x[4 * j + 2] = q.z;
        x[4 * j + 3] = q.w;
    }
    const bool odd = (bb & 1u) != 0u;
    float mine = 0.f;  // lane r: output row row0 + r
#pragma unroll
    for (int r = 0; r < DN_R; ++r) {
        const uint32_t d0 = hf ? z[r] : w[r][0], last = hf ? w[r][0] : z[r];
        const float sc = gd_half(odd ? d0 >> 16 : d0 & 0xffffu);
        float sum = gd_rounded(sc * tq2_half_words_dot(w[r], odd, odd ? last : last << 16,
                                                       reinterpret_cast<const uint32_t *>(book4), x));
        sum = sum + gd_dpp_f<0xB1>(sum);   // the two halves of a block
        sum = sum + gd_dpp_f<0x4E>(sum);   // b0 + b1, b2 + b3
        sum = sum + gd_dpp_f<0x104>(sum);  // row_shl:4: (b0 + b1) + (b2 + b3) in lane 8 k
        float acc = 0.f;  // experts in k order, from lanes 8 k
#pragma unroll
        for (int kx = 0; kx < DN_U; ++kx)
            acc += wts[kx] * gd_bits_f32((uint32_t)__builtin_amdgcn_readlane((int)gd_f32_bits(sum), 8 * kx));
        mine = lane == (uint32_t)r ? acc : mine;
        __builtin_amdgcn_sched_barrier(0);
    }
    if (lane < DN_R) {
        if (residual) mine = res + mine;
        gd_buf_at<float, GD_OUT_ADDR>(a, a.c[13])[a.c[14] + t * E + orow] = mine;
    }
}
