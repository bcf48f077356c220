// Decode path, step 2 for batches: routing, the fused TQ2_T dequant-GEMV of the gate and up rows,
// and their SwiGLU, with several blocks decoded against one register copy of the activations.
//
// What bounds a batch is the LDS: a block costs its lane 64 codebook gathers (about 5.6 clocks of
// the CU's LDS each, bank conflicts included) and 32 16-byte reads of its 128 activations (8 clocks
// each), and moe_decode_gu_b repeats the reads, the staging and the routing for every block. Here a
// lane owns block b of GU_R / 2 rows, gate and up: the activations of half a block are read into
// registers once and GU_R blocks are decoded against them. A group holds whole rows (all K), so it
// also forms silu(g) * u: the down kernel reads one value per slot and column where it read two per
// K-part, and forms none. One wave routes while the others stage the codebook and the token's fp32
// activations (eight waves routing side by side took a third of the instructions issued).
// The products, their order and the block sums are moe_decode_gu's, so the results are equal bit for bit.
// Measured, 8 tokens, hidden 2048, F 512: 21.2 us against 23.2 (moe_decode_gu_b), the LDS
// gathers alone about 11; with moe_decode_down_r4 a replayed step of four layers 176 -> 154 us.
// Grid: x = F / (8 * (64 / (E / 128)) * GU_R / 2), z = n_tok * 8; 512 threads.
// Output act[slot][F] = silu(g) * u (not rotated, no signs).
// Constants: those of moe_decode_gu (16 gu_uav and 17 gu_off name the output).
// Requires TQ2_T experts, E 1024 or 2048, n_expert <= 256, top-8 and F a multiple of the group's rows.
#include "gyro_fast.h"
#include "fwht.h"
#include "route_fast.h"

#ifndef GU_R
#define GU_R 4  // blocks per lane: gate and up of GU_R / 2 rows
#define GU_PIPELINE moe_decode_gu_r4
#endif
#define GU_DEFINE(NAME, WG) GD_PIPELINE_NAMED_OCC(NAME, WG, 4)  // expands NAME before it is named
#define GU_U 8

GU_DEFINE(GU_PIPELINE, 512) {
    __shared__ uint4 book4[512];
    __shared__ uint4 xall[16 * 33];  // the token's E fp32 activations (x33_stage_index order)
    __shared__ uint32_t expert;
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t NE = a.c[2], E = a.c[18], F = a.c[19];
    const uint32_t slot = blockIdx.z, t = slot / GU_U, k = slot - t * GU_U;
    const uint32_t nb = E / 128u, bshift = nb == 16u ? 4u : 3u;  // blocks per row
    const uint32_t rpw = 64u >> bshift;                          // rows of a wave per row set
    const uint32_t b = lane & (nb - 1u), rr = lane >> bshift;
    const uint32_t row0 = (blockIdx.x * 8u + wave) * (GU_R / 2u) * rpw + rr;

    // Waves 1-7 and wave 0 alike request the codebook and the activations; wave 0 routes meanwhile.
    const float *logits = gd_buf<const float>(a, a.c[0]) + a.c[1] + t * NE;
    float lv[4];
    if (wave == 0u) rf_load<4>(logits, NE, lv);
    const gd_u32x4 cbv = gd_global4(gd_buf<const uint32_t>(a, a.c[15]))[tid];
    gd_u32x4 xv;
    const bool has_x = tid * 4u < E;  // uniform per wave
    if (has_x) xv = gd_global4(gd_buf<const uint32_t>(a, a.c[9]) + a.c[10] + t * E)[tid];
    uint32_t ids[GU_U];
    float top[GU_U];
    const bool writer = blockIdx.x == 0u && k == 0u;  // this group records the token's ids and weights
    if (wave == 0u) {
        uint64_t key[4];
        rf_init<4>(lv, NE, key);
        uint32_t e = 0;
#pragma unroll
        for (int j = 0; j < GU_U; ++j) {
            if ((uint32_t)j <= k || writer) {  // uniform
                ids[j] = rf_next<4>(key, top[j]);
                if ((uint32_t)j == k) e = ids[j];
            }
        }
        if (lane == 0u) expert = e < NE ? e : NE - 1u;  // never address past the layer
    }
    reinterpret_cast<gd_u32x4 *>(book4)[tid] = cbv;
    if (has_x) reinterpret_cast<gd_u32x4 *>(xall)[x33_stage_index(tid >> 5, tid & 31u)] = xv;
    __syncthreads();

    // Block b of the lane's GU_R rows (gate and up of each row set): 9 words from the block's
    // 4-byte-aligned start (word aligned for even b).
    const uint32_t e = __builtin_amdgcn_readfirstlane(expert);
    const uint64_t layer_base = (uint64_t)a.c[11] | ((uint64_t)a.c[12] << 32);
    const uint8_t *eb = reinterpret_cast<const uint8_t *>(layer_base) + (uint64_t)e * a.c[13];
    const uint32_t row_bytes = nb * 34u;
    uint32_t d[GU_R][9];
#pragma unroll
    for (int i = 0; i < GU_R; ++i) {
        gd_guint *w = gd_global(reinterpret_cast<const uint32_t *>(
            eb + ((i & 1) ? a.c[14] : 0u) + (uint64_t)(row0 + (uint32_t)(i >> 1) * rpw) * row_bytes + ((b * 34u) & ~3u)));
#pragma unroll
        for (int j = 0; j < 9; ++j) d[i][j] = w[j];
    }
    if (writer && wave == 0u) {  // while the blocks are in flight
        float wts[GU_U];
        rf_weights<GU_U>(top, gd_bits_f32(a.c[4]), wts);
        if (lane < GU_U) {
            uint32_t id = ids[0];
            float wv = wts[0];
#pragma unroll
            for (int j = 1; j < GU_U; ++j) {
                id = lane == (uint32_t)j ? ids[j] : id;
                wv = lane == (uint32_t)j ? wts[j] : wv;
            }
            gd_buf<uint32_t>(a, a.c[5])[a.c[6] + t * GU_U + lane] = id;
            gd_buf<float>(a, a.c[7])[a.c[8] + t * GU_U + lane] = wv;
        }
    }
    const uint32_t *book = reinterpret_cast<const uint32_t *>(book4);
    const uint4 *xb = xall + b * 33u;
    const bool odd = (b & 1u) != 0u;
    float acc0[GU_R], acc1[GU_R];
    tq2_blocks_dot<GU_R>(d, odd, book, xb, acc0, acc1);
    float v[GU_R];
#pragma unroll
    for (int i = 0; i < GU_R; ++i) {
        const float sc = gd_half(odd ? d[i][0] >> 16 : d[i][0] & 0xffffu);
        float s = gd_rounded(sc * (acc0[i] + acc1[i]));
        s = s + gd_dpp_f<0xB1>(s);   // quad_perm [1,0,3,2]: + lane ^ 1
        s = s + gd_dpp_f<0x4E>(s);   // quad_perm [2,3,0,1]: + lane ^ 2
        s = s + gd_dpp_f<0x104>(s);  // row_shl:4: + lane + 4 (read by lanes b < 4)
        if (nb == 16u) s = s + gd_dpp_f<0x108>(s);  // row_shl:8: the second K-part (blocks 8-15)
        v[i] = s;
    }
    if (b == 0u) {
        float *out = gd_buf<float>(a, a.c[16]) + a.c[17] + (size_t)slot * F;
#pragma unroll
        for (int i = 0; i < GU_R; i += 2) out[row0 + (uint32_t)(i >> 1) * rpw] = gd_silu_rcp(v[i]) * v[i + 1];
    }
}
