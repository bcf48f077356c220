// Dots of a shared expert's dense rows (bf16, Q8_0 in the layout of q8_repack, or fp32) with up to
// 8 token rows of fp32 activations, one wave per run of NR rows (moe_router_s: a gate row and its up
// row; moe_decode_shared_down: two down rows), for the decode path's one to eight tokens.
//
// The rows are read once, 16 bytes per lane and load, four loads per row in flight before the first
// product; each token's activations are requested while the previous token's products run, and serve
// all NR rows. Products are fp32 (a Q8_0 value is d * q, exact in fp32), summed per lane in column
// order and over the wave by gd_wave_sum_dpp.
#pragma once
#include "gd_kernel.h"

// Row formats as gm_layer_desc.sh_type.
enum { SHR_BF16 = 0, SHR_Q8 = 1, SHR_F32 = 2 };
#define SHR_MAX_TOK 8

// Values per 16-byte load of a row.
template <int KIND>
constexpr uint32_t shr_per() { return KIND == SHR_Q8 ? 16u : KIND == SHR_BF16 ? 8u : 4u; }

template <int KIND>
__device__ __forceinline__ void shr_values(gd_u32x4 w, float d, float (&v)[shr_per<KIND>()]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        if constexpr (KIND == SHR_Q8) {
#pragma unroll
            for (int b = 0; b < 4; ++b) v[4 * j + b] = d * (float)((int32_t)(w[j] << (24 - 8 * b)) >> 24);
        } else if constexpr (KIND == SHR_BF16) {
            v[2 * j] = gd_bits_f32(w[j] << 16);
            v[2 * j + 1] = gd_bits_f32(w[j] & 0xffff0000u);
        } else {
            v[j] = gd_bits_f32(w[j]);
        }
    }
}

// sum[i][t] = row i . x[t] for the NR rows at row[i] (cols values, a multiple of 64) and the n_tok
// (1 .. 8) activation rows at x + t x_stride (floats, 16-byte aligned); every lane gets the sums. Columns
// past the last read the row's last load again and multiply zeros.
template <int KIND, int NR>
__device__ __forceinline__ void shr_dots(const uint8_t *const (&row)[NR], uint32_t cols, const uint32_t *x,
                                         uint32_t x_stride, uint32_t n_tok, float (&sum)[NR][SHR_MAX_TOK]) {
    constexpr uint32_t PER = shr_per<KIND>(), LOADS = 4;
    const uint32_t lane = threadIdx.x & 63u;
    float acc[NR][SHR_MAX_TOK];
#pragma unroll
    for (int i = 0; i < NR; ++i)
#pragma unroll
        for (int t = 0; t < SHR_MAX_TOK; ++t) acc[i][t] = 0.f;
#pragma unroll 1
    for (uint32_t c0 = 0; c0 < cols; c0 += 64u * PER * LOADS) {
        gd_u32x4 w[NR][LOADS];
        uint16_t d[NR][LOADS];
        uint32_t col[LOADS];
        bool in[LOADS];
#pragma unroll
        for (uint32_t m = 0; m < LOADS; ++m) {
            const uint32_t c = c0 + (64u * m + lane) * PER;
            in[m] = c < cols;
            col[m] = in[m] ? c : cols - PER;
#pragma unroll
            for (int i = 0; i < NR; ++i) {
                w[i][m] = *gd_global4(reinterpret_cast<const uint32_t *>(
                    row[i] + (KIND == SHR_Q8 ? col[m] : KIND == SHR_BF16 ? col[m] * 2u : col[m] * 4u)));
                if constexpr (KIND == SHR_Q8)
                    d[i][m] = *(const __attribute__((address_space(1))) uint16_t *)(uintptr_t)(row[i] + cols + (col[m] / 32u) * 2u);
            }
        }
        gd_u32x4 xv[2][LOADS][PER / 4];
        auto load_x = [&](uint32_t t, gd_u32x4 (&o)[LOADS][PER / 4]) {
#pragma unroll
            for (uint32_t m = 0; m < LOADS; ++m)
#pragma unroll
                for (uint32_t j = 0; j < PER / 4; ++j) o[m][j] = *gd_global4(x + (size_t)t * x_stride + col[m] + 4u * j);
        };
        load_x(0u, xv[0]);
#pragma unroll
        for (int t = 0; t < SHR_MAX_TOK; ++t) {
            if ((uint32_t)t >= n_tok) break;  // uniform
            if (t + 1 < SHR_MAX_TOK) load_x(min((uint32_t)t + 1u, n_tok - 1u), xv[(t + 1) & 1]);
#pragma unroll
            for (uint32_t m = 0; m < LOADS; ++m) {
                if (c0 + 64u * m * PER >= cols) break;  // uniform: no lane has a column here
#pragma unroll
                for (int i = 0; i < NR; ++i) {
                    float v[PER], s = 0.f;
                    shr_values<KIND>(w[i][m], KIND == SHR_Q8 ? gd_half(d[i][m]) : 1.f, v);
#pragma unroll
                    for (uint32_t j = 0; j < PER; ++j) s += v[j] * gd_bits_f32(xv[t & 1][m][j / 4][j % 4]);
                    acc[i][t] += in[m] ? s : 0.f;
                }
            }
        }
    }
#pragma unroll
    for (int t = 0; t < SHR_MAX_TOK; ++t) {
        if ((uint32_t)t >= n_tok) break;  // uniform
#pragma unroll
        for (int i = 0; i < NR; ++i) sum[i][t] = gd_wave_sum_dpp(acc[i][t]);
    }
}
