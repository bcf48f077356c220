// Copies 32-bit words between a device buffer and a mapped host buffer (either way), and optionally
// gathers up to three flag words into a status row, so that a call's output and its flags come back in
// the call's own submission instead of one blocking read each.
// Bound by the host link: 16 bytes per lane, four loads in flight per lane, reach what a pinned copy
// reaches (56 GB/s); small copies are bound by one round trip over the link, so no load waits for another
// (one token's 8 KB with dependent word loads took 12 us).
// Constants: 0 src uav 1 src offset (words) 2 dst uav 3 dst offset (words) 4 words (0: flags only)
// 5 flags (0 to 3) 6 status uav 7 status offset (words), then for flag i: 8 + 2 i uav, 9 + 2 i word.
// Grid: x = ceil(words / 4096), at least 1; 256 threads.
#include "gd_kernel.h"

GD_PIPELINE_NAMED(transfer, 256) {
    const uint32_t tid = threadIdx.x, words = a.c[4];
    const uint32_t flags = a.c[5] < 3u ? a.c[5] : 3u;
    if (blockIdx.x == 0u && tid < 3u) {
        // Constants at fixed places, so that the argument block is not indexed by the lane.
        const uint32_t uav = tid == 0u ? a.c[8] : tid == 1u ? a.c[10] : a.c[12];
        const uint32_t word = tid == 0u ? a.c[9] : tid == 1u ? a.c[11] : a.c[13];
        if (tid < flags) gd_buf<uint32_t>(a, a.c[6])[a.c[7] + tid] = gd_buf<const uint32_t>(a, uav)[word];
    }
    const uint32_t *src = gd_buf<const uint32_t>(a, a.c[0]) + a.c[1];
    uint32_t *dst = gd_buf<uint32_t>(a, a.c[2]) + a.c[3];
    const uint32_t base = blockIdx.x * 4096u;
    if ((((uintptr_t)src | (uintptr_t)dst) & 15u) == 0u) {  // uniform
        // Lane tid's chunks tid + 256 j; the last group's loads past the end repeat the last chunk, so
        // that every load is in flight before the first store.
        const uint32_t chunks = words >> 2, c0 = base >> 2;
        const uint4 *s = reinterpret_cast<const uint4 *>(src);
        uint4 *d = reinterpret_cast<uint4 *>(dst);
        if (c0 < chunks) {
            uint4 v[4];
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) v[j] = s[min(c0 + tid + 256u * j, chunks - 1u)];
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j)
                if (c0 + tid + 256u * j < chunks) d[c0 + tid + 256u * j] = v[j];
        }
        const uint32_t left = words & 3u;  // the words after the last whole chunk
        if (left && words - left >= base && words - left < base + 4096u && tid < left)
            dst[words - left + tid] = src[words - left + tid];
        return;
    }
    const uint32_t end = base + 4096u < words ? base + 4096u : words;
    for (uint32_t i = base + tid; i < end; i += 256u) dst[i] = src[i];
}
