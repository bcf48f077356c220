// Copies 32-bit words between a device buffer and a mapped host buffer (either way), and optionally
// gathers up to three flag words into a status row, so that a call's output and its flags come back in
// the call's own submission instead of one blocking read each.
// Bound by the host link: 16 bytes per lane, four loads in flight per lane, reach what a pinned copy
// reaches (56 GB/s); below about 100 KB the launch itself is the cost.
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
    const bool aligned = (((uintptr_t)src | (uintptr_t)dst) & 15u) == 0u;  // uniform
    if (aligned && base + 4096u <= words) {
        const uint4 *s = reinterpret_cast<const uint4 *>(src + base) + tid;
        uint4 *d = reinterpret_cast<uint4 *>(dst + base) + tid;
        uint4 v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = s[256 * j];
#pragma unroll
        for (int j = 0; j < 4; ++j) d[256 * j] = v[j];
        return;
    }
    const uint32_t end = base + 4096u < words ? base + 4096u : words;
    for (uint32_t i = base + tid; i < end; i += 256u) dst[i] = src[i];
}
