// How the decode path splits a call over the GPU's compute units, as functions of sizes alone.
#pragma once
#include <algorithm>
#include <cstdint>

namespace gyro {

// Blocks a lane of the batch kernels decodes at the tuned shape (n 2 to 8): 4 or 2, where the groups (E n / 32 and
// E n / 16) fill at least 7/8 of whole rounds of one group per CU (at 256 CUs 2, 4 and 6 to 8 tokens at hidden
// 2048, 4, 7 and 8 at 1024), else 0: moe_decode_gu_b and moe_decode_down, whose smaller groups balance better.
// Four layers replayed, us without and with: hidden 2048, 2 tokens 81 -> 76, 4 112 -> 105, 6 145 -> 133,
// 8 176 -> 154; forced at 3 tokens 96 -> 100, at 5 126 -> 147; hidden 1024, 4 tokens 82 -> 77, 8 114 -> 107.
inline uint32_t decode_blocks_per_lane(uint32_t E, uint32_t n, uint32_t cus) {
    for (uint32_t r : {4u, 2u}) {
        const uint32_t groups = E * n / (8 * r), rounds = (groups + cus - 1) / cus;
        if (8 * groups >= 7 * cus * rounds) return r;
    }
    return 0;
}

// Output rows R of a moe_decode_down_g group (E a multiple of R, at most max_rows and the kernel's limits of items
// and sums): the fewest rounds of one group per CU, a round costing a fixed part (ids, inputs and their
// rotation) and twice that per item of a thread. The larger R that save rounds are a batch's: two tokens at
// hidden 2560, F 640, top-10 were two rounds of R 10 and are one of R 20 (two items). Four layers replayed,
// us (E / 256 -> this): that shape 2 tokens 128 -> 121, 4 205 -> 193, 8 363 -> 342; GGUF 148 4 tokens 277 -> 257;
// 1536 / 384 / 6 3 tokens 107 -> 86; 1024 / 256 / 2 8 tokens 149 -> 76. 3 tokens at R 16 or 20 (two rounds, two
// items) took 170 and 172 against 166 at R 10 (three rounds, one item).
// Fewer rows than the most up to E / cus that the kernel takes only where they make no more rounds: groups of half
// the items in one more round pay for the inputs and their rotation once more. Three layers replayed,
// us at that most (R), with the cheapest by cost alone, and with this: one token at 3072 / 1024 / 11 144 (8), 151 (4),
// 144 (6); 3840 / 1024 / 9 153 (12), 152 (5), 143 (8); two tokens at 2304 / 896 / 16 175 (8), 185 (4);
// 3840 / 768 / 11 173 (12), 179 (6), 160 (10); three at 3072 / 512 / 15 174 (12), 187 (8), 174 (12). GGUF 148 gains from
// the extra round at a few shapes (one token at 2816 / 1024 / 16 208 (8), 201 (4)) and more without it at others (3072 / 1024 /
// 15 207 (8), 201 (4), 196 (6)).
inline uint32_t decode_down_rows(uint32_t E, uint32_t F, uint32_t U, uint32_t n, uint32_t cus, uint32_t max_rows) {
    const auto items = [=](uint32_t R) { return U * (F / 128) * 2 * ((R + 1) / 2); };
    const auto takes = [=](uint32_t R) { return E % R == 0 && items(R) <= 1024 && R * U <= 512; };
    const auto rounds = [=](uint32_t R) { return (E / R * n + cus - 1) / cus; };
    uint32_t best = std::min(max_rows, std::max(1u, E / cus)), best_cost = ~0u;
    while (best > 1 && !takes(best)) --best;
    const uint32_t most_rounds = rounds(best);
    for (uint32_t R = 1; R <= max_rows; ++R) {
        if (!takes(R) || rounds(R) > most_rounds) continue;
        const uint32_t cost = rounds(R) * (1 + 2 * ((items(R) + 511) / 512));
        if (cost < best_cost) best = R, best_cost = cost;
    }
    return best;
}

}  // namespace gyro
