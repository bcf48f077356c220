// The decode router with a shared expert of any row format and width in the same launch: the
// sources of moe_router.hip, whose shared-expert groups here run the rows of shared_rows.h (bf16,
// Q8_0 or fp32 rows, SF a multiple of 64, hidden width up to 4096) instead of the bf16 rows that
// moe_decode_down_x goes on with. Group s of them computes shared rows 4 s .. 4 s + 3: its wave reads a
// gate row and the matching up row and writes a[t][r] = silu(W_sg[r] . x[t]) * (W_su[r] . x[t]), what
// moe_decode_shared_down takes; one more group forms the gate dots g . x[t].
// Constants 0 .. 19 as moe_router, then 20 SF (0: no shared groups) 21 sh_w_srv ([2 SF] rows of constant
// 25 bytes: gate rows, then up rows) 22 sh_a_uav (fp32 [n][SF]) 23 sh_gate_srv (fp32 [E]) 24 sh_g_uav
// (fp32 [n]) 25 row bytes 26 row format (0 bf16, 1 Q8_0, 2 fp32) 27 sh_a_off 28 sh_g_off.
// Grid: x = n_expert + E / 128 + SF / 4 + 1 (0 more groups without a shared expert).
// Bound by the latency of its loads: every row is read once, by its own wave.
#define ROUTER_PIPELINE moe_router_s
#define ROUTER_SHARED_ANY 1
#include "moe_router.hip"
