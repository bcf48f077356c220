// moe_decode_down_g with the shared expert's gated down rows in the same launch (see moe_decode_down_g.hip).
#define DG_MAX_ABLK 64
#define DG_SHARED 1
#define DG_PIPELINE moe_decode_down_gs
#include "moe_decode_down_g.hip"
