// moe_decode_down_xg with the shared expert's gated down rows in the same launch (see moe_decode_down_g.hip).
#define DG_MAX_ABLK 128
#define DG_GENERIC 1
#define DG_SHARED 1
#define DG_PIPELINE moe_decode_down_xgs
#include "moe_decode_down_g.hip"
