// moe_decode_gu_xg for batches of 2 to 8 tokens, two groups per CU (see moe_decode_gu_g.hip).
#define GG_PIPELINE moe_decode_gu_xgb
#define GG_GENERIC 1
#define GG_BATCH 1
#include "moe_decode_gu_g.hip"
