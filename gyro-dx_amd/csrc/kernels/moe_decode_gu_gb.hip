// moe_decode_gu_g for batches of 2 to 8 tokens, two groups per CU (see moe_decode_gu_g.hip).
#define GG_PIPELINE moe_decode_gu_gb
#define GG_GENERIC 0
#define GG_BATCH 1
#include "moe_decode_gu_g.hip"
