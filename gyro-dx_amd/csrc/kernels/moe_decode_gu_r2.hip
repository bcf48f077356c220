// moe_decode_gu_r4 with two blocks per lane (gate and up of one row): twice the groups, for batches whose
// groups would not fill the GPU at four. Constants and requirements: those of moe_decode_gu_r4.
#define GU_PIPELINE moe_decode_gu_r2
#define GU_R 2
#include "moe_decode_gu_r4.hip"
