// moe_decode_down_r4 with two output rows per wave: twice the groups, for batches whose groups would not
// fill the GPU at four. Constants and requirements: those of moe_decode_down_r4 (E a multiple of 16).
#define DN_PIPELINE moe_decode_down_r2
#define DN_R 2
#include "moe_decode_down_r4.hip"
