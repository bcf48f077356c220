// moe_decode_down_gs with three shared rows per wave, for groups of 17 to 24 output rows.
#define DG_MAX_ABLK 64
#define DG_SHARED 1
#define DG_SH_ROWS 3
#define DG_PIPELINE moe_decode_down_gs3
#include "moe_decode_down_g.hip"
