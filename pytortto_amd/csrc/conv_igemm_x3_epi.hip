// conv_igemm_x3.hip with an epilogue on what is stored.
#define TT_IGEMM_KERNEL igemm_epi_bf16x3
#define TT_IGEMM_TERMS 3
#define TT_IGEMM_BLOCKS 2
#define TT_IGEMM_EPI 1
#define TT_IGEMM_UNIT igemm_epi_bf16x3_unit
#include "conv_igemm_launch.h"
