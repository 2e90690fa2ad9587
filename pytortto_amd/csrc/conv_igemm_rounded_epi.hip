// conv_igemm_rounded.hip with an epilogue on what is stored.
#define TT_IGEMM_KERNEL igemm_epi_bf16
#define TT_IGEMM_TERMS 1
#define TT_IGEMM_BLOCKS 3
#define TT_IGEMM_EPI 1
#define TT_IGEMM_UNIT igemm_epi_bf16_unit
#include "conv_igemm_launch.h"
