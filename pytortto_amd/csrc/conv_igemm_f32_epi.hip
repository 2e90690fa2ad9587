// conv_igemm_f32.hip with an epilogue on what is stored.
#define TT_IGEMM_KERNEL igemm_epi_f32
#define TT_IGEMM_TERMS 0
#define TT_IGEMM_BLOCKS 2
#define TT_IGEMM_EPI 1
#define TT_IGEMM_UNIT igemm_epi_f32_unit
#include "conv_igemm_launch.h"
