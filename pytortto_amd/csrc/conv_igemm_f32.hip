// The implicit-GEMM convolution on float32 matrix instructions: the default arithmetic.
#define TT_IGEMM_KERNEL igemm_f32
#define TT_IGEMM_KERNEL_MULTI igemm_multi_f32
#define TT_IGEMM_TERMS 0
#define TT_IGEMM_BLOCKS 2
#define TT_IGEMM_EPI 0
#define TT_IGEMM_UNIT igemm_f32_unit
#include "conv_igemm_launch.h"
