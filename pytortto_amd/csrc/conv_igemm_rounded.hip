// The same launches with operands rounded to bfloat16 behind the LDS read (TT_CONV_MATH_BF16), for what
// the kernels written for that arithmetic (conv_igemm_bf16.hip, conv_hwc.hip) do not take; three blocks
// per CU hide the fetches.
#define TT_IGEMM_KERNEL igemm_bf16
#define TT_IGEMM_KERNEL_MULTI igemm_multi_bf16
#define TT_IGEMM_TERMS 1
#define TT_IGEMM_BLOCKS 3
#define TT_IGEMM_EPI 0
#define TT_IGEMM_UNIT igemm_bf16_unit
#include "conv_igemm_launch.h"
