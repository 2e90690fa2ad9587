// Float32 convolution arithmetic on the bf16 matrix instructions of gfx950
// (tt_set_conv_math(TT_CONV_MATH_BF16X3)): the implicit-GEMM kernel body of conv_igemm_kernel.h with
// its three-term matrix step -- every operand value as three bfloat16 terms that add up to it exactly,
// six v_mfma_f32_32x32x16_bf16 per accumulator and 16-deep step -- for Conv2d forward and the input
// gradient.  Same tiles, stream-K grid, addressing modes and epilogues as the float32 kernels.  Large launches of float32
// arithmetic run here too (Igemm::w is set then: operands of any magnitude, and infinities, give what they give there).
#define TT_IGEMM_KERNEL igemm_bf16x3
#define TT_IGEMM_KERNEL_MULTI igemm_multi_bf16x3
#define TT_IGEMM_TERMS 3
#define TT_IGEMM_BLOCKS 2
#define TT_IGEMM_EPI 0
#define TT_IGEMM_UNIT igemm_bf16x3_unit
#include "conv_igemm_launch.h"
