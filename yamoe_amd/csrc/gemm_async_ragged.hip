// The products of gemm_async.hip for contraction lengths that are not multiples of 64.
#define YAMOE_INSTANTIATE_ROWS                \
  YAMOE_INSTANTIATE_ASYNC(bf16_t, 256, true)  \
  YAMOE_INSTANTIATE_ASYNC(f16_t, 256, true)
#include "gemm_async.hip"
