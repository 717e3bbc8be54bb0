// The products of gemm_async.hip on 128 x 128 tiles.
#define YAMOE_INSTANTIATE_ROWS                \
  YAMOE_INSTANTIATE_ASYNC(bf16_t, 128, false) \
  YAMOE_INSTANTIATE_ASYNC(bf16_t, 128, true)  \
  YAMOE_INSTANTIATE_ASYNC(f16_t, 128, false)  \
  YAMOE_INSTANTIATE_ASYNC(f16_t, 128, true)
#include "gemm_async.hip"
