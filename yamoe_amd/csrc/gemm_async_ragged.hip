// The products of gemm_async.hip for contraction lengths that are not multiples of 64.
#define YAMOE_RAGGED true
#define YAMOE_RAGGED_TU 1
#include "gemm_async.hip"
