// Instantiates the whole-CU reverse kernels for bf16 (recurrent_bwd_big.hpp).
#define BIG_TYPE __bf16
#define BIG_NAME bwd_big_bf16
#include "recurrent_big_bwd_inst.inc"
