// Instantiates the whole-CU reverse kernels for fp16 (recurrent_bwd_big.hpp).
#define BIG_TYPE _Float16
#define BIG_NAME bwd_big_f16
#include "recurrent_big_bwd_inst.inc"
