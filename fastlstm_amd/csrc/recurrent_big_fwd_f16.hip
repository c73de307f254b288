// Instantiates the whole-CU forward kernels for fp16 (recurrent_fwd_big.hpp).
#define BIG_TYPE _Float16
#define BIG_NAME fwd_big_f16
#include "recurrent_big_fwd_inst.inc"
