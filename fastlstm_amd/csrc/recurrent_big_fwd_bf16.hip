// Instantiates the whole-CU forward kernels for bf16 (recurrent_fwd_big.hpp).
#define BIG_TYPE __bf16
#define BIG_NAME fwd_big_bf16
#include "recurrent_big_fwd_inst.inc"
