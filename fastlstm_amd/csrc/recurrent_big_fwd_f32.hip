// Instantiates the fp32 whole-CU forward kernels (recurrent_fwd_big.hpp).
#include "recurrent_fwd_big.hpp"
#include "recurrent_launch.hpp"

namespace fastlstm {

// fp32, H = 128 KW, all weights in registers as three parts: 16 units per workgroup in 640 ... 1024, 8 in 1280 ... 2048
hipError_t fwd_big_f32(const FwdStreamParams &p, int kw, int nt, int grid, int lds, hipStream_t s, int *occ) {
#define CASE(KW, MT, NT) \
    if (kw == KW && nt == NT) return launch_one(lstm_fwd_big_parts_kernel<float, KW, MT, NT>, p, grid, lds, s, occ)
    CASE(5, 4, 1); CASE(5, 4, 2); CASE(6, 4, 1); CASE(6, 4, 2); CASE(7, 4, 1); CASE(7, 4, 2); CASE(8, 4, 1); CASE(8, 4, 2);
    CASE(10, 2, 1); CASE(10, 2, 2); CASE(10, 2, 4); CASE(12, 2, 1); CASE(12, 2, 2); CASE(12, 2, 4);
    CASE(14, 2, 1); CASE(14, 2, 2); CASE(14, 2, 4); CASE(16, 2, 1); CASE(16, 2, 2); CASE(16, 2, 4);
#undef CASE
    return hipErrorInvalidConfiguration;
}

}  // namespace fastlstm
