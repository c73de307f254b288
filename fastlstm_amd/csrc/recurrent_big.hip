// Instantiates the 16-bit whole-CU kernels (recurrent_fwd_big.hpp, recurrent_bwd_big.hpp); launches of all of them.
#include "recurrent_bwd_big.hpp"
#include "recurrent_launch.hpp"

namespace fastlstm {

template <typename T>
static hipError_t fwd_big_t(const FwdStreamParams &p, int kw, int mt, int nt, int grid, int lds, hipStream_t s, int *occ) {
#define CASE(KW, MT, NT) \
    if (kw == KW && mt == MT && nt == NT) return launch_one(lstm_fwd_big_kernel<T, KW, MT, NT>, p, grid, lds, s, occ)
    CASE(10, 8, 1); CASE(10, 8, 2);
    CASE(12, 8, 1); CASE(12, 8, 2);
    CASE(14, 8, 1); CASE(14, 8, 2);
    CASE(16, 8, 1); CASE(16, 8, 2);
    CASE(20, 4, 1); CASE(20, 4, 2); CASE(20, 4, 4);
    CASE(24, 4, 1); CASE(24, 4, 2); CASE(24, 4, 4);
    CASE(28, 4, 1); CASE(28, 4, 2); CASE(28, 4, 4);
    CASE(32, 4, 1); CASE(32, 4, 2); CASE(32, 4, 4);
#undef CASE
    return hipErrorInvalidConfiguration;
}

template <typename T>
static hipError_t bwd_big_t(const BwdStreamParams &p, int kw, int mt, int nt, int grid, int lds, hipStream_t s, int *occ) {
#define CASE(KW, MT, NT) \
    if (kw == KW && mt == MT && nt == NT) return launch_one(lstm_bwd_big_kernel<T, KW, MT, NT>, p, grid, lds, s, occ)
    CASE(10, 8, 1); CASE(10, 8, 2);
    CASE(12, 8, 1); CASE(12, 8, 2);
    CASE(14, 8, 1); CASE(14, 8, 2);
    CASE(16, 8, 1); CASE(16, 8, 2);
    CASE(20, 4, 1); CASE(20, 4, 2); CASE(20, 4, 4);
    CASE(24, 4, 1); CASE(24, 4, 2); CASE(24, 4, 4);
    CASE(28, 4, 1); CASE(28, 4, 2); CASE(28, 4, 4);
    CASE(32, 4, 1); CASE(32, 4, 2); CASE(32, 4, 4);
#undef CASE
    return hipErrorInvalidConfiguration;
}

// fp32 (recurrent_big_fwd_f32.hip, recurrent_big_bwd_f32.hip)
hipError_t fwd_big_f32(const FwdStreamParams &p, int kw, int nt, int grid, int lds, hipStream_t s, int *occ);
hipError_t bwd_big_f32(const BwdStreamParams &p, int kw, int nt, int grid, int lds, hipStream_t s, int *occ);

hipError_t launch_fwd_big(int dtype, const FwdStreamParams &p, int kw, int mt, int nt, int grid, hipStream_t s, int *occ) {
    const int lds = big_lds_bytes(kw, mt, nt, elem_bytes(dtype));
    if (dtype == FASTLSTM_FP32) return fwd_big_f32(p, kw, nt, grid, lds, s, occ);
    if (dtype == FASTLSTM_FP16) return fwd_big_t<_Float16>(p, kw, mt, nt, grid, lds, s, occ);
    return fwd_big_t<__bf16>(p, kw, mt, nt, grid, lds, s, occ);
}

hipError_t launch_bwd_big(int dtype, const BwdStreamParams &p, int kw, int mt, int nt, int grid, hipStream_t s, int *occ) {
    const int lds = big_lds_bytes(kw, mt, nt, elem_bytes(dtype));
    if (dtype == FASTLSTM_FP32) return bwd_big_f32(p, kw, nt, grid, lds, s, occ);
    if (dtype == FASTLSTM_FP16) return bwd_big_t<_Float16>(p, kw, mt, nt, grid, lds, s, occ);
    return bwd_big_t<__bf16>(p, kw, mt, nt, grid, lds, s, occ);
}

}  // namespace fastlstm
