// Instantiates the whole-CU kernels (recurrent_fwd_big.hpp, recurrent_bwd_big.hpp) for the 16-bit element types.
#include "recurrent_bwd_big.hpp"
#include "recurrent_launch.hpp"

namespace fastlstm {

template <typename T>
static hipError_t fwd_big_t(const FwdStreamParams &p, int kw, int nt, int grid, int lds, hipStream_t s, int *occ) {
#define CASE(KW, NT) \
    if (kw == KW && nt == NT) return launch_one(lstm_fwd_big_kernel<T, KW, NT>, p, grid, lds, s, occ)
    CASE(20, 1); CASE(20, 2); CASE(20, 4);
    CASE(24, 1); CASE(24, 2); CASE(24, 4);
    CASE(28, 1); CASE(28, 2); CASE(28, 4);
    CASE(32, 1); CASE(32, 2); CASE(32, 4);
#undef CASE
    return hipErrorInvalidConfiguration;
}

template <typename T>
static hipError_t bwd_big_t(const BwdStreamParams &p, int kw, int nt, int grid, int lds, hipStream_t s, int *occ) {
#define CASE(KW, NT) \
    if (kw == KW && nt == NT) return launch_one(lstm_bwd_big_kernel<T, KW, NT>, p, grid, lds, s, occ)
    CASE(20, 1); CASE(20, 2); CASE(20, 4);
    CASE(24, 1); CASE(24, 2); CASE(24, 4);
    CASE(28, 1); CASE(28, 2); CASE(28, 4);
    CASE(32, 1); CASE(32, 2); CASE(32, 4);
#undef CASE
    return hipErrorInvalidConfiguration;
}

hipError_t launch_fwd_big(int dtype, const FwdStreamParams &p, int kw, int nt, int grid, hipStream_t s, int *occ) {
    const int lds = big_lds_bytes(kw, nt, 2);
    if (dtype == FASTLSTM_FP16) return fwd_big_t<_Float16>(p, kw, nt, grid, lds, s, occ);
    return fwd_big_t<__bf16>(p, kw, nt, grid, lds, s, occ);
}

hipError_t launch_bwd_big(int dtype, const BwdStreamParams &p, int kw, int nt, int grid, hipStream_t s, int *occ) {
    const int lds = big_lds_bytes(kw, nt, 2);
    if (dtype == FASTLSTM_FP16) return bwd_big_t<_Float16>(p, kw, nt, grid, lds, s, occ);
    return bwd_big_t<__bf16>(p, kw, nt, grid, lds, s, occ);
}

}  // namespace fastlstm
