// Instantiates the one-CU kernels (recurrent_cu.hpp).
#include "recurrent_cu.hpp"
#include "recurrent_launch.hpp"

namespace fastlstm {

bool cu_shape(int H, int dtype) { return H % 16 == 0 && (dtype == FASTLSTM_FP32 ? H >= 64 && H <= 96 : H > 64 && H <= 160); }

template <typename T> static hipError_t fwd_cu_t(const FwdParams &p, int grid, hipStream_t s) {
#define CASE(CW) \
    if (p.H == 16 * CW) return launch_one(lstm_fwd_cu_kernel<T, CW>, p, grid, CuShape<T, CW>::lds_bytes(false), s, nullptr, CuShape<T, CW>::THREADS)
    CASE(5); CASE(6);
    if constexpr (sizeof(T) == 4) { CASE(4); }
    else { CASE(7); CASE(8); CASE(9); CASE(10); }
#undef CASE
    return hipErrorInvalidConfiguration;
}

template <typename T> static hipError_t bwd_cu_t(const BwdParams &p, int grid, hipStream_t s) {
#define CASE(CW) \
    if (p.H == 16 * CW) return launch_one(lstm_bwd_cu_kernel<T, CW>, p, grid, CuShape<T, CW>::lds_bytes(true), s, nullptr, CuShape<T, CW>::THREADS)
    CASE(5); CASE(6);
    if constexpr (sizeof(T) == 4) { CASE(4); }
    else { CASE(7); CASE(8); CASE(9); CASE(10); }
#undef CASE
    return hipErrorInvalidConfiguration;
}

hipError_t launch_fwd_cu(int dtype, const FwdParams &p, int grid, hipStream_t s) {
    return dtype == FASTLSTM_FP32 ? fwd_cu_t<float>(p, grid, s) : dtype == FASTLSTM_FP16 ? fwd_cu_t<_Float16>(p, grid, s) : fwd_cu_t<__bf16>(p, grid, s);
}
hipError_t launch_bwd_cu(int dtype, const BwdParams &p, int grid, hipStream_t s) {
    return dtype == FASTLSTM_FP32 ? bwd_cu_t<float>(p, grid, s) : dtype == FASTLSTM_FP16 ? bwd_cu_t<_Float16>(p, grid, s) : bwd_cu_t<__bf16>(p, grid, s);
}

}  // namespace fastlstm
