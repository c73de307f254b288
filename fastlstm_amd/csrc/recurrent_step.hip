// Instantiates and launches the one-step inference kernel (recurrent_step.hpp).
#include <algorithm>

#include "internal.hpp"
#include "recurrent_step.hpp"

namespace fastlstm {
namespace {

template <typename T, int MT, int NT> hipError_t launch_nt(StepParams &p, int jobs, bool vec, hipStream_t s) {
    p.tiles = cdiv(p.H, 4 * MT);
    const dim3 grid(jobs * p.tiles, cdiv(p.B, 16 * NT));
    if (vec) lstm_step_kernel<T, MT, NT, true><<<grid, kWave * 8, 0, s>>>(p);
    else lstm_step_kernel<T, MT, NT, false><<<grid, kWave * 8, 0, s>>>(p);
    return hipGetLastError();
}
template <typename T> hipError_t launch_t(StepParams &p, int jobs, bool vec, hipStream_t s) {
    if (p.B <= 16) return launch_nt<T, 1, 1>(p, jobs, vec, s);
    if (p.B <= 32) return launch_nt<T, 1, 2>(p, jobs, vec, s);
    return jobs * cdiv(p.H, 4) >= 512 ? launch_nt<T, 2, 4>(p, jobs, vec, s) : launch_nt<T, 1, 4>(p, jobs, vec, s);
}

}  // namespace

hipError_t launch_step(int dtype, StepParams &p, int jobs, bool vec, hipStream_t s) {
    return dtype == FASTLSTM_FP32 ? launch_t<float>(p, jobs, vec, s)
           : dtype == FASTLSTM_FP16 ? launch_t<_Float16>(p, jobs, vec, s)
                                    : launch_t<__bf16>(p, jobs, vec, s);
}

}  // namespace fastlstm
