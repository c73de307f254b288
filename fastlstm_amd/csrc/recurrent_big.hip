// Launches of the whole-CU kernels (recurrent_fwd_big.hpp, recurrent_bwd_big.hpp), which recurrent_big_{fwd,bwd}_{f32,f16,bf16}.hip instantiate.
#include "recurrent_bwd_big.hpp"
#include "recurrent_launch.hpp"

namespace fastlstm {

hipError_t fwd_big_f16(const FwdStreamParams &p, int kw, int mt, int nt, int grid, int lds, hipStream_t s, int *occ);
hipError_t fwd_big_bf16(const FwdStreamParams &p, int kw, int mt, int nt, int grid, int lds, hipStream_t s, int *occ);
hipError_t bwd_big_f16(const BwdStreamParams &p, int kw, int mt, int nt, int grid, int lds, hipStream_t s, int *occ);
hipError_t bwd_big_bf16(const BwdStreamParams &p, int kw, int mt, int nt, int grid, int lds, hipStream_t s, int *occ);
hipError_t fwd_big_f32(const FwdStreamParams &p, int kw, int nt, int grid, int lds, hipStream_t s, int *occ);
hipError_t bwd_big_f32(const BwdStreamParams &p, int kw, int nt, int grid, int lds, hipStream_t s, int *occ);

hipError_t launch_fwd_big(int dtype, const FwdStreamParams &p, int kw, int mt, int nt, int grid, hipStream_t s, int *occ) {
    const int lds = big_lds_bytes(kw, mt, nt, elem_bytes(dtype), false);
    if (dtype == FASTLSTM_FP32) return fwd_big_f32(p, kw, nt, grid, lds, s, occ);
    if (dtype == FASTLSTM_FP16) return fwd_big_f16(p, kw, mt, nt, grid, lds, s, occ);
    return fwd_big_bf16(p, kw, mt, nt, grid, lds, s, occ);
}

hipError_t launch_bwd_big(int dtype, const BwdStreamParams &p, int kw, int mt, int nt, int grid, hipStream_t s, int *occ) {
    const int lds = big_lds_bytes(kw, mt, nt, elem_bytes(dtype), true);
    if (dtype == FASTLSTM_FP32) return bwd_big_f32(p, kw, nt, grid, lds, s, occ);
    if (dtype == FASTLSTM_FP16) return bwd_big_f16(p, kw, mt, nt, grid, lds, s, occ);
    return bwd_big_bf16(p, kw, mt, nt, grid, lds, s, occ);
}

}  // namespace fastlstm
