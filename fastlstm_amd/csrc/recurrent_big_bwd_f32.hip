// Instantiates the fp32 whole-CU reverse kernels (recurrent_bwd_big.hpp).
#include "recurrent_bwd_big.hpp"
#include "recurrent_launch.hpp"

namespace fastlstm {

// H = 128 kw: 16 units per workgroup and teams of 4 in 640 ... 1024, 8 units and teams of 8 in 1280 ... 2048
hipError_t bwd_big_f32(const BwdStreamParams &p, int kw, int nt, int grid, int lds, hipStream_t s, int *occ) {
    const int team = kw > 8 ? kBigTeamHalf : kBigTeam, kwm = kw > 8 ? kw / 2 : kw;   // (k-steps of a wave: H / 32 / team)
#define CASE(KW, NT, V) \
    if (kwm == KW && nt == NT && team == V) return launch_one(lstm_bwd_big_parts_kernel<float, KW, 4, NT, V>, p, grid, lds, s, occ)
    CASE(5, 1, 4); CASE(5, 2, 4); CASE(6, 1, 4); CASE(6, 2, 4); CASE(7, 1, 4); CASE(7, 2, 4); CASE(8, 1, 4); CASE(8, 2, 4);
    CASE(5, 1, 8); CASE(5, 2, 8); CASE(5, 4, 8); CASE(6, 1, 8); CASE(6, 2, 8); CASE(6, 4, 8);
    CASE(7, 1, 8); CASE(7, 2, 8); CASE(7, 4, 8); CASE(8, 1, 8); CASE(8, 2, 8); CASE(8, 4, 8);
#undef CASE
    return hipErrorInvalidConfiguration;
}

}  // namespace fastlstm
