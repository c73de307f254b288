// Persistent reverse-time kernel for 16-bit elements and 1280 <= H <= 4096, and for fp32 and 640 <= H <= 2048: weights on the CU for the whole launch, as in
// lstm_fwd_big_kernel, and the product split over K among teams.  Same mathematics and results as
// lstm_bwd_persistent_kernel (which replaces fastlstm/kernels.py:1201-1409); the sums over K are taken in another order.
//
// A workgroup that owned its units and all of K = 4H would read the whole d_ifgo[t] of the group's rows every step (H = 4096,
// 64 rows: 2 MiB).  Here a team of 4 neighbouring workgroups owns 16 MT units (64, or 128 where H <= 2048); member m keeps the
// weights of all of them for the m-th part of K (up to 512 KiB: three quarters in registers, the rest in LDS), reads that quarter
// of d_ifgo[t] and sends every member its partial sums through the XCD's L2 (fp32, 4 KiB for 64 rows of 16 units; words that have not been
// written say so, recurrent_fwd_xcd.hpp); the members add what they got in member order.  The K loop is that of lstm_fwd_big_kernel: MT unit tiles (of 16 units) x KW
// k-steps per wave, batch tile after batch tile, a ring of operand blocks in registers, the waves' sums added in LDS behind
// each tile.
//  * the inputs of the next step come in with LDS-direct loads (a tile row is a whole number of 16-byte slots, the last one
//    padding: lane l of wave instruction i fills slot 64 i + l), requested before the wait for the group's flags;
//  * a wave takes the cells of one unit tile and batch tile: lane (q, n) units 4q .. 4q + 3 of row n, which is what a lane
//    holds of a product tile.
// What bounds a step: the operand blocks (512 KiB per CU at H = 4096 and 64 rows) and the two exchanges.  us per step of
// lstm_bwd_stream_kernel and here: H = 4096, 64 rows 33.6 -> 12.8, 16 rows 21.1 -> 6.7; H = 3072, 32 rows 16.8 -> 7.2;
// H = 2560, 64 rows 22.6 -> 9.5.  Of the form with 16 units and 8 waves per CU for H <= 2048 and here, while the team's sums went by flags:
// H = 2048, 128 rows 11.0 -> 8.6, 64 rows 9.0 -> 6.2, 32 rows 6.4 -> 5.3; H = 1280, 128 rows 8.7 -> 7.0.  Since then (sums that say themselves that they
// are there, gate derivatives computed while they travel) 128 rows of H = 2048 9.2 -> 7.6, fp32 H = 1024, 64 rows 7.4 -> 6.1; forward and
// reverse pass together, us per timestep of a training call: bf16 H = 1280, 32 rows 8.9 -> 8.2, H = 2048, 32 rows 10.4 -> 9.6, H = 3072, 16 rows 13.0 -> 11.2, H =
// 4096, 64 rows 33.0 -> 32.0; fp32 H = 640, 16 rows 9.3 -> 8.7, H = 1280, 16 rows 12.8 -> 11.8, H = 2048, 64 rows 43.1 -> 40.4.
// Up to H = 2048 a second recurrence of the same shape may share the launch, in fp32 up to H = 1024 a third and a fourth too (the directions of a
// bidirectional layer, the chunks of a wavefront): the sums are those of a launch of its own, bit by bit.  us per step of a pair on lstm_bwd_wide_kernel and here:
// H = 2048, B = 16 6.8 -> 5.2, B = 32 9.8 -> 6.5; H = 1536, B = 32 7.7 -> 5.6; H = 1280, B = 20 6.6 -> 5.9.
// fp32 (lstm_bwd_big_parts_kernel, MT = 4): d_ifgo[t] is exchanged as the three bf16 parts of its numbers, the weights' are all in
// registers; bounds as in 16 bits with 1.5 times the bytes per number.  H = 1024, us per step of the kernel on the fp32 matrix
// instructions and here: B = 128 12.4 -> 10.4, B = 16 6.6 -> 5.9 (by flags).
// Above H = 1024 a workgroup has 8 units, half a unit tile: teams of 8 own 64 units, members 2 v and 2 v + 1 share tile v's sums, and
// a member reads an eighth of d_ifgo[t] (teams of 4 with two unit tiles would read a quarter; hence the multiples of 256).  T = 100,
// I = 512, training step with lstm_bwd_stream_kernel and here (the forward pass as in recurrent_fwd_big.hpp): H = 2048, B = 1
// 4.05 -> 1.48 ms, 16 4.85 -> 1.91, 64 12.9 -> 4.74, 200 30.3 -> 15.1; H = 1280, B = 16 3.09 -> 1.52, 100 8.63 -> 5.38.
// Requirements (host): H a multiple of 16 MT (fp32: of 128, above 1024 of 256), workgroup ids dealt to the XCDs in turn, all teams co-resident.
#pragma once
#include <type_traits>

#include "recurrent_fwd_big.hpp"

namespace fastlstm {

constexpr int kBigTeam = 4, kBigTeamHalf = 8;   // members of a team; with half a unit tile each

template <typename T, int KW, int MT, int NT>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(1, 1))) void lstm_bwd_big_kernel(const BwdStreamParams p) {
    constexpr int V = kBigTeam;
#include "recurrent_bwd_big.inc"
}
template <typename T, int KW, int MT, int NT, int V>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(1, 1))) void lstm_bwd_big_parts_kernel(const BwdStreamParams p) {
#include "recurrent_bwd_big.inc"
}

}  // namespace fastlstm
