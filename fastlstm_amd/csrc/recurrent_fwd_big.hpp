// Persistent forward kernel for 16-bit elements and 1280 <= H <= 4096, and for fp32 and 640 <= H <= 2048: a workgroup keeps up to
// 512 KiB of weights -- those of 16 hidden units, or of 32 where H <= 2048 in 16 bits, or of 8 where H > 1024 in fp32 -- on its CU for the whole launch, up to 384 KiB of
// them in registers, the rest in LDS.
//
// Same mathematics, stored values and rounding points as lstm_fwd_persistent_kernel (which replaces
// fastlstm/kernels.py:414-663).  lstm_fwd_stream_kernel reads all of W_h (H = 4096: 128 MiB) from memory every timestep;
// here it is read once per launch.
//  * one wave per SIMD with all of its 512 registers: the 4 waves split K (k-step ks = wave + 4 ki), a wave holds
//    MT unit tiles (4 units each) x KW k-steps: 96 blocks in registers (384 per lane), the others in LDS, spread evenly over
//    the k-steps so that an LDS read has the MFMAs of the k-steps between to arrive;
//  * the batch tiles of 16 rows are multiplied one after the other.  Operand blocks go through a ring of R blocks of
//    registers, refilled as they are consumed, across the tiles of a step;
//  * behind each tile the four partial sums meet in LDS and the gates of its rows are computed;
//  * exchange by device-scope stores of whole 16-byte pieces.  What tells a member that they are there goes by big_fwd_data:
//    - the data itself, as in recurrent_fwd_xcd.hpp (unwritten words, four slots, the same argument for what may be overwritten when), tile by
//      tile: the rows of a tile are on their way while the next tile is multiplied, and the first blocks of the next step's first tile are
//      requested behind the last ones of this step's last, so with several tiles nobody waits (of a step of H = 2048 with two tiles 0.7 us are
//      waits, where the flags and the drains in front of them took 2.5);
//    - or one flag per workgroup and step, raised behind the acknowledgement of its stores: with one tile everybody would look for blocks
//      that cannot be there yet, and their loads and the marking of words as unwritten double what the members' L2s have to give up.
//    us per step, flags and data: bf16 H = 2048, 64 rows (one tile) 4.3 and 4.8, 128 rows (two) 7.3 and 6.2; H = 2560, 16, 32, 64 rows (one, two,
//    four tiles of half the units) 4.3, 5.7, 8.4 and 3.7, 3.9, 7.4; H = 4096 5.1, 7.0, 11.4 and 4.6, 5.8, 11.3.  fp32, three times the words: H = 1024, 64 rows
//    (one tile) 4.7 and 5.4, 128 rows (two; the registers do not hold what it takes) 7.2 and 8.0, H = 640, 128 rows 5.8 and 5.3, H = 768 6.4 and 5.5, H = 896, 80
//    rows 6.9 and 5.7, H = 1280, 16 rows 4.8 and 4.2, H = 1536 (activations kept) 4.5 and 4.7, H = 2048, 16, 32, 64 rows 5.7, 8.0, 12.6 and 5.9, 7.7, 14.6.
//    (With 128 rows of H = 2048 these are from whole calls; alone a step takes 5.3 in inference and 5.8 where the activations are kept, within training
//    calls, whose products hold the clocks down, 6.5.  Of the four tiles: before their results left behind the next products, see the .inc.)
// What bounds a step now: the operand blocks, 512 KiB per CU at H = 4096 and 64 rows -- a CU takes 90 KB per us from its L2, whatever is in
// flight --, then the chain behind a tile: sums through LDS, gates (0.2 us per cell of a lane), pieces.  us per step of lstm_fwd_stream_kernel and here:
// H = 4096, 64 rows 24.8 -> 10.2, 16 rows 20.9 -> 4.6; H = 3072, 32 rows 14.1 -> 4.5; H = 2560, 64 rows 15.4 -> 6.9; and no packed copy of W_h per call (118
// us at 4096).
// Up to H = 2048, with 32 units, there are twice as many barrier groups as lstm_fwd_wide_kernel has: half the rows per group, half
// the operand bytes per CU (H = 1280, B = 64 3.99 -> 3.31).
// fp32 (lstm_fwd_big_parts_kernel): every number as the sum of three bf16 parts (recurrent_parts.hpp), the weights' 384 H bytes per
// workgroup all in registers, h_t exchanged as parts; the largest of the six products has a sum of its own.  What bounds it: at two
// batch tiles the 96 H bytes of operand blocks of each (H = 1024: 192 KiB per CU and step), at one the exchange.  H = 1024,
// us per step of the kernels on the fp32 matrix instructions (1/16 of the rate) and here: B = 128 11.1 -> 7.1, B = 16 5.1 -> 3.9.
// Up to four recurrences share a launch (T = 256, I = 256, inference / training of three layers, two of them in a launch and three: H = 1024,
// B = 16 2.93 / 8.48 and 2.20 / 7.38 ms; of four, B = 32 4.23 / 13.4 and 3.76 / 12.8; H = 640, B = 16, three 2.37 / 6.49 and 1.78 / 5.40).
// Above H = 1024 a workgroup holds 8 units (MT = 2: 384 KiB at H = 2048), one group of up to 64 rows is a launch, and every CU reads the
// 6 H bytes of each of its rows every step.  T = 100, I = 512, inference with lstm_fwd_stream_kernel and here: H = 2048, B = 1
// 1.66 -> 0.60 ms, 16 1.74 -> 0.70, 64 4.37 -> 1.65, 200 (four launches) 9.05 -> 5.38; H = 1280, B = 16 1.14 -> 0.57, 100 3.18 -> 2.13.
// Requirements (host): H a multiple of MT * 4 (and of 8; fp32: of 128), the workgroups of all groups co-resident.
#pragma once
#include <type_traits>

#include "gemm16.hpp"
#include "recurrent_parts.hpp"
#include "recurrent_stream.hpp"

namespace fastlstm {

constexpr int kBigRegBlocks = 96;   // blocks of weights per wave (of 4 registers per lane) that stay in registers,
constexpr int kBigAccBlocks = 64;   // the first of them in the accumulator half of the register file

constexpr int big_ring(int kw, int mt) {   // reverse kernel: operand blocks in flight per wave: what the registers hold
    return mt == 8 ? (kw <= 10 ? 16 : kw <= 12 ? 12 : kw <= 14 ? 6 : 8) : kw <= 20 ? 16 : kw <= 24 ? 12 : 10;
}
constexpr int big_fwd_ring(int kw, int mt, int nt) {   // forward (a block more and weights move to scratch memory: tests/test_mfma_wait_states.py)
    return mt == 8 ? (kw <= 10 ? 10 : kw <= 12 ? (nt > 1 ? 8 : 12) : kw <= 14 ? 8 : nt > 1 ? 6 : 8) : kw <= 20 ? 16 : kw <= 24 ? (nt > 1 ? 10 : 12) : kw <= 28 ? (nt > 1 ? 8 : 10) : 8;
}
// The data tells that it is there (see above; figures there).
constexpr bool big_fwd_data(int kw, int mt, int nt, int parts) {
    return parts == 1 ? nt > 1 || mt == 4 : mt == 2 ? (nt == 1 ? kw <= 10 : nt == 2) : nt == 2 && kw < 8;
}
constexpr int big_fwd_slots(int kw, int mt, int nt, int parts) { return big_fwd_data(kw, mt, nt, parts) ? kXchgSlots : 2; }   // exchange slots
// k-steps of weights in LDS.  (14, forward: there is room for one more, and the ring's registers are worth more; reverse pass, H = 1792, T = 256, us with two
// and with three: 1 row 1174 and 1201, 16 1119 and 1132, 64 1245 and 1253, 100 1591 and 1614, 128 1614 and 1620, 256 3321 and 3311)
constexpr int big_lds_steps(int kw, int mt, bool backward) {
    return kw > kBigRegBlocks / mt ? kw - kBigRegBlocks / mt + (kw == 14 && !backward) : 0;
}
// tiles whose partial sums meet in LDS at a time: all, or four where the weights leave room for no more
constexpr int big_sum_tiles(int kw, int mt) { return 4 * big_lds_steps(kw, mt, true) * mt > 48 ? 4 : mt; }
constexpr int big_lds_bytes(int kw, int mt, int nt, int es, bool backward) {   // (es: bytes per element)
    const int bt = 16 * nt, gseg = 4 * mt * es;
    return 4 * (big_lds_steps(kw, mt, backward) * mt + big_sum_tiles(kw, mt)) * kFragBytes + (nt == 1 ? 2 : 1) * bt * (4 * gseg + 16) + 2 * bt * (gseg + 16);
}

// acc (+)= A . B with the A block in the accumulator half of the register file (ACC_HALF) or in the ordinary one.  Inline assembly:
// the compiler's own MFMAs copied every block of weights out of the accumulator half before its use (900 copies per
// step).  FIRST: acc starts from zero.  The reader of acc puts mfma_results in front.
template <typename T, bool ACC_HALF, bool FIRST>
__device__ __forceinline__ void mfma_resident(f32x4 &acc, const u32x4 &a, const u32x4 &b) {
#define FASTLSTM_MFMA(OP)                                                                           \
    if constexpr (FIRST && ACC_HALF) asm(OP " %0, %1, %2, 0" : "=&v"(acc) : "a"(a), "v"(b));        \
    else if constexpr (FIRST) asm(OP " %0, %1, %2, 0" : "=&v"(acc) : "v"(a), "v"(b));               \
    else if constexpr (ACC_HALF) asm(OP " %0, %1, %2, %0" : "+v"(acc) : "a"(a), "v"(b));            \
    else asm(OP " %0, %1, %2, %0" : "+v"(acc) : "v"(a), "v"(b))
    if constexpr (std::is_same_v<T, _Float16>) {
        FASTLSTM_MFMA("v_mfma_f32_16x16x32_f16");
    } else {
        FASTLSTM_MFMA("v_mfma_f32_16x16x32_bf16");
    }
#undef FASTLSTM_MFMA
}
// The wait states between these MFMAs and the first other reader of their results (4 passes: 8 of them).  The results go through
// the statement, so that no reader moves in front of it; that no copy of them does either -- the compiler does not see MFMAs
// here, and would not wait -- is checked in the machine code (tests/test_mfma_wait_states.py).
template <int N> __device__ __forceinline__ void mfma_results(f32x4 (&acc)[N]) {
    static_assert(N == 4 || N == 8, "unit tiles of the whole-CU kernels");
    if constexpr (N == 4)
        asm volatile("s_nop 15\n\ts_nop 7" : "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]), "+v"(acc[3]));
    else
        asm volatile("s_nop 15\n\ts_nop 7"
                     : "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]), "+v"(acc[3]), "+v"(acc[4]), "+v"(acc[5]), "+v"(acc[6]), "+v"(acc[7]));
}

// The parts' products in the order in which they are added (mfma_parts): a[2] b[0], a[0] b[2], a[1] b[1], a[1] b[0], a[0] b[1]; a[0] b[0].
constexpr int part_a(int i) { return i == 0 ? 2 : i == 2 || i == 3 ? 1 : 0; }
constexpr int part_b(int i) { return i == 1 ? 2 : i == 2 || i == 4 ? 1 : 0; }

// One text for both kernels: as an inlined function the 16-bit forms came out otherwise, 1% slower (a training step of H = 2048 in bf16
// 7.63 -> 7.71 ms), since the compiler unrolls the loops before it sees the caller's arguments.
template <typename T, int KW, int MT, int NT>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(1, 1))) void lstm_fwd_big_kernel(const FwdStreamParams p) {
#include "recurrent_fwd_big.inc"
}
template <typename T, int KW, int MT, int NT>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(1, 1))) void lstm_fwd_big_parts_kernel(const FwdStreamParams p) {
#include "recurrent_fwd_big.inc"
}

}  // namespace fastlstm
