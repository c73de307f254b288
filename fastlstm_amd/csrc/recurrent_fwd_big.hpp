// Persistent forward kernel for 16-bit elements and 1280 <= H <= 4096: a workgroup keeps up to 512 KiB of weights -- those of
// 16 hidden units, or of 32 where H <= 2048 -- on its CU for the whole launch, three quarters of them in registers, the rest in LDS.
//
// Same mathematics, stored values and rounding points as lstm_fwd_persistent_kernel (which replaces
// fastlstm/kernels.py:414-663).  lstm_fwd_stream_kernel reads all of W_h (H = 4096: 128 MiB) from memory every timestep;
// here it is read once per launch.
//  * one wave per SIMD with all of its 512 registers: the 4 waves split K (k-step ks = wave + 4 ki), a wave holds
//    MT unit tiles (4 units each) x KW k-steps: 96 blocks in registers (384 per lane), the others in LDS, spread evenly over
//    the k-steps so that an LDS read has the MFMAs of the k-steps between to arrive;
//  * the batch tiles of 16 rows are multiplied one after the other.  Operand blocks go through a ring of R blocks of
//    registers, refilled as they are consumed, across the tiles of a step;
//  * behind each tile the four partial sums meet in LDS and the gates of its rows are computed while the next tile's operand
//    blocks arrive;
//  * exchange and flags as in lstm_fwd_wide_kernel: device-scope stores of 16-byte pieces, two slots, one flag per workgroup.
// What bounds a step now: the operand blocks, 512 KiB per CU at H = 4096 and 64 rows (16 MiB through the L2 of an XCD at about
// 2.1 TB/s), and the exchange.  us per step of lstm_fwd_stream_kernel and here: H = 4096, 64 rows 24.8 -> 11.0, 16 rows
// 20.9 -> 4.8; H = 3072, 32 rows 14.1 -> 5.5; H = 2560, 64 rows 15.4 -> 8.7; and no packed copy of W_h per call (118 us at 4096).
// Up to H = 2048, with 32 units, there are twice as many barrier groups as lstm_fwd_wide_kernel has: half the rows per group, half
// the operand bytes per CU (H = 1280, B = 64 3.99 -> 3.31).
// Requirements (host): H a multiple of MT * 4 (and of 8), the workgroups of all groups co-resident.
#pragma once
#include <type_traits>

#include "gemm16.hpp"
#include "recurrent_stream.hpp"

namespace fastlstm {

constexpr int kBigRegBlocks = 96;   // blocks of weights per wave (of 4 registers per lane) that stay in registers,
constexpr int kBigAccBlocks = 64;   // the first of them in the accumulator half of the register file

constexpr int big_ring(int kw, int mt) {   // operand blocks in flight per wave: what the registers hold
    return mt == 8 ? (kw <= 10 ? 16 : kw <= 12 ? 12 : kw <= 14 ? 6 : 8) : kw <= 20 ? 16 : kw <= 24 ? 12 : 10;
}
constexpr int big_lds_steps(int kw, int mt) { return kw > kBigRegBlocks / mt ? kw - kBigRegBlocks / mt : 0; }
// tiles whose partial sums meet in LDS at a time: all, or four where the weights leave room for no more
constexpr int big_sum_tiles(int kw, int mt) { return 4 * big_lds_steps(kw, mt) * mt > 48 ? 4 : mt; }
constexpr int big_lds_bytes(int kw, int mt, int nt) {   // (16-bit elements)
    const int bt = 16 * nt, gseg = 4 * mt * 2;
    return 4 * (big_lds_steps(kw, mt) * mt + big_sum_tiles(kw, mt)) * kFragBytes + bt * (4 * gseg + 16) + 2 * bt * (gseg + 16);
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

template <typename T, int KW, int MT, int NT>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(1, 1))) void lstm_fwd_big_kernel(const FwdStreamParams p) {
    using E = Elem<T>;
    static_assert(E::BYTES == 2, "16-bit element types");
    constexpr int NWV = 4, TPW = MT / NWV;                 // waves, unit tiles whose cells a wave takes
    constexpr int KL = big_lds_steps(KW, MT), KR = KW - KL, ACC_STEPS = kBigAccBlocks / MT;
    constexpr int ST = big_sum_tiles(KW, MT);
    constexpr int HT = 4 * MT, BT = 16 * NT;
    constexpr int NB = KW * NT, R = big_ring(KW, MT);              // operand blocks of a step, in flight
    constexpr int GSEG = HT * E::BYTES, GROW = 4 * GSEG + 16, SROW = GSEG + 16, PPSEG = GSEG / 16;
    static_assert(BT * PPSEG <= kThreads, "one state piece per thread");
    constexpr auto in_lds = [](int ki) { return ki * KL % KW < KL; };   // evenly spread, the first k-step among them
    constexpr auto reg_of = [](int ki) { return KL ? ki - ki * KL / KW - 1 : ki; };

    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    unsigned char *wl = smem;                                                             // [wave][KL][MT] blocks
    f32x4 *red = reinterpret_cast<f32x4 *>(smem + NWV * KL * MT * kFragBytes);            // [wave][ST][64]
    unsigned char *tiles = reinterpret_cast<unsigned char *>(red + NWV * ST * kWave);     // gates, h, c tiles
    unsigned char *const sth = tiles + BT * GROW, *const stc = sth + BT * SROW;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int q = lane >> 4, n = lane & 15;
    const int KS = p.KS, H = p.H, B = p.B, T_ = p.T;
    const bool keep = p.keep != 0;
    const int lin = xcd_major_id(blockIdx.x, gridDim.x);
    const int g = lin / p.n_ht, j = lin % p.n_ht;
    const int u0 = j * HT, b0 = p.b_base + g * BT;
    T *ifgo = static_cast<T *>(p.ifgo);
    T *out = static_cast<T *>(p.out);
    T *cell = static_cast<T *>(p.cell);
    const T *Wh = static_cast<const T *>(p.Wh);

    // ---- this wave's weights: fragment (unit tile a, k-step ks = wave + 4 ki): lane (q, n) holds row (unit a*4 + n/4,
    // gate n%4), k = ks*KSTEP + q*EPL ..: 16 contiguous bytes of W_h; zeros past H
    u32x4 wreg[KR][MT];
    auto fragment = [&](int ki, int a) {
        const int k0 = (wave + NWV * ki) * E::KSTEP + q * E::EPL, unit = u0 + a * 4 + (n >> 2);
        u32x4 v = *reinterpret_cast<const u32x4 *>(Wh + ((size_t)(n & 3) * H + unit) * H + (k0 < H ? k0 : 0));
        if (k0 >= H) v = u32x4{0u, 0u, 0u, 0u};
        return v;
    };
    // (whole 4-register tuples in the half that they are used from; the loads of a k-step are under way together)
    static_for<0, KW>([&](auto kc) __attribute__((always_inline)) {
        constexpr int ki = decltype(kc)::value, k = in_lds(ki) ? 0 : reg_of(ki);
        u32x4 f[MT];
#pragma unroll
        for (int a = 0; a < MT; ++a) f[a] = fragment(ki, a);
#pragma unroll
        for (int a = 0; a < MT; ++a) {
            if constexpr (in_lds(ki)) *reinterpret_cast<u32x4 *>(wl + ((wave * KL + ki * KL / KW) * MT + a) * kFragBytes + lane * 16) = f[a];
            else if constexpr (k < ACC_STEPS) asm volatile("" : "+a"(f[a]));
            else asm volatile("" : "+v"(f[a]));
            if constexpr (!in_lds(ki)) wreg[k][a] = f[a];
        }
    });

    // ---- this lane's cells: unit tiles wave + 4 h, row 16 i + n of batch tile i -------------
    float c_state[NT][TPW];
    bool live[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) {
        const int b = b0 + i * 16 + n;
        live[i] = i * 16 + n < rows_computed(B - b0);
#pragma unroll
        for (int h = 0; h < TPW; ++h)
            c_state[i][h] = b < B ? E::to_f32(cell[(size_t)b * H + u0 + (wave + NWV * h) * 4 + q]) : 0.f;
    }
    const int goff = n * GROW + (wave * 4 + q) * E::BYTES, soff = n * SROW + (wave * 4 + q) * E::BYTES;

    // ---- this thread's 16-byte piece of the state tiles and of the exchange blocks ------------------
    const unsigned xslot = (unsigned)p.n_bt * NT * p.KSP * kFragBytes;
    const unsigned xgrp = (unsigned)g * NT * p.KSP * kFragBytes;
    const XchgGlobal xch(p.xbuf, 2u * xslot);
    int *grp_flags = p.flags + (size_t)g * p.flag_stride;
    const size_t BH = (size_t)B * H, B4H = (size_t)B * 4 * H, state_org = (size_t)b0 * H + u0, tile_org = (size_t)b0 * 4 * H + u0;
    const int st_row = tid / PPSEG, st_k = tid % PPSEG;
    const bool st_ok = tid < BT * PPSEG && b0 + st_row < B;
    const unsigned st_off = st_ok ? (unsigned)(((size_t)st_row * H + st_k * E::EPL) * E::BYTES) : 0u;
    const int st_lds = st_ok ? st_row * SROW + st_k * 16 : 0;
    const unsigned x_off = st_ok ? xgrp + (unsigned)((st_row >> 4) * p.KSP * kFragBytes + frag_offset<T>(st_row & 15, u0 + st_k * E::EPL)) : 0u;

    // ---- tile I/O as in lstm_fwd_wide_kernel: the gates tile comes in with LDS-direct loads a step ahead, lane l of wave
    // instruction i filling 16-byte slot 64 i + l of the tile (the last slot of a row is padding) -------------------
    constexpr int SPR = GROW / 16, SLOTS = BT * SPR, DMA_N = (SLOTS + kWave - 1) / kWave, DPW = (DMA_N + NWV - 1) / NWV;
    unsigned dma_off[DPW];
    bool dma_ok[DPW];
#pragma unroll
    for (int d = 0; d < DPW; ++d) {
        const int i = wave + NWV * d, sl = i * kWave + lane, row = sl / SPR, idx = sl % SPR;
        dma_ok[d] = i < DMA_N && sl < SLOTS && idx < 4 * PPSEG && b0 + row < B;
        dma_off[d] = dma_ok[d] ? (unsigned)(((size_t)row * 4 * H + (size_t)(idx / PPSEG) * H + (idx % PPSEG) * E::EPL) * E::BYTES) : 0u;
    }
    const unsigned tiles_addr = (unsigned)(size_t)((FASTLSTM_LDS_PTR unsigned char *)tiles);
    const unsigned g_bytes = (unsigned)((size_t)BT * 4 * H * E::BYTES), s_bytes = (unsigned)((size_t)BT * H * E::BYTES);
    auto request_tile = [&](int t) {
        if (t >= T_) return;
        const unsigned long long addr = reinterpret_cast<unsigned long long>(uniform_ptr(ifgo + (size_t)t * B4H + tile_org));
        const u32x4 rs = {(unsigned)addr, (unsigned)(addr >> 32) & 0xffffu, g_bytes, 0x00020000u};
        const unsigned base = (unsigned)uniform_int((int)tiles_addr);
#pragma unroll
        for (int d = 0; d < DPW; ++d)
            if (dma_ok[d]) dma_block_asm<false>(rs, base + (wave + NWV * d) * kFragBytes, dma_off[d], 0u);
    };
    auto tiles_to_global = [&](int t) {
        if (keep) {
            const __amdgpu_buffer_rsrc_t rg = __builtin_amdgcn_make_buffer_rsrc(ifgo + (size_t)t * B4H + tile_org, 0, g_bytes, 0x00020000);
#pragma unroll
            for (int d = 0; d < DPW; ++d)
                if (dma_ok[d])
                    __builtin_amdgcn_raw_buffer_store_b128(
                        *reinterpret_cast<const u32x4 *>(tiles + (size_t)(wave + NWV * d) * kFragBytes + lane * 16), rg, dma_off[d], 0, 0);
        }
        if (st_ok) {
            const __amdgpu_buffer_rsrc_t rh = __builtin_amdgcn_make_buffer_rsrc(out + (size_t)(t + 1) * BH + state_org, 0, s_bytes, 0x00020000);
            const __amdgpu_buffer_rsrc_t rc = __builtin_amdgcn_make_buffer_rsrc(cell + (size_t)(t + 1) * BH + state_org, 0, s_bytes, 0x00020000);
            __builtin_amdgcn_raw_buffer_store_b128(*reinterpret_cast<const u32x4 *>(sth + st_lds), rh, st_off, 0, 0);
            if (keep || t + 1 == T_)
                __builtin_amdgcn_raw_buffer_store_b128(*reinterpret_cast<const u32x4 *>(stc + st_lds), rc, st_off, 0, 0);
        }
    };

    // ---- h_0 is version 1 in slot 0 -----------------------------
    request_tile(0);
    if (st_ok) xch.store16(x_off, *reinterpret_cast<const u32x4 *>(reinterpret_cast<const unsigned char *>(out + state_org) + st_off));
    publish_version(grp_flags + j, 1);

    for (int t = 0; t < T_; ++t) {
        const unsigned xb = xgrp + (unsigned)(t & 1) * xslot, xn = (unsigned)((t + 1) & 1) * xslot;
        if (wave == 0) wait_versions(grp_flags, p.n_ht, t + 1, p.hdr, p.spin_limit, g, t);
        __syncthreads();

        u32x4 ring[R], wf[4];
        auto request = [&](int b) {   // (past KS: zero weights times some block)
            const int ks = min(wave + NWV * (b % KW), KS - 1);
            ring[b % R] = xch.load16(lane * 16u, xb + (unsigned)((b / KW) * p.KSP + ks) * kFragBytes);
        };
        auto read_weights = [&](int l, int half) {   // four tiles at a time
#pragma unroll
            for (int a = 0; a < 4; ++a)
                wf[a] = *reinterpret_cast<const u32x4 *>(wl + ((wave * KL + l) * MT + half * 4 + a) * kFragBytes + lane * 16);
        };
#pragma unroll
        for (int b = 0; b < R; ++b) request(b);
        if constexpr (KL > 0) read_weights(0, 0);
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            f32x4 acc[MT];
            static_for<0, KW>([&](auto kc) __attribute__((always_inline)) {
                constexpr int ki = decltype(kc)::value, l = ki * KL / KW;
                constexpr bool halves_ = KL > 0 && MT == 8;   // the upper tiles of a k-step in LDS follow behind the next k-step
                const int b = i * KW + ki;
                if constexpr (in_lds(ki)) {
#pragma unroll
                    for (int a = 0; a < 4; ++a) mfma_resident<T, false, ki == 0>(acc[a], wf[a], ring[b % R]);
                    if constexpr (halves_) read_weights(l, 1);
                    else if (i + 1 < NT || l + 1 < KL) read_weights((l + 1) % (KL > 0 ? KL : 1), 0);
                } else {
#pragma unroll
                    for (int a = 0; a < MT; ++a) {
                        if (halves_ && ki == 1 && a >= 4) mfma_resident<T, (reg_of(ki) < ACC_STEPS), true>(acc[a], wreg[reg_of(ki)][a], ring[b % R]);
                        else mfma_resident<T, (reg_of(ki) < ACC_STEPS), ki == 0>(acc[a], wreg[reg_of(ki)][a], ring[b % R]);
                    }
                    if constexpr (halves_ && in_lds(ki - 1)) {
#pragma unroll
                        for (int a = 4; a < MT; ++a) mfma_resident<T, false, false>(acc[a], wf[a - 4], ring[(b - 1) % R]);
                        if (i + 1 < NT || l + 1 < KL) read_weights((l + 1) % KL, 0);
                        if (b - 1 + R < NB) request(b - 1 + R);
                    }
                }
                if (!(halves_ && in_lds(ki)) && b + R < NB) request(b + R);
                __builtin_amdgcn_sched_barrier(0);   // (the order above is the schedule)
            });
            mfma_results(acc);
#pragma unroll
            for (int a0 = 0; a0 < MT; a0 += ST) {
#pragma unroll
                for (int a = 0; a < ST; ++a) red[(wave * ST + a) * kWave + lane] = acc[a0 + a];
                __syncthreads();
#pragma unroll
                for (int h = a0 / NWV; h < (a0 + ST) / NWV; ++h) {   // unit tile wave + 4 h
                    const int tl = wave + NWV * h - a0;
                    f32x4 s = red[tl * kWave + lane];
#pragma unroll
                    for (int pp = 1; pp < NWV; ++pp) s += red[(pp * ST + tl) * kWave + lane];
                    if (live[i]) {   // (us per step with rows past the batch masked and so: H = 2048, 33 rows 5.5 -> 3.9, H = 4096, 1 row 5.1 -> 4.6)
                        T *gl_ = reinterpret_cast<T *>(tiles + i * 16 * GROW + goff) + h * NWV * 4;
                        const float pi = E::to_f32(gl_[0]) + s[0];
                        const float pf = E::to_f32(gl_[HT]) + s[1];
                        const float pg = E::to_f32(gl_[2 * HT]) + s[2];
                        const float po = E::to_f32(gl_[3 * HT]) + s[3];
                        const float c1 = sigmoidf_<false>(pf) * c_state[i][h] + sigmoidf_<false>(pi) * tanhf_<false>(pg);
                        const float h1 = sigmoidf_<false>(po) * tanhf_<false>(c1);
                        c_state[i][h] = c1;
                        if (keep) {
                            gl_[0] = E::from_f32(pi);
                            gl_[HT] = E::from_f32(pf);
                            gl_[2 * HT] = E::from_f32(pg);
                            gl_[3 * HT] = E::from_f32(po);
                        }
                        *(reinterpret_cast<T *>(sth + i * 16 * SROW + soff) + h * NWV * 4) = E::from_f32(h1);
                        *(reinterpret_cast<T *>(stc + i * 16 * SROW + soff) + h * NWV * 4) = E::from_f32(c1);
                    }
                }
                __syncthreads();   // `red` is read; behind the last tile: the state tiles are complete
            }
        }
        if (t + 1 < T_) {
            if (st_ok) xch.store16(xn + x_off, *reinterpret_cast<const u32x4 *>(sth + st_lds));
            publish_version(grp_flags + j, t + 2);
        }
        tiles_to_global(t);
        request_tile(t + 1);   // (this lane's slots of the tile are read)
    }
}

}  // namespace fastlstm
