// Persistent recurrent kernels for 64 < H <= 160 (fp32: 64 < H <= 96): a workgroup holds all of W_h in its registers and takes four
// batch rows through all timesteps by itself, so that no step waits for another CU.
//
// Same mathematics, stored values and rounding points as lstm_fwd_persistent_kernel and lstm_bwd_persistent_kernel (which replace
// fastlstm/kernels.py:414-663 and 1201-1409); the sums over K are taken in another order.
//  * CW = H / 16 computing waves with 16 units each.  Forward: four row tiles of (unit, gate) per wave, ordered so that the accumulators
//    of lane (q, n) for tile a are the gates of unit 16 wave + 4 q + a; reverse: one tile of 16 units, accumulator e of lane (q, n) is
//    unit 16 wave + 4 q + e.  The MFMAs produce 16 columns for 4 rows; the lanes of the others take over cells (fold_quarters): every
//    lane has one cell, unit 16 wave + 4 q + n / 4 of row n % 4.
//  * fp32: the columns that a 16-bit layer leaves idle hold the second and the third part of h (of d_ifgo), numbers being exact sums of
//    three bf16 numbers (gemm_f32.hpp).  One MFMA multiplies a part of the weights with all three, three MFMAs make all nine
//    products -- 48 matrix cycles per 16 x 32 weights where v_mfma_f32_16x16x4_f32 takes 256 --, and the fold adds the columns up (the
//    last four hold the least number of h's sign, or zero: an infinite weight times an idle zero would be no number).
//  * h_t (d_ifgo[t]) goes through LDS in operand order, two slots in turn, one workgroup barrier per step.  The tiles of the step
//    come and go through LDS by MV waves that do nothing else (see lstm_fwd_persistent_kernel: every memory instruction of theirs
//    is unconditional, so that the waits count exactly).
// What bounds a step: its chain of latencies (LDS, MFMAs, gates, barrier).
// Requirements (host): H a multiple of 16, rows and pointers 16-byte aligned.
#pragma once
#include "recurrent_bwd.hpp"
#include "recurrent_fwd.hpp"
#include "recurrent_parts.hpp"

namespace fastlstm {

template <typename T, int CW> struct CuShape {
    static constexpr bool F32 = sizeof(T) == 4;
    static constexpr int H = 16 * CW, P = F32 ? 3 : 1;               // parts of a number
    static constexpr int MV = F32 || CW > 8 ? 2 : 4, THREADS = (CW + MV) * kWave;   // tile-moving waves
    static constexpr int KF = (H + 31) / 32, KB = (4 * H + 31) / 32;   // k-steps forward, reverse
    static constexpr int GSEG = H * (int)sizeof(T), GROW = 4 * GSEG + 16, SROW = GSEG + 16, EPC = 16 / (int)sizeof(T);
    static constexpr int GPIECES = 16 * (GSEG / 16), SPIECES = 4 * (GSEG / 16), IOT = MV * kWave;
    static constexpr int GPT = (GPIECES + IOT - 1) / IOT, SPT = (SPIECES + IOT - 1) / IOT;
    static constexpr int SET = 4 * GROW + 2 * 4 * SROW;                // LDS tiles of a step: gates, two state tiles
    static constexpr int lds_bytes(bool backward) { return 2 * (backward ? KB : KF) * kFragBytes + 2 * SET; }
};

// One value per lane: tile j's columns 0 .. 3 for lanes 4j .. 4j + 3.  fp32: the four groups of columns are
// added first, in all lanes: two additions with a rotation each, then the lanes of a tile only have to pick.
template <bool F32> __device__ __forceinline__ float fold_cells(float v0, float v1, float v2, float v3) {
    if constexpr (!F32) {
        return fold_quarters(v0, v1, v2, v3);
    } else {
        auto rot = [](float v, auto c) { return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), decltype(c)::value, 0xf, 0xf, true)); };
        auto total = [&](float v) {
            v += rot(v, std::integral_constant<int, 0x128>{});          // row_ror:8
            return v + rot(v, std::integral_constant<int, 0x124>{});    // row_ror:4
        };
        int r = __builtin_bit_cast(int, total(v0));
        r = __builtin_amdgcn_update_dpp(r, __builtin_bit_cast(int, total(v1)), 0xe4, 0xf, 0x2, false);
        r = __builtin_amdgcn_update_dpp(r, __builtin_bit_cast(int, total(v2)), 0xe4, 0xf, 0x4, false);
        r = __builtin_amdgcn_update_dpp(r, __builtin_bit_cast(int, total(v3)), 0xe4, 0xf, 0x8, false);
        return __builtin_bit_cast(float, r);
    }
}

// Tiles between global memory and LDS by the waves that do nothing else: thread io of MV waves.  LOADS state tiles come in besides
// the gates (reverse: cell, dout), STORES go out (forward: out, cell).
template <typename T, int CW> struct CuMover {
    using C = CuShape<T, CW>;
    unsigned gv[C::GPT], sv[C::SPT];   // byte offsets inside a timestep of [.., 4H] and [.., H]; kOut: no such piece
    int gl[C::GPT], sl[C::SPT];        // byte offsets inside the LDS tiles; -1: no such piece
    unsigned g_bytes, s_bytes;
    static constexpr unsigned kOut = 0xfffffff0u;
    __device__ __forceinline__ CuMover(int io, int b0, int B) {
        constexpr int PPSEG = C::GSEG / 16;
        g_bytes = (unsigned)((size_t)B * 4 * C::GSEG);
        s_bytes = (unsigned)((size_t)B * C::GSEG);
#pragma unroll
        for (int i = 0; i < C::GPT; ++i) {
            const int pc = io + C::IOT * i, row = pc / (4 * PPSEG), at = pc % (4 * PPSEG);
            const bool ok = pc < C::GPIECES && b0 + row < B;
            gv[i] = ok ? (unsigned)((size_t)(b0 + row) * 4 * C::GSEG + at * 16) : kOut;
            gl[i] = ok ? row * C::GROW + at * 16 : -1;
        }
#pragma unroll
        for (int i = 0; i < C::SPT; ++i) {
            const int pc = io + C::IOT * i, row = pc / PPSEG, at = pc % PPSEG;
            const bool ok = pc < C::SPIECES && b0 + row < B;
            sv[i] = ok ? (unsigned)((size_t)(b0 + row) * C::GSEG + at * 16) : kOut;
            sl[i] = ok ? row * C::SROW + at * 16 : -1;
        }
    }
    // timestep t of [T, B, ..]; an empty buffer where there is none (loads return zeros, stores are dropped)
    static __device__ __forceinline__ __amdgpu_buffer_rsrc_t at(const void *base, long long t, unsigned bytes, bool exists) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char *>(static_cast<const unsigned char *>(base)) + (exists ? (size_t)t * bytes : 0), 0,
                                                 exists ? bytes : 0u, 0x00020000);
    }
    // as many dropped stores as a step issues, each at an offset of its own (or the compiler keeps one of them)
    template <int N> __device__ __forceinline__ void dropped_stores(const void *base, unsigned group) const {
        const __amdgpu_buffer_rsrc_t r = at(base, 0, g_bytes, true);
        const u32x4 zero = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int i = 0; i < N; ++i) __builtin_amdgcn_raw_buffer_store_b128(zero, r, kOut - 16u * (group * N + i), 0, 0);
    }
};

template <typename T, int CW>
__global__ __launch_bounds__((CuShape<T, CW>::THREADS)) void lstm_fwd_cu_kernel(const FwdParams p) {
    using C = CuShape<T, CW>;
    using E = Elem<T>;
    using O = OperandType<T>;
    constexpr int H = C::H, KS = C::KF, P = C::P, PD = 4;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    unsigned char *const xl = smem, *const tiles = smem + 2 * KS * kFragBytes;   // operand blocks of h_t; tile sets of two steps
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int q = lane >> 4, n = lane & 15, B = p.B, T_ = p.T;
    const bool keep = p.keep != 0;
    const int rec = blockIdx.x / p.n_bt_launch, b0 = p.b_base + (blockIdx.x - rec * p.n_bt_launch) * 4;
    auto pick = [&](auto a0, auto a1, auto a2, auto a3) { return rec == 0 ? a0 : rec == 1 ? a1 : rec == 2 ? a2 : a3; };
    T *ifgo = static_cast<T *>(pick(p.ifgo, p.ifgo_x[0], p.ifgo_x[1], p.ifgo_x[2]));
    T *out = static_cast<T *>(pick(p.out, p.out_x[0], p.out_x[1], p.out_x[2]));
    T *cell = static_cast<T *>(pick(p.cell, p.cell_x[0], p.cell_x[1], p.cell_x[2]));
    const T *Wh = static_cast<const T *>(pick(p.Wh, p.Wh_x[0], p.Wh_x[1], p.Wh_x[2]));
    const size_t BH = (size_t)B * H;

    for (int i = tid; i < 2 * KS * kWave; i += C::THREADS) reinterpret_cast<u32x4 *>(xl)[i] = u32x4{0u, 0u, 0u, 0u};
    __syncthreads();

    if (wave >= CW) {   // ---- tiles -----------------------------------------------------------------
        const CuMover<T, CW> mv(tid - CW * kWave, b0, B);
        u32x4 ring[PD][C::GPT];
        auto load = [&](int t, auto uc) __attribute__((always_inline)) {
            const __amdgpu_buffer_rsrc_t r = mv.at(ifgo, t, mv.g_bytes, t < T_);
#pragma unroll
            for (int i = 0; i < C::GPT; ++i) ring[decltype(uc)::value][i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, mv.gv[i], 0, 0));
        };
        auto to_lds = [&](int t, auto uc) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < C::GPT; ++i)
                if (mv.gl[i] >= 0) *reinterpret_cast<u32x4 *>(tiles + (t & 1) * C::SET + mv.gl[i]) = ring[decltype(uc)::value][i];
        };
        auto step = [&](int t, auto uc) __attribute__((always_inline)) {
            to_lds(t + 1, std::integral_constant<int, (decltype(uc)::value + 1) % PD>{});
            __syncthreads();
            const unsigned char *g = tiles + (t & 1) * C::SET, *h = g + 4 * C::GROW, *c = h + 4 * C::SROW;
            const __amdgpu_buffer_rsrc_t rg = mv.at(ifgo, t, mv.g_bytes, keep);
            const __amdgpu_buffer_rsrc_t rh = mv.at(out, t + 1, mv.s_bytes, true), rc = mv.at(cell, t + 1, mv.s_bytes, keep || t + 1 == T_);
#pragma unroll
            for (int i = 0; i < C::GPT; ++i) __builtin_amdgcn_raw_buffer_store_b128(*reinterpret_cast<const u32x4 *>(g + max(mv.gl[i], 0)), rg, mv.gv[i], 0, 0);
#pragma unroll
            for (int i = 0; i < C::SPT; ++i) {
                __builtin_amdgcn_raw_buffer_store_b128(*reinterpret_cast<const u32x4 *>(h + max(mv.sl[i], 0)), rh, mv.sv[i], 0, 0);
                __builtin_amdgcn_raw_buffer_store_b128(*reinterpret_cast<const u32x4 *>(c + max(mv.sl[i], 0)), rc, mv.sv[i], 0, 0);
            }
            load(t + PD, uc);
        };
        static_for<0, PD>([&](auto uc) __attribute__((always_inline)) {
            load(decltype(uc)::value, uc);
            if constexpr (decltype(uc)::value + 1 < PD) mv.template dropped_stores<C::GPT + 2 * C::SPT>(ifgo, decltype(uc)::value);
        });
        to_lds(0, std::integral_constant<int, 0>{});
        __syncthreads();
        int t0 = 0;
        for (; t0 + PD <= T_; t0 += PD) static_for<0, PD>([&](auto uc) __attribute__((always_inline)) { step(t0 + decltype(uc)::value, uc); });
        static_for<0, PD - 1>([&](auto uc) __attribute__((always_inline)) {
            if (t0 + decltype(uc)::value < T_) step(t0 + decltype(uc)::value, uc);
        });
        return;
    }

    // ---- weights: fragment (tile a, k-step ks): lane (q, r) holds row r = (unit 16 wave + 4 (r / 4) + a, gate r % 4), k = 32 ks + 8 q ..
    u32x4 w[4][KS][P];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const int k0 = ks * 32 + q * 8;
            const T *src = Wh + ((size_t)(n & 3) * H + wave * 16 + (n >> 2) * 4 + a) * H + (k0 < H ? k0 : 0);   // (H a multiple of 16)
            operand_parts<T>([&](int e) { return src[e]; }, w[a][ks]);
            if (k0 >= H)
#pragma unroll
                for (int i = 0; i < P; ++i) w[a][ks][i] = u32x4{0u, 0u, 0u, 0u};
        }
    // ---- this lane's cell
    const int unit = wave * 16 + q * 4 + (n >> 2), row = n & 3;
    const bool valid = b0 + row < B;
    const size_t off = valid ? (size_t)(b0 + row) * H + unit : 0;
    const int goff = row * C::GROW + unit * E::BYTES, soff = row * C::SROW + unit * E::BYTES;
    float c_state = valid ? E::to_f32(cell[off]) : 0.f;
    auto put_h = [&](int slot, T h) {
        unsigned char *x = xl + slot * KS * kFragBytes;
        if constexpr (C::F32) {
            const ThreeParts s(h);
#pragma unroll
            for (int i = 0; i < 4; ++i)
                *reinterpret_cast<unsigned short *>(x + frag_offset<O>(4 * i + row, unit)) = (unsigned short)(__builtin_bit_cast(unsigned, s.part(i)) >> 16);
        } else {
            *reinterpret_cast<T *>(x + frag_offset<O>(row, unit)) = h;
        }
    };
    put_h(0, valid ? out[off] : E::from_f32(0.f));
    __syncthreads();   // (the movers': the tile of step 0 is in LDS)

    for (int t = 0; t < T_; ++t) {
        const unsigned char *x = xl + (t & 1) * KS * kFragBytes;
        unsigned char *g = tiles + (t & 1) * C::SET;
        u32x4 h[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) h[ks] = *reinterpret_cast<const u32x4 *>(x + (ks * kWave + lane) * 16);
        T *gl = reinterpret_cast<T *>(g + goff);
        const T g0 = gl[0], g1 = gl[H], g2 = gl[2 * H], g3 = gl[3 * H];
        __builtin_amdgcn_sched_barrier(0);
        f32x4 acc[4];
#pragma unroll
        for (int a = 0; a < 4; ++a) acc[a] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = P - 1; i >= 0; --i)   // (the small parts first)
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
#pragma unroll
                for (int a = 0; a < 4; ++a) acc[a] = mfma_kstep<O>(w[a][ks][i], h[ks], acc[a]);
        float f[4][4];
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            f[a][0] = acc[a][0]; f[a][1] = acc[a][1]; f[a][2] = acc[a][2]; f[a][3] = acc[a][3];
        }
        const float pi = E::to_f32(g0) + fold_cells<C::F32>(f[0][0], f[1][0], f[2][0], f[3][0]);
        const float pf = E::to_f32(g1) + fold_cells<C::F32>(f[0][1], f[1][1], f[2][1], f[3][1]);
        const float pg = E::to_f32(g2) + fold_cells<C::F32>(f[0][2], f[1][2], f[2][2], f[3][2]);
        const float po = E::to_f32(g3) + fold_cells<C::F32>(f[0][3], f[1][3], f[2][3], f[3][3]);
        const float c1 = sigmoidf_<C::F32>(pf) * c_state + sigmoidf_<C::F32>(pi) * tanhf_<C::F32>(pg);
        const float h1 = sigmoidf_<C::F32>(po) * tanhf_<C::F32>(c1);
        c_state = c1;
        const T hv = E::from_f32(valid ? h1 : 0.f);   // (rows past the batch stay zero in the operand blocks)
        put_h((t + 1) & 1, hv);
        gl[0] = E::from_f32(pi);
        gl[H] = E::from_f32(pf);
        gl[2 * H] = E::from_f32(pg);
        gl[3 * H] = E::from_f32(po);
        *reinterpret_cast<T *>(g + 4 * C::GROW + soff) = hv;
        *reinterpret_cast<T *>(g + 4 * C::GROW + 4 * C::SROW + soff) = E::from_f32(c1);
        __syncthreads();
    }
}

template <typename T, int CW>
__global__ __launch_bounds__((CuShape<T, CW>::THREADS)) void lstm_bwd_cu_kernel(const BwdParams p) {
    using C = CuShape<T, CW>;
    using E = Elem<T>;
    using O = OperandType<T>;
    constexpr int H = C::H, KS = C::KB, P = C::P, PD = 4;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    unsigned char *const xl = smem, *const tiles = smem + 2 * KS * kFragBytes;   // operand blocks of d_ifgo[t]; tile sets of two steps
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int q = lane >> 4, n = lane & 15, B = p.B, T_ = p.T;
    const int rec = blockIdx.x / p.n_bt_launch, b0 = p.b_base + (blockIdx.x - rec * p.n_bt_launch) * 4;
    auto pick = [&](auto a0, auto a1, auto a2, auto a3) { return rec == 0 ? a0 : rec == 1 ? a1 : rec == 2 ? a2 : a3; };
    const T *dout = static_cast<const T *>(pick(p.dout, p.dout_x[0], p.dout_x[1], p.dout_x[2]));
    const T *ifgo = static_cast<const T *>(pick(p.ifgo, p.ifgo_x[0], p.ifgo_x[1], p.ifgo_x[2]));
    const T *cell = static_cast<const T *>(pick(p.cell, p.cell_x[0], p.cell_x[1], p.cell_x[2]));
    const T *Wh = static_cast<const T *>(pick(p.Wh, p.Wh_x[0], p.Wh_x[1], p.Wh_x[2]));
    T *dh = static_cast<T *>(pick(p.dh, p.dh_x[0], p.dh_x[1], p.dh_x[2]));
    T *dc = static_cast<T *>(pick(p.dc, p.dc_x[0], p.dc_x[1], p.dc_x[2]));
    T *d_ifgo = static_cast<T *>(pick(p.d_ifgo, p.d_ifgo_x[0], p.d_ifgo_x[1], p.d_ifgo_x[2]));

    for (int i = tid; i < 2 * KS * kWave; i += C::THREADS) reinterpret_cast<u32x4 *>(xl)[i] = u32x4{0u, 0u, 0u, 0u};

    if (wave >= CW) {   // ---- tiles: gates, cell and dout of reverse step s (timestep T - 1 - s) in, d_ifgo out
        const CuMover<T, CW> mv(tid - CW * kWave, b0, B);
        u32x4 rg[PD][C::GPT], rc[PD][C::SPT], rd[PD][C::SPT];
        auto load = [&](int s, auto uc) __attribute__((always_inline)) {
            constexpr int u = decltype(uc)::value;
            const int t = T_ - 1 - s;
            const __amdgpu_buffer_rsrc_t bg = mv.at(ifgo, t, mv.g_bytes, t >= 0), bc = mv.at(cell, t, mv.s_bytes, t >= 0), bd = mv.at(dout, t, mv.s_bytes, t >= 0);
#pragma unroll
            for (int i = 0; i < C::GPT; ++i) rg[u][i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(bg, mv.gv[i], 0, 0));
#pragma unroll
            for (int i = 0; i < C::SPT; ++i) {
                rc[u][i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(bc, mv.sv[i], 0, 0));
                rd[u][i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(bd, mv.sv[i], 0, 0));
            }
        };
        auto to_lds = [&](int s, auto uc) __attribute__((always_inline)) {
            constexpr int u = decltype(uc)::value;
            unsigned char *g = tiles + (s & 1) * C::SET, *c = g + 4 * C::GROW, *d = c + 4 * C::SROW;
#pragma unroll
            for (int i = 0; i < C::GPT; ++i)
                if (mv.gl[i] >= 0) *reinterpret_cast<u32x4 *>(g + mv.gl[i]) = rg[u][i];
#pragma unroll
            for (int i = 0; i < C::SPT; ++i)
                if (mv.sl[i] >= 0) {
                    *reinterpret_cast<u32x4 *>(c + mv.sl[i]) = rc[u][i];
                    *reinterpret_cast<u32x4 *>(d + mv.sl[i]) = rd[u][i];
                }
        };
        auto step = [&](int s, auto uc) __attribute__((always_inline)) {
            to_lds(s + 1, std::integral_constant<int, (decltype(uc)::value + 1) % PD>{});
            __syncthreads();
            const unsigned char *g = tiles + (s & 1) * C::SET;
            const __amdgpu_buffer_rsrc_t ro = mv.at(d_ifgo, T_ - 1 - s, mv.g_bytes, true);
#pragma unroll
            for (int i = 0; i < C::GPT; ++i) __builtin_amdgcn_raw_buffer_store_b128(*reinterpret_cast<const u32x4 *>(g + max(mv.gl[i], 0)), ro, mv.gv[i], 0, 0);
            load(s + PD, uc);
        };
        static_for<0, PD>([&](auto uc) __attribute__((always_inline)) {
            load(decltype(uc)::value, uc);
            if constexpr (decltype(uc)::value + 1 < PD) mv.template dropped_stores<C::GPT>(d_ifgo, decltype(uc)::value);
        });
        to_lds(0, std::integral_constant<int, 0>{});
        __syncthreads();
        int s0 = 0;
        for (; s0 + PD <= T_; s0 += PD) static_for<0, PD>([&](auto uc) __attribute__((always_inline)) { step(s0 + decltype(uc)::value, uc); });
        static_for<0, PD - 1>([&](auto uc) __attribute__((always_inline)) {
            if (s0 + decltype(uc)::value < T_) step(s0 + decltype(uc)::value, uc);
        });
        return;
    }

    // ---- weights: fragment (k-step ks): lane (q, n) holds unit 16 wave + n, k = 32 ks + 8 q + e with k = 4 * source unit + gate
    u32x4 w[KS][P];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        const T *src = Wh + (size_t)(ks * 8 + q * 2) * H + wave * 16 + n;   // (4H is a multiple of 32)
        operand_parts<T>([&](int e) { return src[((size_t)(e & 3) * H + (e >> 2)) * H]; }, w[ks]);
    }
    // ---- this lane's cell
    const int unit = wave * 16 + q * 4 + (n >> 2), row = n & 3;
    const bool valid = b0 + row < B;
    const size_t off = valid ? (size_t)(b0 + row) * H + unit : 0;
    const int goff = row * C::GROW + unit * E::BYTES, soff = row * C::SROW + unit * E::BYTES;
    constexpr float GS = C::F32 ? kGradScale : 1.f, GU = C::F32 ? kGradUnscale : 1.f;   // (all gradients of the loop: recurrent_parts.hpp)
    float dh_rec = valid ? GS * E::to_f32(dh[off]) : 0.f, dc_state = valid ? GS * E::to_f32(dc[off]) : 0.f;
    float c1 = valid ? E::to_f32(cell[(size_t)T_ * B * H + off]) : 0.f;
    T nx[6];   // the gates, c_{t-1} and dout of the step, read a step ahead
    auto read_items = [&](const unsigned char *g) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) nx[i] = reinterpret_cast<const T *>(g + goff)[i * H];
        nx[4] = *reinterpret_cast<const T *>(g + 4 * C::GROW + soff);
        nx[5] = *reinterpret_cast<const T *>(g + 4 * C::GROW + 4 * C::SROW + soff);
    };
    __syncthreads();   // (the movers': the tiles of step 0 are in LDS)
    read_items(tiles);

    for (int s = 0; s < T_; ++s) {
        unsigned char *x = xl + (s & 1) * KS * kFragBytes, *g = tiles + (s & 1) * C::SET;
        const float si = sigmoidf_<C::F32>(E::to_f32(nx[0])), sf = sigmoidf_<C::F32>(E::to_f32(nx[1]));
        const float tg = tanhf_<C::F32>(E::to_f32(nx[2])), so = sigmoidf_<C::F32>(E::to_f32(nx[3]));
        const float tc = tanhf_<C::F32>(c1), c0 = E::to_f32(nx[4]), dhv = dh_rec + GS * E::to_f32(nx[5]);
        const float dc1 = dc_state + dhv * so * (1.f - tc * tc);
        const T d[4] = {E::from_f32(dc1 * tg * si * (1.f - si)), E::from_f32(dc1 * c0 * sf * (1.f - sf)), E::from_f32(dc1 * si * (1.f - tg * tg)),
                        E::from_f32(dhv * tc * so * (1.f - so))};
        dc_state = dc1 * sf;
        c1 = c0;   // c_{t-1} is the next step's c_t
        if (valid) {   // (rows past the batch stay zero in the operand blocks): k = 4 unit + gate
            if constexpr (C::F32) {
                const ThreeParts p0(d[0]), p1(d[1]), p2(d[2]), p3(d[3]);
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    *reinterpret_cast<u32x2 *>(x + frag_offset<O>(4 * i + row, 4 * unit)) =
                        u32x2{upper_halves(p0.part(i), p1.part(i)), upper_halves(p2.part(i), p3.part(i))};
            } else {
                __builtin_memcpy(x + frag_offset<O>(row, 4 * unit), d, 8);
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (C::F32) reinterpret_cast<T *>(g + goff)[i * H] = d[i] * GU;
            else reinterpret_cast<T *>(g + goff)[i * H] = d[i];
        }
        __syncthreads();
        // dh_rec(units of this wave, rows) = Wh[:, units]^T . d_ifgo[t](rows, :)^T over K = 4H, in independent sums
        constexpr int CH = P == 3 ? 3 : 2;
        f32x4 acc[CH];
#pragma unroll
        for (int i = 0; i < CH; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        constexpr int R = KS > 16 ? 8 : KS;   // operand blocks in registers
        u32x4 b[R];
#pragma unroll
        for (int ks = 0; ks < R; ++ks) b[ks] = *reinterpret_cast<const u32x4 *>(x + (ks * kWave + lane) * 16);
        if (s + 1 < T_) read_items(tiles + ((s + 1) & 1) * C::SET);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
            for (int i = 0; i < P; ++i) acc[P == 3 ? i : ks & 1] = mfma_kstep<O>(w[ks][i], b[ks % R], acc[P == 3 ? i : ks & 1]);
            if (ks + R < KS) {
                b[ks % R] = *reinterpret_cast<const u32x4 *>(x + ((ks + R) * kWave + lane) * 16);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        f32x4 sum = acc[CH - 1];
#pragma unroll
        for (int i = CH - 2; i >= 0; --i) sum += acc[i];
        const float s0 = sum[0], s1 = sum[1], s2 = sum[2], s3 = sum[3];
        dh_rec = fold_cells<C::F32>(s0, s1, s2, s3);
    }
    if (valid) {
        dh[off] = E::from_f32(GU * dh_rec);
        dc[off] = E::from_f32(GU * dc_state);
    }
}

}  // namespace fastlstm
