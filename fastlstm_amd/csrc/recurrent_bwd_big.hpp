// Persistent reverse-time kernel for 16-bit elements and 1280 <= H <= 4096: weights on the CU for the whole launch, as in
// lstm_fwd_big_kernel, and the product split over K among teams.  Same mathematics and results as
// lstm_bwd_persistent_kernel (which replaces fastlstm/kernels.py:1201-1409); the sums over K are taken in another order.
//
// A workgroup that owned its units and all of K = 4H would read the whole d_ifgo[t] of the group's rows every step (H = 4096,
// 64 rows: 2 MiB).  Here a team of 4 neighbouring workgroups owns 16 MT units (64, or 128 where H <= 2048); member m keeps the
// weights of all of them for the m-th part of K (up to 512 KiB: three quarters in registers, the rest in LDS), reads that quarter
// of d_ifgo[t] and sends every member its partial sums through the workspace (fp32, 4 KiB for 64 rows of 16 units); the
// members add what they got in member order.  The K loop is that of lstm_fwd_big_kernel: MT unit tiles (of 16 units) x KW
// k-steps per wave, batch tile after batch tile, a ring of operand blocks in registers, the waves' sums added in LDS behind
// each tile.
//  * the inputs of the next step come in with LDS-direct loads (a tile row is a whole number of 16-byte slots, the last one
//    padding: lane l of wave instruction i fills slot 64 i + l), requested before the wait for the group's flags;
//  * a wave takes the cells of one unit tile and batch tile: lane (q, n) units 4q .. 4q + 3 of row n, which is what a lane
//    holds of a product tile.
// What bounds a step: the operand blocks (512 KiB per CU at H = 4096 and 64 rows) and the two exchanges.  us per step of
// lstm_bwd_stream_kernel and here: H = 4096, 64 rows 33.6 -> 12.8, 16 rows 21.1 -> 6.7; H = 3072, 32 rows 16.8 -> 7.2;
// H = 2560, 64 rows 22.6 -> 9.5.  Of the form with 16 units and 8 waves per CU for H <= 2048 and here: H = 2048, 128 rows 11.0 -> 8.6,
// 64 rows 9.0 -> 6.2, 32 rows 6.4 -> 5.3; H = 1280, 128 rows 8.7 -> 7.0.
// Up to H = 2048 a second recurrence of the same shape may share the launch (the directions of a bidirectional layer, the chunks of
// a wavefront): the sums are those of a launch of its own, bit by bit.  us per step of a pair on lstm_bwd_wide_kernel and here:
// H = 2048, B = 16 6.8 -> 5.2, B = 32 9.8 -> 6.5; H = 1536, B = 32 7.7 -> 5.6; H = 1280, B = 20 6.6 -> 5.9.
// Requirements (host): H a multiple of 16 MT, workgroup ids dealt to the XCDs in turn, all teams co-resident.
#pragma once
#include <type_traits>

#include "recurrent_fwd_big.hpp"

namespace fastlstm {

constexpr int kBigTeam = 4;

template <typename T, int KW, int MT, int NT>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(1, 1))) void lstm_bwd_big_kernel(const BwdStreamParams p) {
    using E = Elem<T>;
    static_assert(E::BYTES == 2, "16-bit element types");
    constexpr int NWV = 4, V = kBigTeam, UT = MT / V;      // waves, members of a team, unit tiles of a member
    constexpr int KL = big_lds_steps(KW, MT), KR = KW - KL, ACC_STEPS = kBigAccBlocks / MT;
    constexpr int ST = big_sum_tiles(KW, MT);
    constexpr int HT = 16 * UT, BT = 16 * NT;
    static_assert(UT * NT <= NWV, "one tile of cells per wave");
    constexpr int NB = KW * NT, R = big_ring(KW, MT);
    constexpr int GSEG = HT * E::BYTES, GROW = 4 * GSEG + 16, SROW = GSEG + 16, PPSEG = GSEG / 16;
    constexpr auto in_lds = [](int ki) { return ki * KL % KW < KL; };   // evenly spread, the first k-step among them
    constexpr auto reg_of = [](int ki) { return KL ? ki - ki * KL / KW - 1 : ki; };

    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    unsigned char *wl = smem;                                                             // [wave][KL][MT] blocks
    f32x4 *red = reinterpret_cast<f32x4 *>(smem + NWV * KL * MT * kFragBytes);            // [wave][ST][64]
    unsigned char *tiles = reinterpret_cast<unsigned char *>(red + NWV * ST * kWave);     // gates, c, dout tiles
    unsigned char *const stc = tiles + BT * GROW, *const std_ = stc + BT * SROW;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int q = lane >> 4, n = lane & 15;
    const int KSB = p.KSB, H = p.H, B = p.B, T_ = p.T;

    // ---- placement: whole teams on one XCD (hardware deals workgroup i to XCD i % 8), teams spread evenly ------
    const int n_groups = p.n_rec * p.n_bt;   // (the groups of the second recurrence behind those of the first)
    const int tpg = p.n_ht / V, teams = n_groups * tpg, tpx = (teams + kNumXcd - 1) / kNumXcd;
    const int slot = blockIdx.x / kNumXcd, id = (int)(blockIdx.x % kNumXcd) * tpx + slot / V;
    if (slot / V >= tpx || id >= teams) return;
    check_xcd_placement(p.hdr);
    const int g = id / tpg, team = id % tpg, mem = slot % V, j = team * V + mem;
    const bool second = g >= p.n_bt;
    const int u0 = j * HT, b0 = p.b_base + (second ? g - p.n_bt : g) * BT;
    const T *dout = static_cast<const T *>(second ? p.dout2 : p.dout);
    const T *ifgo = static_cast<const T *>(second ? p.ifgo2 : p.ifgo);
    const T *cell = static_cast<const T *>(second ? p.cell2 : p.cell);
    T *d_ifgo = static_cast<T *>(second ? p.d_ifgo2 : p.d_ifgo);
    const T *Wh = static_cast<const T *>(second ? p.Wh2 : p.Wh);

    // ---- Wh[k-part, team units]^T, gathered: fragment (unit tile v, k-step ks = (mem KW + ki) 4 + wave): lane (q, n) holds
    // row n = unit team*16*MT + 16 v + n and k = ks*KSTEP + q*EPL + e, e < EPL, with k = 4 * source unit + gate
    u32x4 wreg[KR][MT];
    const int ks0 = mem * NWV * KW + wave;
#pragma unroll
    for (int ki = 0; ki < KW; ++ki)
#pragma unroll
        for (int v = 0; v < MT; ++v) {
            const int k0 = (ks0 + NWV * ki) * E::KSTEP + q * E::EPL;
            const bool inside = k0 < 4 * H;   // (4H is a multiple of EPL)
            const T *src = Wh + (size_t)((inside ? k0 : 0) >> 2) * H + team * V * HT + v * 16 + n;
            T tmp[E::EPL];
#pragma unroll
            for (int e = 0; e < E::EPL; ++e) tmp[e] = src[((size_t)(e & 3) * H + (e >> 2)) * H];
            u32x4 f = *reinterpret_cast<u32x4 *>(tmp);
            if (!inside) f = u32x4{0u, 0u, 0u, 0u};
            const int k = reg_of(ki);
            if (in_lds(ki)) {
                *reinterpret_cast<u32x4 *>(wl + ((wave * KL + ki * KL / KW) * MT + v) * kFragBytes + lane * 16) = f;
            } else if (k < ACC_STEPS) {   // (whole 4-register tuples in the half that they are used from)
                asm volatile("" : "+a"(f));
                wreg[k][v] = f;
            } else {
                asm volatile("" : "+v"(f));
                wreg[k][v] = f;
            }
        }

    // ---- this lane's cells: units u0 + 16 ut + 4q .. + 3, row 16 ci + n -------------
    const size_t BH = (size_t)B * H, B4H = (size_t)B * 4 * H;
    const int ut = wave % UT, ci = wave / UT;
    const int b = b0 + ci * 16 + n;
    const bool mine = ci < NT, valid = mine && b < B;
    // (H > 2048: few rows cost nothing, and the other bound 0.6 % of a step with 64 rows)
    const bool live = mine && ci * 16 + n < (UT > 1 ? rows_computed(B - b0) : B - b0);
    const size_t off_h = valid ? (size_t)b * H + u0 + 16 * ut + 4 * q : (size_t)b0 * H + u0;
    f32x4 dc_state = {0.f, 0.f, 0.f, 0.f}, dh_rec = {0.f, 0.f, 0.f, 0.f};
    u32x2 c1v = {0u, 0u};   // cell[t + 1] of the four units
    auto halves = [](u32x2 v) { return f32x4{E::to_f32(reinterpret_cast<T *>(&v)[0]), E::to_f32(reinterpret_cast<T *>(&v)[1]),
                                             E::to_f32(reinterpret_cast<T *>(&v)[2]), E::to_f32(reinterpret_cast<T *>(&v)[3])}; };
    auto packed = [](f32x4 v) {
        T o[4] = {E::from_f32(v[0]), E::from_f32(v[1]), E::from_f32(v[2]), E::from_f32(v[3])};
        return *reinterpret_cast<u32x2 *>(o);
    };
    if (valid) {
        dh_rec = halves(*reinterpret_cast<const u32x2 *>(static_cast<const T *>(second ? p.dh2 : p.dh) + off_h));
        dc_state = halves(*reinterpret_cast<const u32x2 *>(static_cast<const T *>(second ? p.dc2 : p.dc) + off_h));
        c1v = *reinterpret_cast<const u32x2 *>(cell + (size_t)T_ * BH + off_h);
    }
    const int goff = (ci * 16 + n) * GROW + (16 * ut + 4 * q) * E::BYTES, soff = (ci * 16 + n) * SROW + (16 * ut + 4 * q) * E::BYTES;
    const unsigned xslot = (unsigned)n_groups * NT * p.KSBP * kFragBytes, xgrp = (unsigned)g * NT * p.KSBP * kFragBytes;
    const XchgGlobal xch(p.xbuf, 2u * xslot);
    const unsigned x_off = mine ? xgrp + (unsigned)(ci * p.KSBP * kFragBytes + frag_offset<T>(n, (u0 + 16 * ut + 4 * q) * 4)) : 0u;
    int *grp_flags = p.flags + (size_t)g * p.flag_stride, *team_flags = p.team_flags + (size_t)g * p.flag_stride + team * V;

    // partial sums in the workspace: [receiver][sender][UT][NT][64] f32x4, one set (a sender passes the next step's group
    // barrier only after the receiver published that step, i.e. after it read this one)
    constexpr unsigned kSetBytes = UT * NT * kFragBytes;
    const XchgGlobal part(p.partials, (unsigned)(n_groups * p.n_ht) * V * kSetBytes);
    const unsigned part_team = (unsigned)(g * p.n_ht + team * V) * V * kSetBytes;
    auto part_to = [&](int v, int i) {   // unit tile v of the team is tile v % UT of member v / UT
        return part_team + (unsigned)((v / UT) * V + mem) * kSetBytes + (unsigned)((v % UT) * NT + i) * kFragBytes;
    };
    const unsigned part_mine = part_team + (unsigned)mem * V * kSetBytes + (unsigned)(ut * NT + ci) * kFragBytes;

    // ---- tile I/O (see above); the same (instruction, lane) -> slot map drains the gates tile ------------------
    constexpr int SPRG = GROW / 16, SPRS = SROW / 16;
    constexpr int NG = (BT * SPRG + kWave - 1) / kWave, NS = (BT * SPRS + kWave - 1) / kWave;
    constexpr int DT = (NG + 2 * NS + NWV - 1) / NWV;
    unsigned g_off[DT];
    bool g_ok[DT];
    const size_t tile_org = (size_t)b0 * 4 * H + u0, state_org = (size_t)b0 * H + u0;
    const unsigned g_bytes = (unsigned)((size_t)BT * 4 * H * E::BYTES), s_bytes = (unsigned)((size_t)BT * H * E::BYTES);
    auto kind_of = [&](int i) { const int w = wave + NWV * i; return w < NG ? 0 : w < NG + NS ? 1 : w < NG + 2 * NS ? 2 : 3; };
#pragma unroll
    for (int i = 0; i < DT; ++i) {
        const int w = wave + NWV * i, kind = kind_of(i);
        const int wi = kind == 0 ? w : kind == 1 ? w - NG : w - NG - NS, sl = wi * kWave + lane;
        const int spr = kind == 0 ? SPRG : SPRS, row = sl / spr, idx = sl % spr;
        g_ok[i] = kind < 3 && sl < BT * spr && idx < (kind == 0 ? 4 : 1) * PPSEG && b0 + row < B;
        g_off[i] = !g_ok[i] ? 0u : kind == 0 ? (unsigned)(((size_t)row * 4 * H + (size_t)(idx / PPSEG) * H + (idx % PPSEG) * E::EPL) * E::BYTES)
                                             : (unsigned)(((size_t)row * H + idx * E::EPL) * E::BYTES);
    }
    const unsigned tiles_addr = (unsigned)(size_t)((FASTLSTM_LDS_PTR unsigned char *)tiles);
    auto rsrc_of = [](const T *base, unsigned bytes) {
        const unsigned long long a = reinterpret_cast<unsigned long long>(uniform_ptr(base));
        return u32x4{(unsigned)a, (unsigned)(a >> 32) & 0xffffu, bytes, 0x00020000u};
    };
    auto request_tiles = [&](int t) {
        if (t < 0) return;
        const u32x4 rg = rsrc_of(ifgo + (size_t)t * B4H + tile_org, g_bytes);
        const u32x4 rc = rsrc_of(cell + (size_t)t * BH + state_org, s_bytes);
        const u32x4 rd = rsrc_of(dout + (size_t)t * BH + state_org, s_bytes);
        const unsigned base = (unsigned)uniform_int((int)tiles_addr);
#pragma unroll
        for (int i = 0; i < DT; ++i) {
            const int w = wave + NWV * i, kind = kind_of(i);
            if (kind == 0) {
                if (g_ok[i]) dma_block_asm<false>(rg, base + w * kFragBytes, g_off[i], 0u);
            } else if (kind == 1) {
                if (g_ok[i]) dma_block_asm<false>(rc, base + BT * GROW + (w - NG) * kFragBytes, g_off[i], 0u);
            } else if (kind == 2) {
                if (g_ok[i]) dma_block_asm<false>(rd, base + BT * GROW + BT * SROW + (w - NG - NS) * kFragBytes, g_off[i], 0u);
            }
        }
    };
    auto tile_to_global = [&](int t) {
        const __amdgpu_buffer_rsrc_t rg = __builtin_amdgcn_make_buffer_rsrc(d_ifgo + (size_t)t * B4H + tile_org, 0, g_bytes, 0x00020000);
#pragma unroll
        for (int i = 0; i < DT; ++i)
            if (kind_of(i) == 0 && g_ok[i])
                __builtin_amdgcn_raw_buffer_store_b128(
                    *reinterpret_cast<const u32x4 *>(tiles + (size_t)(wave + NWV * i) * kFragBytes + lane * 16), rg, g_off[i], 0, 0);
    };
    request_tiles(T_ - 1);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();

    for (int s = 0; s < T_; ++s) {
        const int t = T_ - 1 - s;
        const unsigned xs = (unsigned)(s & 1) * xslot;

        // ---- point-wise gate backward of this lane's cells --------------------------
        if (mine) {
            u32x2 d[4] = {};   // [gate]: the four units
            if (live) {   // (us per step with rows past the batch masked and so: 4 rows, H = 1280 5.6 -> 4.5, H = 2048 6.5 -> 5.2)
                const unsigned char *gl_ = tiles + goff;
                const f32x4 pi = halves(*reinterpret_cast<const u32x2 *>(gl_)), pf = halves(*reinterpret_cast<const u32x2 *>(gl_ + GSEG));
                const f32x4 pg = halves(*reinterpret_cast<const u32x2 *>(gl_ + 2 * GSEG)), po = halves(*reinterpret_cast<const u32x2 *>(gl_ + 3 * GSEG));
                const u32x2 c0v = *reinterpret_cast<const u32x2 *>(stc + soff);
                const f32x4 c0 = halves(c0v), c1 = halves(c1v), dh = dh_rec + halves(*reinterpret_cast<const u32x2 *>(std_ + soff));
                f32x4 di, df, dg, do_;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float si = sigmoidf_<false>(pi[e]), sf = sigmoidf_<false>(pf[e]), tg = tanhf_<false>(pg[e]), so = sigmoidf_<false>(po[e]);
                    const float tc = tanhf_<false>(c1[e]);
                    const float dc1 = dc_state[e] + dh[e] * so * (1.f - tc * tc);
                    do_[e] = dh[e] * tc * so * (1.f - so);
                    df[e] = dc1 * c0[e] * sf * (1.f - sf);
                    di[e] = dc1 * tg * si * (1.f - si);
                    dg[e] = dc1 * si * (1.f - tg * tg);
                    dc_state[e] = dc1 * sf;
                }
                c1v = c0v;   // c_{t-1} is the next step's c_t
                d[0] = packed(di);
                d[1] = packed(df);
                d[2] = packed(dg);
                d[3] = packed(do_);
#pragma unroll
                for (int gt = 0; gt < 4; ++gt) *reinterpret_cast<u32x2 *>(tiles + goff + gt * GSEG) = d[gt];
                // exchange copy: k = (unit, gate 0..3): 16 consecutive k of the lane, 8 per operand-block lane
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const unsigned if0 = __builtin_amdgcn_perm(d[1][h], d[0][h], 0x05040100u), if1 = __builtin_amdgcn_perm(d[1][h], d[0][h], 0x07060302u);
                    const unsigned go0 = __builtin_amdgcn_perm(d[3][h], d[2][h], 0x05040100u), go1 = __builtin_amdgcn_perm(d[3][h], d[2][h], 0x07060302u);
                    xch.store16(xs + x_off + h * 256u, u32x4{if0, go0, if1, go1});
                }
            }
        }
        publish_version(grp_flags + j, s + 1);   // waits for the stores, workgroup barrier, raises the flag
        tile_to_global(t);
        request_tiles(t - 1);   // (this lane's slots of the gates tile are read, the others before the barrier)
        if (wave == 0) wait_versions(grp_flags, p.n_ht, s + 1, p.hdr, p.spin_limit, g, s);
        __syncthreads();

        // ---- partial dh_rec(team units, rows) = Wh[k-part, team units]^T . d_ifgo[t](rows, k-part)^T ----
        u32x4 ring[R], wf[4];
        auto request = [&](int bl) {   // (past KSB: zero weights times some block)
            const int ks = min(ks0 + NWV * (bl % KW), KSB - 1);
            ring[bl % R] = xch.load16(lane * 16u, xs + xgrp + (unsigned)((bl / KW) * p.KSBP + ks) * kFragBytes);
        };
        auto read_weights = [&](int l, int half) {   // four tiles at a time
#pragma unroll
            for (int a = 0; a < 4; ++a)
                wf[a] = *reinterpret_cast<const u32x4 *>(wl + ((wave * KL + l) * MT + half * 4 + a) * kFragBytes + lane * 16);
        };
#pragma unroll
        for (int bl = 0; bl < R; ++bl) request(bl);
        if constexpr (KL > 0) read_weights(0, 0);
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            f32x4 acc[MT];
            static_for<0, KW>([&](auto kc) __attribute__((always_inline)) {
                constexpr int ki = decltype(kc)::value, l = ki * KL / KW;
                constexpr bool halves_ = KL > 0 && MT == 8;   // the upper tiles of a k-step in LDS follow behind the next k-step
                const int bl = i * KW + ki;
                if constexpr (in_lds(ki)) {
#pragma unroll
                    for (int a = 0; a < 4; ++a) mfma_resident<T, false, ki == 0>(acc[a], wf[a], ring[bl % R]);
                    if constexpr (halves_) read_weights(l, 1);
                    else if (i + 1 < NT || l + 1 < KL) read_weights((l + 1) % (KL > 0 ? KL : 1), 0);
                } else {
#pragma unroll
                    for (int a = 0; a < MT; ++a) {
                        if (halves_ && ki == 1 && a >= 4) mfma_resident<T, (reg_of(ki) < ACC_STEPS), true>(acc[a], wreg[reg_of(ki)][a], ring[bl % R]);
                        else mfma_resident<T, (reg_of(ki) < ACC_STEPS), ki == 0>(acc[a], wreg[reg_of(ki)][a], ring[bl % R]);
                    }
                    if constexpr (halves_ && in_lds(ki - 1)) {
#pragma unroll
                        for (int a = 4; a < MT; ++a) mfma_resident<T, false, false>(acc[a], wf[a - 4], ring[(bl - 1) % R]);
                        if (i + 1 < NT || l + 1 < KL) read_weights((l + 1) % KL, 0);
                        if (bl - 1 + R < NB) request(bl - 1 + R);
                    }
                }
                if (!(halves_ && in_lds(ki)) && bl + R < NB) request(bl + R);
                __builtin_amdgcn_sched_barrier(0);   // (the order above is the schedule)
            });
            mfma_results(acc);
#pragma unroll
            for (int a0 = 0; a0 < MT; a0 += ST) {
#pragma unroll
                for (int a = 0; a < ST; ++a) red[(wave * ST + a) * kWave + lane] = acc[a0 + a];
                __syncthreads();
#pragma unroll
                for (int tl = 0; tl < ST; tl += NWV) {   // this wave: tile a0 + tl + wave
                    f32x4 sum = red[(tl + wave) * kWave + lane];
#pragma unroll
                    for (int w = 1; w < NWV; ++w) sum += red[(w * ST + tl + wave) * kWave + lane];
                    // (an ordinary store: the team shares one XCD, whose L2 the receivers' device-scope loads read)
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, sum), part.rsrc, lane * 16u, part_to(a0 + tl + wave, i), 0);
                }
                if (i + 1 < NT || a0 + ST < MT) __syncthreads();   // `red` is read
            }
        }

        // ---- the team's exchange: every member gets the others' sums for its 16 units, adds in member order ----
        publish_version(team_flags + mem, s + 1);
        if (mine) {
            wait_versions(team_flags, V, s + 1, p.hdr, p.spin_limit, g, s);
            u32x4 got[V];
#pragma unroll
            for (int v = 0; v < V; ++v) got[v] = part.load16(lane * 16u, part_mine + (unsigned)v * kSetBytes);
            dh_rec = __builtin_bit_cast(f32x4, got[0]);
#pragma unroll
            for (int v = 1; v < V; ++v) dh_rec += __builtin_bit_cast(f32x4, got[v]);
        }
    }
    if (valid) {
        *reinterpret_cast<u32x2 *>(static_cast<T *>(second ? p.dh2 : p.dh) + off_h) = packed(dh_rec);
        *reinterpret_cast<u32x2 *>(static_cast<T *>(second ? p.dc2 : p.dc) + off_h) = packed(dc_state);
    }
}

}  // namespace fastlstm
