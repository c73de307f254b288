// Persistent reverse-time kernel for 16-bit elements and 2048 < H <= 4096: weights on the CU for the whole launch, as in
// lstm_fwd_big_kernel, and the product split over K among teams, as in lstm_bwd_wide_split_kernel.  Same mathematics and
// results as lstm_bwd_persistent_kernel (which replaces fastlstm/kernels.py:1201-1409); the sums over K are taken in
// another order.
//
// A team of 4 neighbouring workgroups owns 64 units; member m keeps the weights of all of them for the m-th part of K = 4H
// (up to 512 KiB: three quarters in registers, the rest in LDS), reads that quarter of d_ifgo[t] and sends every member
// its partial sums through the workspace (4 KiB for 64 rows).  The K loop is that of lstm_fwd_big_kernel: 4 unit tiles x KW
// k-steps per wave, batch tile after batch tile, a ring of operand blocks in registers, the waves' sums added in LDS behind
// each tile.
//  * the inputs of the next step come in with LDS-direct loads, requested before the wait for the group's flags;
//  * wave i takes the cells of batch tile i: lane (q, n) units 4q .. 4q + 3 of row n, which is what a lane holds of a product tile.
// What bounds a step: the operand blocks (512 KiB per CU at H = 4096 and 64 rows; without teams 2 MiB) and the two exchanges.
// us per step of lstm_bwd_stream_kernel and here: H = 4096, 64 rows 33.6 -> 12.8, 16 rows 21.1 -> 6.7; H = 3072, 32 rows
// 16.8 -> 7.2; H = 2560, 64 rows 22.6 -> 9.5.
// Requirements (host): H a multiple of 64, workgroup ids dealt to the XCDs in turn, all teams co-resident.
#pragma once
#include <type_traits>

#include "recurrent_fwd_big.hpp"

namespace fastlstm {

constexpr int kBigTeam = 4;

template <typename T, int KW, int NT>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(1, 1))) void lstm_bwd_big_kernel(const BwdStreamParams p) {
    using E = Elem<T>;
    static_assert(E::BYTES == 2, "16-bit element types");
    constexpr int NWV = 4, MT = 4, V = kBigTeam;
    constexpr int KR = KW < kBigRegSteps ? KW : kBigRegSteps, KL = KW - KR;
    constexpr int HT = 16, BT = 16 * NT;
    constexpr int NB = KW * NT, R = big_ring(KW);
    constexpr int GSEG = HT * E::BYTES, GROW = 4 * GSEG + 16, SROW = GSEG + 16, PPSEG = GSEG / 16;
    constexpr auto in_lds = [](int ki) { return (ki + 1) * KL / KW > ki * KL / KW; };

    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    unsigned char *wl = smem;                                                             // [wave][KL][MT] blocks
    f32x4 *red = reinterpret_cast<f32x4 *>(smem + NWV * KL * MT * kFragBytes);            // [wave][MT][64]
    unsigned char *tiles = reinterpret_cast<unsigned char *>(red + NWV * MT * kWave);     // gates, c, dout tiles
    unsigned char *const stc = tiles + BT * GROW, *const std_ = stc + BT * SROW;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int q = lane >> 4, n = lane & 15;
    const int KSB = p.KSB, H = p.H, B = p.B, T_ = p.T;

    // ---- placement: whole teams on one XCD (hardware deals workgroup i to XCD i % 8), teams spread evenly ------
    const int teams = p.n_ht / V, tpx = (teams + kNumXcd - 1) / kNumXcd;
    const int slot = blockIdx.x / kNumXcd, team = (int)(blockIdx.x % kNumXcd) * tpx + slot / V;
    if (slot / V >= tpx || team >= teams) return;
    check_xcd_placement(p.hdr);
    const int mem = slot % V, j = team * V + mem;
    const int u0 = j * HT, b0 = p.b_base;
    const T *dout = static_cast<const T *>(p.dout);
    const T *ifgo = static_cast<const T *>(p.ifgo);
    const T *cell = static_cast<const T *>(p.cell);
    T *d_ifgo = static_cast<T *>(p.d_ifgo);
    const T *Wh = static_cast<const T *>(p.Wh);

    // ---- Wh[k-part, team units]^T, gathered: fragment (unit tile v, k-step ks = (mem KW + ki) 4 + wave): lane (q, n) holds
    // row n = unit team*64 + 16 v + n and k = ks*KSTEP + q*EPL + e, e < EPL, with k = 4 * source unit + gate
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
            const int k = ki - ki * KL / KW;
            if (in_lds(ki)) {
                *reinterpret_cast<u32x4 *>(wl + ((wave * KL + ki * KL / KW) * MT + v) * kFragBytes + lane * 16) = f;
            } else if (k < kBigAccSteps) {   // (whole 4-register tuples in the half that they are used from)
                asm volatile("" : "+a"(f));
                wreg[k][v] = f;
            } else {
                asm volatile("" : "+v"(f));
                wreg[k][v] = f;
            }
        }

    // ---- this lane's cells: units u0 + 4q .. + 3, row 16 wave + n -------------
    const size_t BH = (size_t)B * H, B4H = (size_t)B * 4 * H;
    const int b = b0 + wave * 16 + n;
    const bool mine = wave < NT, valid = mine && b < B;
    const size_t off_h = valid ? (size_t)b * H + u0 + 4 * q : (size_t)b0 * H + u0;
    f32x4 dc_state = {0.f, 0.f, 0.f, 0.f}, dh_rec = {0.f, 0.f, 0.f, 0.f};
    u32x2 c1v = {0u, 0u};   // cell[t + 1] of the four units
    auto halves = [](u32x2 v) { return f32x4{E::to_f32(reinterpret_cast<T *>(&v)[0]), E::to_f32(reinterpret_cast<T *>(&v)[1]),
                                             E::to_f32(reinterpret_cast<T *>(&v)[2]), E::to_f32(reinterpret_cast<T *>(&v)[3])}; };
    auto packed = [](f32x4 v) {
        T o[4] = {E::from_f32(v[0]), E::from_f32(v[1]), E::from_f32(v[2]), E::from_f32(v[3])};
        return *reinterpret_cast<u32x2 *>(o);
    };
    if (valid) {
        dh_rec = halves(*reinterpret_cast<const u32x2 *>(static_cast<const T *>(p.dh) + off_h));
        dc_state = halves(*reinterpret_cast<const u32x2 *>(static_cast<const T *>(p.dc) + off_h));
        c1v = *reinterpret_cast<const u32x2 *>(cell + (size_t)T_ * BH + off_h);
    }
    const int goff = (wave * 16 + n) * GROW + 4 * q * E::BYTES, soff = (wave * 16 + n) * SROW + 4 * q * E::BYTES;
    const unsigned xslot = (unsigned)NT * p.KSBP * kFragBytes;
    const XchgGlobal xch(p.xbuf, 2u * xslot);
    const unsigned x_off = mine ? (unsigned)(wave * p.KSBP * kFragBytes + frag_offset<T>(n, (u0 + 4 * q) * 4)) : 0u;
    int *grp_flags = p.flags, *team_flags = p.team_flags;

    // partial sums in the workspace: [receiver][sender][NT][64] f32x4, one set (a sender passes the next step's group
    // barrier only after the receiver published that step, i.e. after it read this one)
    constexpr unsigned kSetBytes = NT * kFragBytes;
    const XchgGlobal part(p.partials, (unsigned)p.n_ht * V * kSetBytes);
    const unsigned part_to = (unsigned)((team * V + wave) * V + mem) * kSetBytes;   // wave w adds up and sends unit tile w
    const unsigned part_mine = (unsigned)j * V * kSetBytes;

    // ---- tile I/O as in lstm_bwd_wide_split_kernel ------------------
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
            if (valid) {
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
        if (wave == 0) wait_versions(grp_flags, p.n_ht, s + 1, p.hdr, p.spin_limit, 0, s);
        __syncthreads();

        // ---- partial dh_rec(team units, rows) = Wh[k-part, team units]^T . d_ifgo[t](rows, k-part)^T ----
        u32x4 ring[R], wf[MT];
        auto request = [&](int bl) {   // (past KSB: zero weights times some block)
            const int ks = min(ks0 + NWV * (bl % KW), KSB - 1);
            ring[bl % R] = xch.load16(lane * 16u, xs + (unsigned)((bl / KW) * p.KSBP + ks) * kFragBytes);
        };
        auto read_weights = [&](int l) {
#pragma unroll
            for (int a = 0; a < MT; ++a)
                wf[a] = *reinterpret_cast<const u32x4 *>(wl + ((wave * KL + l) * MT + a) * kFragBytes + lane * 16);
        };
#pragma unroll
        for (int bl = 0; bl < R; ++bl) request(bl);
        if constexpr (KL > 0) read_weights(0);
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            f32x4 acc[MT];
            static_for<0, KW>([&](auto kc) __attribute__((always_inline)) {
                constexpr int ki = decltype(kc)::value, l = ki * KL / KW;
                const int bl = i * KW + ki;
                if constexpr (in_lds(ki)) {
#pragma unroll
                    for (int a = 0; a < MT; ++a) mfma_resident<T, false, ki == 0>(acc[a], wf[a], ring[bl % R]);
                    if (i + 1 < NT || l + 1 < KL) read_weights((l + 1) % (KL > 0 ? KL : 1));
                } else {
#pragma unroll
                    for (int a = 0; a < MT; ++a) mfma_resident<T, (ki - l < kBigAccSteps), ki == 0>(acc[a], wreg[ki - l][a], ring[bl % R]);
                }
                if (bl + R < NB) request(bl + R);
                __builtin_amdgcn_sched_barrier(0);   // (the order above is the schedule)
            });
            mfma_results(acc);
#pragma unroll
            for (int a = 0; a < MT; ++a) red[(wave * MT + a) * kWave + lane] = acc[a];
            __syncthreads();
            f32x4 sum = red[wave * kWave + lane];
#pragma unroll
            for (int w = 1; w < NWV; ++w) sum += red[(w * MT + wave) * kWave + lane];
            // (an ordinary store: the team shares one XCD, whose L2 the receivers' device-scope loads read)
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, sum), part.rsrc, part_to + lane * 16u, i * kFragBytes, 0);
            if (i + 1 < NT) __syncthreads();   // `red` is read
        }

        // ---- the team's exchange: every member gets the others' sums for its 16 units, adds in member order ----
        publish_version(team_flags + j, s + 1);
        if (mine) {
            wait_versions(team_flags + team * V, V, s + 1, p.hdr, p.spin_limit, 0, s);
            u32x4 got[V];
#pragma unroll
            for (int v = 0; v < V; ++v) got[v] = part.load16(lane * 16u, part_mine + (unsigned)v * kSetBytes + wave * kFragBytes);
            dh_rec = __builtin_bit_cast(f32x4, got[0]);
#pragma unroll
            for (int v = 1; v < V; ++v) dh_rec += __builtin_bit_cast(f32x4, got[v]);
        }
    }
    if (valid) {
        *reinterpret_cast<u32x2 *>(static_cast<T *>(p.dh) + off_h) = packed(dh_rec);
        *reinterpret_cast<u32x2 *>(static_cast<T *>(p.dc) + off_h) = packed(dc_state);
    }
}

}  // namespace fastlstm
