// fp32 products on the bf16 matrix units, at the precision of fp32:
//     C[m][n] = sum_k A(m,k) * B(n,k)   [+ bias0[n] + bias1[n]]
// the contraction of gemm.hpp for every shape, with each operand K-contiguous or K-major.
//
// An fp32 number is the exact sum of three bf16 numbers: the nearest one, the one nearest to what is left, and the rest, which is at
// most half a step of the second and fits 8 bits.  The products of two such sums go to v_mfma_f32_32x32x16_bf16, which runs at 16 times
// the rate of the fp32 MFMA, and are added in fp32, the small ones first.
//  * K > 64: six of the nine.  Left out are the three smallest, each below 2^-24 of the largest and of either sign.  (Parts that are cut
//    off instead of rounded all have the number's sign: results came out 4e-8 low, and x.Wx^T of K = 4096 terms of one sign, where the
//    MFMA drops what lies far below the running sum, 1e-5.)  Six roundings of the sum per 16 terms: fewer than v_mfma_f32_16x16x4_f32's.
//  * K <= 64: all nine, the eight small ones in sums of their own, so that the large ones are rounded once per 16 terms.
//  Error against 64 bits (2-norm over that of the result) in tiles of v_mfma_f32_16x16x4_f32 and here, x.Wx^T: K = 1 2.5e-8, 2.5e-8; 2 3.1e-8,
//  2.6e-8; 8 5.4e-8, 2.8e-8; 64 1.4e-7, 4.9e-8; 65 1.5e-7, 1.2e-7; 1024 5.7e-7, 4.9e-7; 16384 2.3e-6, 2.1e-6; terms of one sign: K = 64 1.2e-7,
//  4.1e-8; 1024 4.7e-7, 3.2e-7; 16384 1.9e-6, 1.2e-6.
//  * what bounds it: the matrix units (16-bit products at 1.65 PFLOP/s are what they reach on random data; that is 275 here) and, next
//    to them, the LDS (half of its cycles) and the conversions, which lie among the MFMAs, three vector instructions to each (behind
//    them instead: 205).  TFLOP/s of fp32, on the fp32 MFMA and here: M = 8192, N = 8192, K = 2048 x.Wx^T 136 -> 235, d.Wx 136 -> 234, weight
//    gradients 133 -> 235; M = 16384, I = H = 1024 weight gradients 131 -> 229; M = 8192, I = 512, H = 1024 97 -> 205.
//  * small numbers: the operands are taken times 2^24, which makes the last bit of the least fp32 number a normal bf16 number, and the
//    sums times 2^-48.  (Without that the parts of numbers below 2^-110 lose bits: of an operand of 1e-36 the products were off by 6e-5, of
//    1e-38 by 1e-2.)  A sum beyond 2^80, or one with an operand beyond 2^104, is dealt with as an infinity:
//  * infinities: what is left of one is no number, as of a finite one that is rounded to one.  Sums that are not finite are taken from
//    the fp32 MFMA, 32 x 32 results at a time (behind the main loop): they come out as they do there, and the sums beside them keep their
//    bits.  (One infinity in x or d, T*B = 16384, I = H = 1024: x.Wx^T 0.7 -> 1.1 ms, weight gradients 1.2 -> 3.8; a NaN costs nothing.)
//  * staging: global -> registers, a k-tile ahead of the conversion -> three bf16 planes in LDS, in MFMA operand order, double
//    buffered; one barrier per k-tile of 16.  Half of the waves stage A, the others B.
//  * a K-major operand is transposed on the way: a thread loads 4 k x 4 rows and stores 4 rows x 4 k; rows are stored at
//    row ^ (row tile & 3), which spreads these stores over the banks.
#pragma once
#include <type_traits>

#include "common.hpp"
#include "gemm.hpp"
#include "recurrent_parts.hpp"

namespace fastlstm {

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kF32BK = 16;   // k of a stage: one MFMA k-step
constexpr int kF32AllK = 64;   // up to this K all nine products are added (see above)
constexpr float kF32Scale = 0x1p24f, kF32Unscale = 0x1p-48f;   // of an operand, of a product of two

struct GemmF32Params {
    GemmParams p;
    // a second product of the same A (the weight gradients): its column tiles follow the first one's
    const void *B2;
    void *C2;
    float *Cpart2;
    int N2, ldb2, ldc2, tiles_n1;   // N2 = 0: none
    float *db_part;                 // [splits][M]: sums of A over k (K-major A), or nullptr
};

template <int BM, int BN, int WM, int WN> struct F32Tile {
    static constexpr int WAVES = WM * WN, THREADS = WAVES * kWave, TA = BM / WM / 32, TB = BN / WN / 32;
    static constexpr int A_BYTES = BM / 32 * 3 * kFragBytes, STAGE = A_BYTES + BN / 32 * 3 * kFragBytes, LDS_BYTES = 2 * STAGE;
    static_assert(BM == BN && BM == THREADS / 2, "half of the threads stage 16 elements each of either operand");
};

// The largest magnitude met (a NaN does not count).
__device__ __forceinline__ void max_magnitude(float &top, float a, float b) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm("v_max3_f32 %0, %0, abs(%1), abs(%2)" : "+v"(top) : "v"(a), "v"(b));
#endif
}

// Two values, rounded to bf16 and packed in order; and the values of such a pair.
__device__ __forceinline__ unsigned bf16_pair(float a, float b) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{a, b}, bf16x2));
}
__device__ __forceinline__ float pair_first(unsigned p) { return __builtin_bit_cast(float, p << 16); }
__device__ __forceinline__ float pair_second(unsigned p) { return __builtin_bit_cast(float, p & 0xffff0000u); }

// Four values -> their three bf16 parts, packed in order.
struct F32Planes {
    float r[4];
    u32x2 hi, mid, lo;
    __device__ __forceinline__ void cut(const f32x4 v, float &top) {
        const float x[4] = {v[0] * kF32Scale, v[1] * kF32Scale, v[2] * kF32Scale, v[3] * kF32Scale};
        max_magnitude(top, x[0], x[1]);
        max_magnitude(top, x[2], x[3]);
        split(x, hi);
    }
    __device__ __forceinline__ void pack() {
        split(r, mid);
        lo = u32x2{bf16_pair(r[0], r[1]), bf16_pair(r[2], r[3])};
    }
    __device__ __forceinline__ void split(const float *x, u32x2 &part) {   // x -> its first part, and what is left of it in r
        part = u32x2{bf16_pair(x[0], x[1]), bf16_pair(x[2], x[3])};
#pragma unroll
        for (int e = 0; e < 4; e += 2) {
            r[e] = x[e] - pair_first(part[e / 2]);
            r[e + 1] = x[e + 1] - pair_second(part[e / 2]);
        }
    }
};

// One operand of a tile as a staging thread sees it: rows r0 .. r0 + BM - 1, 16 elements per thread and k-tile.
template <int BM> struct F32Stager {
    const float *base;   // at row r0 (K-major: column r0)
    int ld, rows, ke;    // rows left from r0 on; end of the k range
    int th;              // 0 .. BM - 1
    template <bool KM> __device__ __forceinline__ void load(int k0, f32x4 (&v)[4]) const {
        const bool whole = k0 + kF32BK <= ke;
        if constexpr (!KM) {   // piece i: row th / 4 + BM / 4 * i, k (th % 4) * 4 ..
            const int k = k0 + (th & 3) * 4;
            unsigned at[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) at[i] = (unsigned)min(th / 4 + BM / 4 * i, rows - 1) * (unsigned)ld + (th & 3) * 4;
            if (whole) {
#pragma unroll
                for (int i = 0; i < 4; ++i) __builtin_memcpy(&v[i], base + k0 + at[i], 16);
            } else {   // (clamped, so that all loads are under way together; what lies past the end is dropped behind them)
                const int last = ke - 1 - k0;
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[i][e] = base[k0 + at[i] - (th & 3) * 4 + min((th & 3) * 4 + e, last)];
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[i][e] = k + e < ke ? v[i][e] : 0.f;
            }
        } else {               // piece i: k (th / (BM / 4)) * 4 + i, rows (th % (BM / 4)) * 4 ..
            const int c = th % (BM / 4) * 4, k = th / (BM / 4) * 4;
            const float *src = base + (size_t)k0 * ld;
            if (whole && ((rows & 3) == 0 || rows >= BM)) {   // (a piece is inside or outside as a whole; outside: rows nobody stores)
#pragma unroll
                for (int i = 0; i < 4; ++i) __builtin_memcpy(&v[i], src + ((unsigned)(k + i) * (unsigned)ld + (c < rows ? c : 0)), 16);
            } else {
                const int last = ke - 1 - k0;
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[i][e] = src[(unsigned)min(k + i, last) * (unsigned)ld + min(c + e, rows - 1)];
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[i][e] = k + i <= last ? v[i][e] : 0.f;
            }
        }
    }
    // piece i of a thread into the three planes of a stage's operand, [row tile of 32][plane][lane: k half, row][8 k], in three
    // parts that the main loop deals out among its MFMAs
    template <bool KM> __device__ __forceinline__ void store(int part, int i, unsigned char *op, const f32x4 (&v)[4], F32Planes &w, float &top) const {
        if (part == 0) {
            w.cut(KM ? f32x4{v[0][i], v[1][i], v[2][i], v[3][i]} : v[i], top);
        } else if (part == 1) {
            w.pack();
        } else {
            const int row = KM ? th % (BM / 4) * 4 + i : th / 4 + BM / 4 * i, k4 = KM ? th / (BM / 4) : th & 3;
            unsigned char *dst = op + (row >> 5) * 3 * kFragBytes + ((k4 >> 1) * 32 + ((row & 31) ^ (row >> 5 & 3))) * 16 + (k4 & 1) * 8;
            *reinterpret_cast<u32x2 *>(dst) = w.hi;
            *reinterpret_cast<u32x2 *>(dst + kFragBytes) = w.mid;
            *reinterpret_cast<u32x2 *>(dst + 2 * kFragBytes) = w.lo;
        }
    }
};

// A workgroup barrier for what went through the LDS: unlike __syncthreads it does not wait for the loads in flight.
__device__ __forceinline__ void lds_barrier() {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#endif
}

// TWO: the small products have sums of their own, so that the large ones are rounded once per 16 k instead of six times (an error
// 2.6 times smaller: fewer parts of K for the same one).  Only where the sums are split anyway: without a split tiles of 64, 128 and 256 add up
// in the same order, so that a range of rows has the bits that it has within the whole.
// ALL: nine products (K <= kF32AllK).
template <bool A_KM, bool B_KM, int BM, int BN, int WM, int WN, bool TWO, bool ALL>
__global__ __launch_bounds__(64 * WM * WN, 2) void gemm_f32_kernel(const GemmF32Params g) {
    using F = F32Tile<BM, BN, WM, WN>;
    constexpr int TA = F::TA, TB = F::TB;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN;
    GemmParams p = g.p;
    const int tiles_m = cdiv(p.M, BM), tiles_n = g.N2 ? g.tiles_n1 + cdiv(g.N2, BN) : cdiv(p.N, BN);
    int bid = blockIdx.x;
    const int split = bid / (tiles_m * tiles_n);
    bid -= split * tiles_m * tiles_n;
    // eight row tiles by all column tiles at a time, XCD-major: the workgroups of an XCD share panels through its L2
    const int lin = xcd_major_id(bid, tiles_m * tiles_n), per_group = 8 * tiles_n, first_m = lin / per_group * 8;
    const int gsz = min(tiles_m - first_m, 8);
    const int m0 = (first_m + lin % per_group % gsz) * BM, nt = lin % per_group / gsz;
    if (g.N2 && nt >= g.tiles_n1) {
        p.B = g.B2; p.C = g.C2; p.Cpart = g.Cpart2;
        p.N = g.N2; p.ldb = g.ldb2; p.ldc = g.ldc2;
    }
    const int n0 = (g.N2 && nt >= g.tiles_n1 ? nt - g.tiles_n1 : nt) * BN;
    const int kb = split * p.k_per_split, ke = min(p.K, kb + p.k_per_split), nkt = cdiv(ke - kb, kF32BK);
    const float *A = static_cast<const float *>(p.A) + (A_KM ? (size_t)m0 : (size_t)m0 * p.lda);
    const float *B = static_cast<const float *>(p.B) + (B_KM ? (size_t)n0 : (size_t)n0 * p.ldb);

    const bool stages_a = wave < F::WAVES / 2;
    const F32Stager<BM> st{stages_a ? A : B, stages_a ? p.lda : p.ldb, stages_a ? p.M - m0 : p.N - n0, ke, tid & (F::THREADS / 2 - 1)};
    const bool sums = A_KM && g.db_part && nt == 0 && stages_a;
    f32x4 dsum = {0.f, 0.f, 0.f, 0.f}, dsum16 = {0.f, 0.f, 0.f, 0.f};   // (of the last up to 16 k-tiles, of those before)

    float top = 0.f;
    f32x16 acc[TA][TB], acc2[TWO ? TA : 1][TWO ? TB : 1];
    auto clear = [&](auto &c) {
#pragma unroll
        for (auto &row : c)
#pragma unroll
            for (auto &t : row)
#pragma unroll
                for (int i = 0; i < 16; ++i) t[i] = 0.f;
    };
    clear(acc);
    clear(acc2);
    // (a function of its own for the waves of either operand: the conversions of a k-tile lie among its MFMAs)
    auto mainloop = [&](auto km) __attribute__((always_inline)) {
        constexpr bool KM = decltype(km)::value;
        f32x4 v[4];
        F32Planes w;
        auto sum = [&](int kt) {
            if (!sums) return;
            dsum += (v[0] + v[1]) + (v[2] + v[3]);
            if (kt % 16 == 15) {
                dsum16 += dsum;
                dsum = f32x4{0.f, 0.f, 0.f, 0.f};
            }
        };
        // MFMAs of the k-tile in stage kt % 2; NEXT: and k-tile kt + 1 from the registers into the other stage
        auto multiply = [&](int kt, auto next) __attribute__((always_inline)) {
            constexpr bool NEXT = decltype(next)::value;
            const unsigned char *sa = smem + (kt & 1) * F::STAGE, *sb = sa + F::A_BYTES;
            unsigned char *op = smem + (~kt & 1) * F::STAGE + (stages_a ? 0 : F::A_BYTES);
            auto frag = [&](const unsigned char *o, int tile, int plane) {
                return __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4 *>(o + (tile * 3 + plane) * kFragBytes + (lane ^ (tile & 3)) * 16));
            };
            bf16x8 fb[TB][3], fa[2][3];
#pragma unroll
            for (int s = 0; s < 3; ++s) fa[0][s] = frag(sa, wm * TA, s);
#pragma unroll
            for (int b = 0; b < TB; ++b)
#pragma unroll
                for (int s = 0; s < 3; ++s) fb[b][s] = frag(sb, wn * TB + b, s);
            // (the parts of A and B that a product takes; the twelve steps of the conversion are spread over the products of the tile)
            constexpr int pa[9] = {2, 2, 1, 2, 0, 1, 1, 0, 0}, pb[9] = {2, 1, 2, 0, 2, 1, 0, 1, 0}, P0 = ALL ? 0 : 3, NP = 9 - P0;
            constexpr auto slot_of = [](int step) { return step * NP * TA / 12; };
            int step = 0;
#pragma unroll
            for (int sl = 0; sl < NP * TA; ++sl) {
                const int a = sl / NP, i = sl % NP;
                if (i == 2 && a + 1 < TA)
#pragma unroll
                    for (int s = 0; s < 3; ++s) fa[(a + 1) & 1][s] = frag(sa, wm * TA + a + 1, s);
#pragma unroll
                for (int b = 0; b < TB; ++b) {
                    f32x16 &c = TWO && i < NP - 1 ? acc2[TWO ? a : 0][TWO ? b : 0] : acc[a][b];
                    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[b][pb[P0 + i]], fa[a & 1][pa[P0 + i]], c, 0, 0, 0);
                }
                if constexpr (NEXT)
                    for (; step < 12 && slot_of(step) == sl; ++step) st.template store<KM>(step % 3, step / 3, op, v, w, top);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        st.template load<KM>(kb, v);
        sum(0);
#pragma unroll
        for (int i = 0; i < 12; ++i) st.template store<KM>(i % 3, i / 3, smem + (stages_a ? 0 : F::A_BYTES), v, w, top);
        if (nkt > 1) st.template load<KM>(kb + kF32BK, v);
        lds_barrier();
        for (int kt = 0; kt + 1 < nkt; ++kt) {
            multiply(kt, std::true_type{});
            sum(kt + 1);
            if (kt + 2 < nkt) st.template load<KM>(kb + (kt + 2) * kF32BK, v);
            lds_barrier();
        }
        multiply(nkt - 1, std::false_type{});
    };
    if (A_KM == B_KM || stages_a) mainloop(std::bool_constant<A_KM>{});
    else mainloop(std::bool_constant<B_KM>{});
    if constexpr (TWO)
#pragma unroll
        for (int a = 0; a < TA; ++a)
#pragma unroll
            for (int b = 0; b < TB; ++b) acc[a][b] += acc2[a][b];

    // lane: row m = lane % 32 of a tile, columns 8 (i / 4) + 4 (lane / 32) + i % 4
    const int ml = lane & 31, q = lane >> 5;
    // 32 x 32 results (a, b) of this wave on the fp32 MFMA, 16 k under way at a time
    auto in_fp32 = [&](int a, int b) {
        const int m = min((wm * TA + a) * 32 + ml, p.M - m0 - 1), n = min((wn * TB + b) * 32 + ml, p.N - n0 - 1);
        f32x16 c;
#pragma unroll
        for (int i = 0; i < 16; ++i) c[i] = 0.f;
        for (int k0 = kb; k0 < ke; k0 += 16) {
            float ea[8], eb[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int k = min(k0 + 2 * i + q, ke - 1);
                ea[i] = A_KM ? A[(size_t)k * p.lda + m] : A[(size_t)m * p.lda + k];
                eb[i] = B_KM ? B[(size_t)k * p.ldb + n] : B[(size_t)n * p.ldb + k];
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const bool in = k0 + 2 * i + q < ke;
                c = __builtin_amdgcn_mfma_f32_32x32x2f32(in ? eb[i] : 0.f, in ? ea[i] : 0.f, c, 0, 0, 0);
            }
        }
        return c;
    };
    if (A_KM && g.db_part && nt == 0) {   // the threads of a column: k (th / (BM / 4)) * 4 .. + 3 of every k-tile each
        float *red = reinterpret_cast<float *>(smem);
        if (stages_a) *reinterpret_cast<f32x4 *>(red + st.th / (BM / 4) * BM + st.th % (BM / 4) * 4) = dsum + dsum16;
        __syncthreads();
        if (tid < BM && m0 + tid < p.M)
            g.db_part[(size_t)split * p.M + m0 + tid] = (red[tid] + red[BM + tid]) + (red[2 * BM + tid] + red[3 * BM + tid]);
    }

    // C leaves by rows: a wave's 32 rows go through its part of the LDS (rows padded by 16 bytes), 16 lanes store 256 bytes of a row.
    // Straight from the accumulators an instruction stores 32 bytes of every row: with few k that was most of the time.  x.Wx^T, us:
    // T*B = 40000, I = 64, H = 256 102 -> 63, H = 1024 383 -> 250; 280000, 64, 256 682 -> 453; 16384, 1024, 1024 685 -> 627.
    constexpr int CN = TB * 32, CROW = CN * 4 + 16, LPR = CN / 4, RPI = 64 / LPR;   // columns of a wave, lanes per row, rows per instruction
    static_assert(F::WAVES * 32 * CROW <= F::LDS_BYTES, "a row tile of every wave");
    const float *bias0 = static_cast<const float *>(p.bias0), *bias1 = static_cast<const float *>(p.bias1);
    const bool part = p.splits > 1;
    float *C = part ? p.Cpart + (size_t)split * p.M * p.N : static_cast<float *>(p.C);
    const int ldc = part ? p.N : p.ldc;
    unsigned char *const mine = smem + wave * 32 * CROW;
    const int n = n0 + wn * CN + lane % LPR * 4;
    f32x4 bias = {0.f, 0.f, 0.f, 0.f};
    if (bias0 && !part)
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (n + e < p.N) bias[e] = bias0[n + e] + (bias1 ? bias1[n + e] : 0.f);
    // (the last k-tile and the sums of A are read)  Products of scaled operands below 2^64 cannot overflow: a sum that is no number has a NaN among
    // its operands then, and stays one.
    const bool large = __syncthreads_or(top >= 0x1p64f);
#pragma unroll
    for (int a = 0; a < TA; ++a) {
#pragma unroll
        for (int b = 0; b < TB; ++b) {
            f32x16 c = acc[a][b];
            float zero = 0.f, most = 0.f;   // (zero: not if one of the sums is infinite or no number)
#pragma unroll
            for (int i = 0; i < 16; ++i) zero = __builtin_fmaf(c[i], 0.f, zero);
#pragma unroll
            for (int i = 0; i < 16; i += 2) max_magnitude(most, c[i], c[i + 1]);
            if (__ballot(most == __builtin_inff() || (large && zero != 0.f))) {   // (see above: those sums are taken from there, the others stay as they are)
                const f32x16 other = in_fp32(a, b);
#pragma unroll
                for (int i = 0; i < 16; ++i) c[i] = c[i] * 0.f == 0.f ? c[i] * kF32Unscale : other[i];
            } else {
                c *= kF32Unscale;
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
                *reinterpret_cast<f32x4 *>(mine + ml * CROW + (b * 32 + 8 * i + 4 * q) * 4) = f32x4{c[4 * i], c[4 * i + 1], c[4 * i + 2], c[4 * i + 3]};
        }
        __builtin_amdgcn_wave_barrier();   // (a wave's LDS accesses are done in order)
#pragma unroll
        for (int k = 0; k < 32 / RPI; ++k) {
            const int row = lane / LPR + RPI * k, m = m0 + (wm * TA + a) * 32 + row;
            const f32x4 r = *reinterpret_cast<const f32x4 *>(mine + row * CROW + lane % LPR * 16) + bias;
            if (m >= p.M || n >= p.N) continue;
            float *dst = C + (size_t)m * ldc + n;
            typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
            if (n + 3 < p.N) {   // (non-temporal: GemmParams::keep_c)
                if (part || p.keep_c) *reinterpret_cast<f32x4u *>(dst) = r;
                else __builtin_nontemporal_store(r, reinterpret_cast<f32x4u *>(dst));
            } else
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < p.N) dst[e] = r[e];
        }
        __builtin_amdgcn_wave_barrier();
    }
}

}  // namespace fastlstm
