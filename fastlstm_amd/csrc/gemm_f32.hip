// Host side of the fp32 products (gemm_f32.hpp): which tile, how many parts of K, the launch.
#include "gemm_f32.hpp"
#include "internal.hpp"

namespace fastlstm {

namespace {

template <bool A_KM, bool B_KM, int T, bool TWO, bool ALL = false> hipError_t launch_t(const GemmF32Params &g, hipStream_t s) {
    constexpr int WN = T / 64;
    using F = F32Tile<T, T, 2, WN>;
    static bool attr_set = false;
    auto kern = gemm_f32_kernel<A_KM, B_KM, T, T, 2, WN, TWO, ALL>;
    if (!attr_set) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, F::LDS_BYTES);
        if (e != hipSuccess) return e;
        attr_set = true;
    }
    const int tiles = cdiv(g.p.M, T) * (cdiv(g.p.N, T) + cdiv(g.N2, T)) * g.p.splits;
    hipLaunchKernelGGL(kern, dim3(tiles), dim3(F::THREADS), F::LDS_BYTES, s, g);
    return hipGetLastError();
}

}  // namespace

// Tile edge (256: one workgroup per CU, 128: two, 64: few tiles) and parts of K of C[M][N1 | N2]: the least time, put together from measured parts.
// A k-tile of 16 takes a 256 x 256 tile 2.2 us and two 128 x 128 tiles of a CU 1.35 us (0.7 us one alone); a tile takes 5 and 4 us
// besides (start, epilogue); partial sums are written and read back at 3.5 TB/s, by a launch of 4 us.
// M = 16384, N = 4096, K = 1024: 256 0.69 ms, 128 0.75; M = 2048, N = 1024, K = 256: 256 0.051 ms, 128 0.023.
// K is cut at least so that the parts fill the device: the sums over them stay short, and so does what they are rounded by.  two: the
// 128 x 128 tile has sums of its own for the small products whether K is cut or not (the weight gradients), and need not be cut for it.
void gemm_f32_plan(int M, int N1, int N2, int K, bool allow_split, bool two, int *tile, int *splits, int *k_per_split) {
    double best = 0.;
    *splits = 0;
    for (int t = K > kF32AllK ? 256 : 128; t >= 128; t /= 2) {
        const long long tiles = (long long)cdiv(M, t) * (cdiv(N1, t) + cdiv(N2, t));
        const int cap = (int)std::max<long long>(64, 256 / tiles);   // (one or two tiles: as many parts as fill the device.  T*B = 280000, I = 1, H = 8 with 64 parts 343 us, now 167)
        const int most = !allow_split ? 1 : std::max(1, std::min(cap, K / (N2 ? 128 : 160)));
        const int least = (int)std::min<long long>(most, t == 256 ? 256 / tiles : tiles >= 512 ? 1 : std::max<long long>(two ? 1 : 2, (255 + tiles) / tiles));
        for (int sp = std::max(1, least); sp <= most; ++sp) {
            const int kps = sp == 1 ? K : cdiv(cdiv(K, sp), 64) * 64;
            if (sp > least && cdiv(K, kps) != sp) continue;
            const double kt = cdiv(kps, kF32BK), per_cu = (double)((tiles * cdiv(K, kps) + 255) / 256);
            double us = t == 256 ? per_cu * (2.2 * kt + 5.)
                                 : (double)((long long)per_cu / 2) * (1.35 * kt + 4.) + (double)((long long)per_cu % 2) * (0.7 * kt + 4.);
            if (sp > 1) us += 4. + (2. * sp + 1.) * M * ((double)N1 + N2) * sizeof(float) / 3.5e6;
            if (*splits == 0 || us < best) {
                best = us;
                *tile = t;
                *splits = cdiv(K, kps);
                *k_per_split = kps;
            }
        }
    }
    // Up to one 64 x 64 tile per CU, each on a CU of its own: a quarter of the products per k-tile and of the rows to store (x.Wx^T, rows, K, N, us
    // on 128 x 128 and here: 512, 80, 384 8.5 and 6.5; 256, 256, 1024 15.5 and 11.9; 1024, 256, 1024 16.0 and 12.3; 256, 1024, 4096 46 and 36; with 304
    // tiles, 1000, 300, 1200, 18.7 and 19.1, with 512, 8192, 40, 256, 9.4 and 12.6).
    // (K <= 64: the sums of all nine products take more registers than two waves of a SIMD have, for 8.5 -> 8.0.)
    if (!two && K > kF32AllK && *tile == 128 && *splits == 1 && (long long)cdiv(M, 64) * (cdiv(N1, 64) + cdiv(N2, 64)) <= 256) *tile = 64;
}

hipError_t launch_gemm_f32(const GemmF32Params &g, bool a_km, bool b_km, int tile, hipStream_t s) {
    if (tile == 64) {
        if (a_km || g.p.splits > 1 || g.p.K <= kF32AllK) return hipErrorInvalidValue;
        return b_km ? launch_t<false, true, 64, false>(g, s) : launch_t<false, false, 64, false>(g, s);
    }
    if (g.p.K <= kF32AllK && tile == 128 && g.p.splits == 1) {
        if (a_km && b_km) return launch_t<true, true, 128, true, true>(g, s);
        if (!a_km) return b_km ? launch_t<false, true, 128, true, true>(g, s) : launch_t<false, false, 128, true, true>(g, s);
    }
    if (a_km && b_km) return tile == 256 ? launch_t<true, true, 256, false>(g, s) : launch_t<true, true, 128, true>(g, s);
    if (a_km || (!b_km && g.p.splits > 1)) return hipErrorInvalidValue;
    if (!b_km) return tile == 256 ? launch_t<false, false, 256, false>(g, s) : launch_t<false, false, 128, false>(g, s);
    if (tile == 256) return launch_t<false, true, 256, false>(g, s);
    return g.p.splits > 1 ? launch_t<false, true, 128, true>(g, s) : launch_t<false, true, 128, false>(g, s);
}

}  // namespace fastlstm
