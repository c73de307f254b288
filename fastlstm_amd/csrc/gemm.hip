// Host launchers for the MFMA GEMM stages (K1, K5, K8, K9) and the db column sum.
#include "gemm.hpp"
#include "gemm16.hpp"
#include "gemm_f32.hpp"
#include <atomic>
#include "internal.hpp"

namespace fastlstm {

namespace {

// C = the sum over the parts of a split product
template <typename T> hipError_t launch_splitk_reduce(const GemmParams &p, hipStream_t stream) {
    const size_t total = (size_t)p.M * p.N;
    const int slices = p.splits >= 16 ? 4 : 1;     // many splits: four threads per output
    const int blocks = (int)((total * slices + 255) / 256);
    hipLaunchKernelGGL(splitk_reduce_kernel<T>, dim3(blocks), dim3(256), 0, stream, p.Cpart, static_cast<T *>(p.C), p.M, p.N,
                       p.ldc, p.splits, slices);
    return hipGetLastError();
}

template <typename T, bool A_KM, bool B_KM>
hipError_t launch_gemm_t(const GemmParams &p, hipStream_t stream) {
    using G = GemmTile<T>;
    static bool attr_set = false;
    auto kern = gemm_kernel<T, A_KM, B_KM>;
    if (!attr_set) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, G::LDS_BYTES);
        if (e != hipSuccess) return e;
        attr_set = true;
    }
    const int grid = cdiv(p.M, kBM) * cdiv(p.N, kBN) * p.splits;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(kThreads), G::LDS_BYTES, stream, p);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    return p.splits > 1 ? launch_splitk_reduce<T>(p, stream) : hipSuccess;
}

std::atomic<int> g_gemm_baseline{0};   // diagnostics: 1 = stand-alone 16-bit 256 x 256 launches run gemm16_onetile_kernel

// one 256 x 256 tile per workgroup (gemm16_onetile_kernel); with splits > 1 the caller reduces the partials
template <typename T, bool A_KM, bool B_KM> static hipError_t launch_onetile_t(const GemmParams &p, hipStream_t stream) {
    using C = Gemm16Cfg<256, 256, 2, 2, 4, 2>;
    static bool attr_set = false;
    auto kern = gemm16_onetile_kernel<T, A_KM, B_KM>;
    if (!attr_set) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                           C::LDS_BYTES);
        if (e != hipSuccess) return e;
        attr_set = true;
    }
    hipLaunchKernelGGL(kern, dim3(cdiv(p.M, 256) * cdiv(p.N, 256) * p.splits), dim3(C::THREADS), C::LDS_BYTES, stream, p);
    return hipGetLastError();
}

template <typename T, bool A_KM, bool B_KM, int BM, int BN, int NS, int WVM, int WVN, int KSPT>
hipError_t launch_gemm16_t(const GemmParams &p, hipStream_t stream) {
    using C = Gemm16Cfg<BM, BN, NS, WVM, WVN, KSPT>;
    static bool attr_set = false;
    const bool baseline = BM == 256 && BN == 256 && sizeof(T) == 2 && g_gemm_baseline.load() != 0;
    auto kern = gemm16_kernel<T, A_KM, B_KM, BM, BN, NS, WVM, WVN, KSPT>;
    if constexpr (BM == 256 && BN == 256 && sizeof(T) == 2) {
        if (baseline)
            if (hipError_t e = launch_onetile_t<T, A_KM, B_KM>(p, stream)) return e;
    }
    if (!attr_set) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS_BYTES);
        if (e != hipSuccess) return e;
        attr_set = true;
    }
    // the 256 x 256 configuration (one workgroup per CU) walks through a longer tile list with one workgroup per CU
    const int tiles = cdiv(p.M, BM) * cdiv(p.N, BN) * p.splits;
    const int grid = (BM == 256 && BN == 256) ? std::min(tiles, kNumXcd * 32) : tiles;
    if (!baseline) hipLaunchKernelGGL(kern, dim3(grid), dim3(C::THREADS), C::LDS_BYTES, stream, p);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    return p.splits > 1 ? launch_splitk_reduce<T>(p, stream) : hipSuccess;
}

template <typename T, int BM, int BN, int NS, int WVM, int WVN, int KSPT>
hipError_t launch_gemm16_dt(const GemmParams &p, bool a_km, bool b_km, hipStream_t s) {
    if (!a_km && !b_km) return launch_gemm16_t<T, false, false, BM, BN, NS, WVM, WVN, KSPT>(p, s);
    if (!a_km && b_km) return launch_gemm16_t<T, false, true, BM, BN, NS, WVM, WVN, KSPT>(p, s);
    if (a_km && b_km) return launch_gemm16_t<T, true, true, BM, BN, NS, WVM, WVN, KSPT>(p, s);
    return hipErrorInvalidValue;
}

template <typename T> hipError_t launch_gemm_dt(const GemmParams &p, bool a_km, bool b_km, hipStream_t s) {
    if (!a_km && !b_km) return launch_gemm_t<T, false, false>(p, s);
    if (!a_km && b_km) return launch_gemm_t<T, false, true>(p, s);
    if (a_km && b_km) return launch_gemm_t<T, true, true>(p, s);
    return hipErrorInvalidValue;
}

template <typename T>
hipError_t launch_colsum_t(const void *in, void *out, float *part, int R, int C, int chunks, hipStream_t s) {
    using E = Elem<T>;
    const int rpc = cdiv(R, chunks);
    // column groups per block: the power of two that covers the columns, at most the whole block
    auto col_threads = [](int groups) {
        int ct = 1;
        while (ct < 128 && ct < groups) ct *= 2;
        return ct;
    };
    if (C % E::EPL == 0) {
        const int ct = col_threads(C / E::EPL);
        dim3 grid(cdiv(C, ct * E::EPL), chunks);
        hipLaunchKernelGGL((colsum_partial_kernel<T, E::EPL>), grid, dim3(128), 0, s,
                           static_cast<const T *>(in), part, R, C, rpc, ct);
    } else {
        const int ct = col_threads(C);
        dim3 grid(cdiv(C, ct), chunks);
        hipLaunchKernelGGL((colsum_partial_kernel<T, 1>), grid, dim3(128), 0, s, static_cast<const T *>(in),
                           part, R, C, rpc, ct);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(colsum_final_kernel<T>, dim3(cdiv(C, kColsumFinalCols)), dim3(256), 0, s, part, static_cast<T *>(out),
                       C, chunks);
    return hipGetLastError();
}

}  // namespace

// The 16-bit fast kernel needs: K range of every split a multiple of 64, 16-byte aligned
// rows, operands addressable with 32-bit byte offsets.
bool gemm16_eligible(int dtype, int M, int N, int K, int lda, int ldb, bool a_km, bool b_km) {
    if (dtype == FASTLSTM_FP32) return false;
    const int es = 2, epc = 16 / es;
    // K-major x K-major (the weight gradients, K = T*B rows): any K -- the loop runs to the next multiple of 64 and the
    // rows past K lie outside both operands' buffer ranges, where loads return zero
    if ((K % 64 != 0 && !(a_km && b_km)) || lda % epc != 0 || ldb % epc != 0) return false;
    // 32-bit byte offsets, with room for the rows a partial tile reaches past the operand
    const size_t a_bytes = (size_t)((a_km ? K : M) + 256) * lda * es, b_bytes = (size_t)((b_km ? K : N) + 256) * ldb * es;
    return a_bytes < (1ull << 32) && b_bytes < (1ull << 32);
}

// Parts of K for 64 x 64 tiles, the least time: 0.22 us per k-tile of 64, twice that for two tiles of a CU; adding the parts up is a launch of
// 3.5 us that moves them at 3.5 TB/s.  us, whole and in parts: M = 1000, N = 64, K = 2048 10.3 -> 7.4; 700, 704, 5632 24 -> 18; both weight
// gradients of T*B = 4004, I = 104, H = 112 47 -> 24; 640, 640, 2048 stays whole (10.9, in two parts 11.8).
static int parts_of_few_tiles(int M, int N, int K, int t64) {
    const int kt = cdiv(K, 64), most = std::max(1, std::min({2 * kNumXcd * 32 / t64, kt / 4, 64}));
    int best = 1;
    double least = 0.;
    for (int sp = 1; sp <= most; ++sp) {
        double us = cdiv(kt, sp) * (t64 * sp > kNumXcd * 32 ? 0.44 : 0.22);
        if (sp > 1) us += 3.5 + (2. * sp + 1.) * M * N * sizeof(float) / 3.5e6;
        if (sp == 1 || us < least) {
            least = us;
            best = sp;
        }
    }
    return best;
}

// Tile edge (256, 128 or 64; 0 = generic kernel) and split-K factor for a product.
void gemm_plan(int dtype, int M, int N, int K, int lda, int ldb, bool a_km, bool b_km, bool allow_split,
               int *tile, int *splits) {
    if (dtype == FASTLSTM_FP32) {
        int kps;
        gemm_f32_plan(M, N, 0, K, allow_split, a_km && b_km, tile, splits, &kps);
        return;
    }
    *splits = 1;
    if (!gemm16_eligible(dtype, M, N, K, lda, ldb, a_km, b_km)) {
        *tile = 0;
        const int tiles = cdiv(M, kBM) * cdiv(N, kBN);
        if (allow_split && tiles < 128) {
            const int bk = gemm_bk();
            *splits = std::max(1, std::min(std::min(cdiv(512, tiles), std::max(1, K / (4 * bk))), 1024));
        }
        return;
    }
    const int t256 = cdiv(M, 256) * cdiv(N, 256), t128 = cdiv(M, 128) * cdiv(N, 128), t64 = cdiv(M, 64) * cdiv(N, 64);
    // At most two 64 x 64 tiles per CU: a k-tile takes them 0.22 us, the 128 x 128 tile 0.55, and four times as many CUs work (us with
    // 64 and 128: M = 700, N = 2816, K = 704, 484 tiles, 8.7 and 9.9; M = N = 700, K = 2816 14.4 and 25.2; with 768 tiles, M = 1024,
    // N = 3072, K = 512, 9.7 and 8.1).
    // Not for weight gradients of very many rows: what bounds those is reading the operands, a 64 x 64 tile twice as often (us with 64
    // and 128, thin products of T*B rows, I, H: 173400, 1024, 64 312 and 182; 65536, 64, 256 171 and 123; 32768, 80, 512 204 and 147,
    // 16384 106 and 102, 8192 65 and 81; 32768, 96, 96 49 and 44, 16384 33 and 37).
    const bool many_rows = a_km && b_km && (K >= 32768 || (long long)t64 * K > 1 << 21);
    // With room for parts and more tiles than CUs, a long sum goes to 128 x 128 tiles in as many parts as one round of them holds (us, 64 x
    // 64 whole and 128 x 128 in parts: M = 2869, N = 408, K = 4096 32 and 28, 14080 108 and 68; 1100, 1000, 8192 58 and 36; 2000, 640, 4096
    // 25 and 26).
    if (t64 <= 2 * kNumXcd * 32 && !many_rows) {
        const int round128 = kNumXcd * 32 / t128;
        const bool parts128 = allow_split && t64 > kNumXcd * 32 && K >= 4096 && round128 > 1;
        *tile = parts128 ? 128 : 64;
        if (allow_split) *splits = parts128 ? round128 : parts_of_few_tiles(M, N, K, t64);
        return;
    }
    const int max_split = allow_split ? std::max(1, K / 512) : 1;  // >= 8 k-tiles per split
    // d.Wx has a large output beside its sum, and moving parts of that costs: a k-tile takes 256 x 256 1.8 us, 128 x 128 0.55 alone on a CU and
    // 1.0 two at a time; parts are added up at 5 TB/s (us, whole on 128 x 128 and in parts on 256 x 256: M = 27870, N = 160, K = 1152 22 and
    // 39; 3267, 1432, 2688 40 and 53; 7725, 1024, 5632 97 and 114).
    const auto parts_repay = [&](int t, int tiles, int sp) {
        const double kt = cdiv(K, 64), per_tile = t == 256 ? 1.8 : tiles * sp > 256 ? 1.0 : 0.55;
        const double whole = cdiv(t128, 512) * kt * (t128 > 256 ? 1.0 : 0.55);
        return (a_km && b_km) || cdiv(tiles * sp, t == 256 ? 256 : 512) * kt / sp * per_tile + 3.5 + (2. * sp + 1.) * M * N * sizeof(float) / 5e6 < whole;
    };
    const int split256 = std::min(256 / t256, max_split), split128 = t128 < 192 ? std::max(1, std::min(cdiv(512, t128), max_split)) : 1;
    if (t256 >= 192) {
        *tile = 256;
    } else if (split256 * t256 >= 192 && (split256 == 1 || parts_repay(256, t256, split256))) {   // (one round of workgroups: the factor rounded down)
        *tile = 256;
        *splits = split256;
    } else {
        *tile = 128;
        if (split128 > 1 && parts_repay(128, t128, split128)) *splits = split128;
    }
}

// ---- both weight gradients + the bias gradient on the tile kernel (gemm16_wgrad_kernel) ------------------------
// Taken for fp32 (gemm_f32.hpp) and for 16-bit products that the 256 x 256 tile kernel holds.  *merged: both products as one tile grid with
// one split factor (K = T*B is split so that the tiles of both together fill the device); otherwise each product
// fills the device on its own and they run as two launches of one round of tiles each, the bias gradient with
// the first (a second round of tiles starts out of step with its neighbours and shares less in the L2:
// M = 8192, I = H = 2048, K = 32768: 1.85 ms merged against 2 x 0.86).
bool wgrad_merged_plan(int dtype, int M, int I, int H, int K, int *splits, int *k_per_split, bool *merged) {
    if (dtype == FASTLSTM_FP32) {   // any shape, always one grid
        int tile;
        *merged = true;
        gemm_f32_plan(M, I, H, K, true, true, &tile, splits, k_per_split);
        return true;
    }
    if (!gemm16_eligible(dtype, M, I, K, M, I, true, true) || !gemm16_eligible(dtype, M, H, K, M, H, true, true)) return false;
    if (M < 256 || I < 128 || H < 128) return false;   // thin outputs: the 128 x 128 tiles waste less
    const int tx = cdiv(M, 256) * cdiv(I, 256), th = cdiv(M, 256) * cdiv(H, 256);
    *merged = !(tx >= 192 && th >= 192 && tx <= 256 && th <= 256);
    int sp = 1;
    // (rounded down: one round of at most 256 workgroups; 60 tiles x 5 splits would be a full round and a sixth of one)
    if (*merged && tx + th < 192) sp = std::max(1, std::min(256 / (tx + th), K / 512));   // >= 8 k-tiles per split
    const int kps = cdiv(cdiv(K, sp), 64) * 64;
    *k_per_split = kps;
    *splits = cdiv(K, kps);
    return true;
}

// workspace: [splits][column tiles][M] for the bias gradient + [splits][M][I] + [splits][M][H] floats with a split
size_t wgrad_merged_workspace(int dtype, int M, int I, int H, int K) {
    int sp, kps;
    bool merged;
    if (!wgrad_merged_plan(dtype, M, I, H, K, &sp, &kps, &merged)) return 0;
    const size_t dbp = align_up((size_t)sp * (cdiv(I, 256) + cdiv(H, 256)) * M * sizeof(float), 256);
    return dbp + (sp > 1 ? (size_t)sp * M * ((size_t)I + H) * sizeof(float) : 0);
}

template <typename T>
static hipError_t launch_wgrad_kernel_t(const WgradParams &w, hipStream_t s) {
    using C = Gemm16Cfg<256, 256, 2, 2, 4, 2>;
    static bool attr_set = false;
    auto kern = gemm16_wgrad_kernel<T>;
    if (!attr_set) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                           C::LDS_BYTES);
        if (e != hipSuccess) return e;
        attr_set = true;
    }
    const int grid = cdiv(w.x.M, 256) * (w.tiles_nx + cdiv(w.h.N, 256)) * w.x.splits;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(C::THREADS), C::LDS_BYTES, s, w);
    return hipGetLastError();
}

template <typename T> static hipError_t launch_wgrad_reduce(const WgradParams &w, void *db, int db_parts, hipStream_t s) {
    const int M = w.x.M, splits = w.x.splits;
    const int ri = splits > 1 ? w.x.N : 0, rh = splits > 1 ? w.h.N : 0;   // the products need no pass without a split
    const size_t threads = (size_t)M * ri / 4 + (size_t)M * rh / 4 + M;
    hipLaunchKernelGGL(wgrad_reduce_kernel<T>, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s, w.x.Cpart,
                       static_cast<T *>(w.x.C), w.h.Cpart, static_cast<T *>(w.h.C), w.db_part, static_cast<T *>(db), M, ri, rh,
                       splits, db_parts);
    return hipGetLastError();
}

template <typename T>
static hipError_t launch_wgrad_merged_t(const WgradParams &w, bool merged, void *db, hipStream_t s) {
    const int M = w.x.M, I = w.x.N, H = w.h.N, splits = w.x.splits;
    int db_parts;
    if (merged) {
        if (hipError_t e = launch_wgrad_kernel_t<T>(w, s)) return e;
        db_parts = splits * (w.tiles_nx + cdiv(H, 256));
    } else {   // the x product with the bias gradient, then the h product alone
        WgradParams a = w;
        a.h.N = 0;
        if (hipError_t e = launch_wgrad_kernel_t<T>(a, s)) return e;
        // one round of tiles, both operands K-major: the symmetric loop (gemm16_onetile_kernel)
        if (hipError_t e = launch_onetile_t<T, true, true>(w.h, s)) return e;
        db_parts = splits * w.tiles_nx;
    }
    return launch_wgrad_reduce<T>(w, db, db_parts, s);
}

// The fp32 products (gemm_f32.hpp): one grid over both, the bias gradient with the first column of tiles.
static hipError_t launch_wgrad_f32(const WgradParams &w, int tile, void *db, hipStream_t s) {
    GemmF32Params g{};
    g.p = w.x;
    g.B2 = w.h.B; g.C2 = w.h.C; g.Cpart2 = w.h.Cpart; g.N2 = w.h.N; g.ldb2 = w.h.ldb; g.ldc2 = w.h.ldc;
    g.tiles_n1 = cdiv(w.x.N, tile);
    g.db_part = w.db_part;
    if (hipError_t e = launch_gemm_f32(g, true, true, tile, s)) return e;
    return launch_wgrad_reduce<float>(w, db, w.x.splits, s);
}

hipError_t launch_wgrad_merged(int dtype, const void *d_ifgo, const void *x, const void *h, void *dWx, void *dWh, void *db,
                               void *ws, int M, int I, int H, int K, hipStream_t s) {
    WgradParams w{};
    int sp, kps;
    bool merged;
    if (!wgrad_merged_plan(dtype, M, I, H, K, &sp, &kps, &merged)) return hipErrorInvalidValue;
    float *db_part = static_cast<float *>(ws);
    float *part_x = reinterpret_cast<float *>(static_cast<unsigned char *>(ws) +
                                              align_up((size_t)sp * (cdiv(I, 256) + cdiv(H, 256)) * M * sizeof(float), 256));
    GemmParams g{};
    g.A = d_ifgo; g.M = M; g.K = K; g.lda = M; g.splits = sp; g.k_per_split = kps;
    w.x = g; w.x.B = x; w.x.C = dWx; w.x.N = I; w.x.ldb = I; w.x.ldc = I; w.x.Cpart = part_x;
    w.h = g; w.h.B = h; w.h.C = dWh; w.h.N = H; w.h.ldb = H; w.h.ldc = H; w.h.Cpart = part_x + (size_t)sp * M * I;
    w.tiles_nx = cdiv(I, 256);
    w.db_part = db_part;
    if (dtype == FASTLSTM_FP32) {
        int tile;
        gemm_f32_plan(M, I, H, K, true, true, &tile, &sp, &kps);
        return launch_wgrad_f32(w, tile, db, s);
    }
    return dtype == FASTLSTM_FP16 ? launch_wgrad_merged_t<_Float16>(w, merged, db, s)
                                    : launch_wgrad_merged_t<__bf16>(w, merged, db, s);
}

void set_gemm_baseline(int on) { g_gemm_baseline.store(on ? 1 : 0); }
int gemm_baseline() { return g_gemm_baseline.load(); }

static long long *g_trace = nullptr;
void set_gemm_trace(long long *buf) { g_trace = buf; }

hipError_t launch_gemm_tiled(int dtype, const GemmParams &p_in, bool a_km, bool b_km, int tile, hipStream_t s) {
    GemmParams p = p_in;
    p.trace = g_trace;
#define FASTLSTM_TILE_CASE(ID, BM, BN, NS, WVM, WVN, KSPT)                                                  \
    if (tile == ID)                                                                                         \
        return dtype == FASTLSTM_FP16 ? launch_gemm16_dt<_Float16, BM, BN, NS, WVM, WVN, KSPT>(p, a_km, b_km, s) \
                                      : launch_gemm16_dt<__bf16, BM, BN, NS, WVM, WVN, KSPT>(p, a_km, b_km, s);
    if (dtype == FASTLSTM_FP32) {
        GemmF32Params g{};
        g.p = p;
        if (hipError_t e = launch_gemm_f32(g, a_km, b_km, tile, s)) return e;
        return p.splits > 1 ? launch_splitk_reduce<float>(p, s) : hipSuccess;
    }
    // 8 waves each (gemm16_mainloop, SHORT).  Four stages of 32 KiB where a CU has one of the 128 x 128 tiles, two where it has two
    // (us with four and two: M = 1280, N = 2048, K = 8192 in one pass, 160 tiles, 65.5 and 86.6; M = 4096, N = 2048, K = 256, 512 tiles,
    // 11.9 and 10.4); four of 16 KiB for the 64 x 64 tiles, of which a CU takes two.
    if (tile == 128 && cdiv(p.M, 128) * cdiv(p.N, 128) * p.splits <= kNumXcd * 32) tile = 4 * 128;
    FASTLSTM_TILE_CASE(64, 64, 64, 4, 2, 4, 2)
    FASTLSTM_TILE_CASE(128, 128, 128, 2, 2, 4, 2)
    FASTLSTM_TILE_CASE(4 * 128, 128, 128, 4, 2, 4, 2)
    FASTLSTM_TILE_CASE(256, 256, 256, 2, 2, 4, 2)   // 8 waves, 128 x 64 per wave, 2 x 64 KiB stages
#undef FASTLSTM_TILE_CASE
    return launch_gemm(dtype, p, a_km, b_km, s);
}

hipError_t launch_gemm(int dtype, const GemmParams &p, bool a_km, bool b_km, hipStream_t s) {
    switch (dtype) {
        case FASTLSTM_FP16: return launch_gemm_dt<_Float16>(p, a_km, b_km, s);
        default: return launch_gemm_dt<__bf16>(p, a_km, b_km, s);
    }
}

hipError_t launch_colsum(int dtype, const void *in, void *out, float *part, int R, int C, int chunks,
                         hipStream_t s) {
    switch (dtype) {
        case FASTLSTM_FP32: return launch_colsum_t<float>(in, out, part, R, C, chunks, s);
        case FASTLSTM_FP16: return launch_colsum_t<_Float16>(in, out, part, R, C, chunks, s);
        default: return launch_colsum_t<__bf16>(in, out, part, R, C, chunks, s);
    }
}

// the second stage alone: out[C] = the sum over `chunks` rows of part[chunks][C]
hipError_t launch_colsum_final(int dtype, const float *part, void *out, int C, int chunks, hipStream_t s) {
    const dim3 grid(cdiv(C, kColsumFinalCols)), block(256);
    if (dtype == FASTLSTM_FP32) hipLaunchKernelGGL(colsum_final_kernel<float>, grid, block, 0, s, part, static_cast<float *>(out), C, chunks);
    else if (dtype == FASTLSTM_FP16) hipLaunchKernelGGL(colsum_final_kernel<_Float16>, grid, block, 0, s, part, static_cast<_Float16 *>(out), C, chunks);
    else hipLaunchKernelGGL(colsum_final_kernel<__bf16>, grid, block, 0, s, part, static_cast<__bf16 *>(out), C, chunks);
    return hipGetLastError();
}

int gemm_bk() { return GemmTile<_Float16>::BK; }

}  // namespace fastlstm
