// What surrounds the layers of a call, as one launch per stage of it: zero-padding and converting parameters, inputs,
// states and gradients, cutting results back, packing and unpacking sequences of different lengths, reversing
// them in time for the second direction, taking final states.  (fastlstm_copy_blocks, fastlstm_upload_ints; the
// reference leaves such work to torch operators around its kernels, fastlstm/lstm.py:509-515, 685-698.)
//
// Each copy on its own is a few microseconds of memory traffic, so a call with twenty of them was bound by the launches and by
// the host's work for each: they are descriptors of one launch instead.  A thread moves eight neighbouring
// elements of a destination row; rows may start on any boundary (H = 257): the loads and stores are full-width all the same.
// 2 layers, T = 35, B = 20, I = H = 650 under bf16 autocast (13.5 M fp32 parameters in, as many gradients out): the parameters
// in 14 us, 16 launches of 4 ... 8 us before.
#include <algorithm>

#include "common.hpp"

namespace fastlstm {
namespace {

constexpr int kMaxCopies = 32;   // descriptors per launch (they travel in the kernel's arguments)

struct Copy {
    const void *src, *src2;      // src2: added (null: none)
    void *dst;
    int groups, rows_src, rows_dst, blocks, cols_src, cols_dst;
    int ld_src, ld_src2, ld_dst;
    unsigned char smode, s2mode, dmode, dt_src, dt_dst;
    int first_wg, cpieces;       // first workgroup of the copy; eight-element pieces per block row
    unsigned pieces;
};
struct CopyParams {
    Copy c[kMaxCopies];
    int n, T, B;
    const int *lens, *offs;      // [B], [T] or null: every sequence has T steps, step t starts at row t * B
    const long long *order;      // [B] or null
};
static_assert(sizeof(CopyParams) <= 4096, "kernel arguments");

struct F8 { float v[8]; };

template <typename T> __device__ __forceinline__ F8 load8_t(const T *p, int n) {
    F8 r;
    if (n >= 8) {
        typedef u32x4 __attribute__((aligned(2))) piece;
        T tmp[8];
#pragma unroll
        for (unsigned i = 0; i < 8 * sizeof(T) / 16; ++i) *reinterpret_cast<u32x4 *>(tmp + i * 16 / sizeof(T)) = *reinterpret_cast<const piece *>(p + i * 16 / sizeof(T));
#pragma unroll
        for (int e = 0; e < 8; ++e) r.v[e] = (float)tmp[e];
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) r.v[e] = e < n ? (float)p[e] : 0.f;
    }
    return r;
}
__device__ __forceinline__ F8 load8(const void *p, size_t at, int dt, int n) {
    if (dt == FASTLSTM_FP32) return load8_t(static_cast<const float *>(p) + at, n);
    if (dt == FASTLSTM_FP16) return load8_t(static_cast<const _Float16 *>(p) + at, n);
    return load8_t(static_cast<const __bf16 *>(p) + at, n);
}
template <typename T> __device__ __forceinline__ void store8_t(T *p, const F8 &r, int n) {
    if (n >= 8) {
        typedef u32x4 __attribute__((aligned(2))) piece;
        T tmp[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) tmp[e] = (T)r.v[e];
#pragma unroll
        for (unsigned i = 0; i < 8 * sizeof(T) / 16; ++i) *reinterpret_cast<piece *>(p + i * 16 / sizeof(T)) = *reinterpret_cast<const u32x4 *>(tmp + i * 16 / sizeof(T));
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
            if (e < n) p[e] = (T)r.v[e];
    }
}
__device__ __forceinline__ void store8(void *p, size_t at, int dt, const F8 &r, int n) {
    if (dt == FASTLSTM_FP32) store8_t(static_cast<float *>(p) + at, r, n);
    else if (dt == FASTLSTM_FP16) store8_t(static_cast<_Float16 *>(p) + at, r, n);
    else store8_t(static_cast<__bf16 *>(p) + at, r, n);
}

// Row of a tensor for slot (t, b); -1: none.
__device__ __forceinline__ int slot_row(int mode, int t, int b, int len, const CopyParams &p) {
    const bool in = t < len;
    switch (mode) {
        case FASTLSTM_ROWS_PADDED: return t * p.B + b;
        case FASTLSTM_ROWS_PADDED_REVERSED: return (in ? len - 1 - t : t) * p.B + b;
        case FASTLSTM_ROWS_PACKED: return in ? (p.offs ? p.offs[t] : t * p.B) + b : -1;
        case FASTLSTM_ROWS_PACKED_REVERSED: return in ? (p.offs ? p.offs[len - 1 - t] : (len - 1 - t) * p.B) + b : -1;
        case FASTLSTM_ROWS_LAST: return (len - 1) * p.B + b;
        case FASTLSTM_ROWS_ORDERED: return p.order ? (int)p.order[b] : b;
        default: return b;
    }
}

__global__ __launch_bounds__(256) void copy_blocks_kernel(const CopyParams p) {
    int k = 0;
    for (int i = 1; i < p.n; ++i) k = (int)blockIdx.x >= p.c[i].first_wg ? i : k;   // (scalar: one copy per workgroup)
    const Copy &c = p.c[k];
    const unsigned i = (blockIdx.x - c.first_wg) * 256u + threadIdx.x;
    if (i >= c.pieces) return;
    const unsigned c8 = i % (unsigned)c.cpieces, rb = i / (unsigned)c.cpieces;
    const int col = (int)c8 * 8, n = c.cols_dst - col;   // (>= 8: a whole piece)
    F8 r;
    size_t to;
    if (c.dmode == 0) {
        const int blk = (int)(rb % (unsigned)c.blocks), row = (int)(rb / (unsigned)c.blocks);
        const int g = row / c.rows_dst, ri = row % c.rows_dst;
        const int have = c.src && ri < c.rows_src ? c.cols_src - col : 0;
        if (have > 0) {
            r = load8(c.src, (size_t)(g * c.rows_src + ri) * c.ld_src + (size_t)blk * c.cols_src + col, c.dt_src, have);
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) r.v[e] = 0.f;
        }
        to = (size_t)row * c.ld_dst + (size_t)blk * c.cols_dst + col;
    } else {
        const int slot = (int)rb, b = slot % p.B, t = slot / p.B;
        const int len = p.lens ? p.lens[b] : p.T;
        const int row = slot_row(c.dmode, t, b, len, p);
        if (row < 0) return;
        const int have = c.cols_src - col, from = c.src && have > 0 ? slot_row(c.smode, t, b, len, p) : -1;
        if (from >= 0) {
            r = load8(c.src, (size_t)from * c.ld_src + col, c.dt_src, have);
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) r.v[e] = 0.f;
        }
        const int from2 = c.src2 && have > 0 ? slot_row(c.s2mode, t, b, len, p) : -1;
        if (from2 >= 0) {
            const F8 s = load8(c.src2, (size_t)from2 * c.ld_src2 + col, c.dt_src, have);
#pragma unroll
            for (int e = 0; e < 8; ++e) r.v[e] += s.v[e];
        }
        to = (size_t)row * c.ld_dst + col;
    }
    store8(c.dst, to, c.dt_dst, r, n);
}

constexpr int kUploadInts = 960;
struct UploadParams { int n; int v[kUploadInts]; };
static_assert(sizeof(UploadParams) <= 4096, "kernel arguments");
__global__ void upload_ints_kernel(const UploadParams p, int *dst) {
    for (int i = threadIdx.x; i < p.n; i += blockDim.x) dst[i] = p.v[i];
}

}  // namespace
}  // namespace fastlstm

using namespace fastlstm;

extern "C" {

int fastlstm_copy_blocks(int n, const long long *d, int T, int B, const int *lens, const int *offs, const long long *order,
                         void *stream) {
    if (n < 0 || T < 0 || B < 0) return FASTLSTM_ERR_DIM;
    if (n && !d) return FASTLSTM_ERR_NULL;
    for (int base = 0; base < n; base += kMaxCopies) {
        CopyParams p{};
        p.T = T; p.B = B; p.lens = lens; p.offs = offs; p.order = order;
        int wgs = 0;
        for (int i = base; i < std::min(n, base + kMaxCopies); ++i) {
            const long long *f = d + (size_t)i * FASTLSTM_COPY_FIELDS;
            Copy c{};
            c.src = reinterpret_cast<const void *>(f[0]); c.src2 = reinterpret_cast<const void *>(f[1]); c.dst = reinterpret_cast<void *>(f[2]);
            c.smode = (unsigned char)f[3]; c.s2mode = (unsigned char)f[4]; c.dmode = (unsigned char)f[5];
            c.groups = (int)f[6]; c.rows_src = (int)f[7]; c.rows_dst = (int)f[8]; c.blocks = (int)f[9];
            c.cols_src = (int)f[10]; c.cols_dst = (int)f[11];
            c.ld_src = (int)f[12]; c.ld_src2 = (int)f[13]; c.ld_dst = (int)f[14];
            c.dt_src = (unsigned char)(f[15] & 15); c.dt_dst = (unsigned char)(f[15] >> 4);
            if (!c.dst) return FASTLSTM_ERR_NULL;
            if (!dtype_ok(c.dt_src) || !dtype_ok(c.dt_dst)) return FASTLSTM_ERR_DTYPE;
            if (f[3] < 0 || f[3] > 7 || f[4] < 0 || f[4] > 7 || f[5] < 0 || f[5] > 7) return FASTLSTM_ERR_DIM;
            for (int k = 6; k < 15; ++k)
                if (f[k] < 0 || f[k] >= (1ll << 31)) return FASTLSTM_ERR_DIM;
            if (c.dmode && c.blocks != 1) return FASTLSTM_ERR_DIM;
            // one destination row per slot: (t, b), or b alone where the rows are the batch's
            const long long rows = !c.dmode ? (long long)c.groups * c.rows_dst
                                            : c.dmode >= FASTLSTM_ROWS_LAST ? B : (long long)T * B;
            c.cpieces = cdiv(c.cols_dst, 8);
            const long long pieces = rows * c.blocks * c.cpieces;
            if (rows >= (1ll << 31) || pieces >= (1ll << 31)) return FASTLSTM_ERR_DIM;
            if (!pieces) continue;
            c.pieces = (unsigned)pieces;
            c.first_wg = wgs;
            wgs += (int)((pieces + 255) / 256);
            p.c[p.n++] = c;
        }
        if (!p.n) continue;
        copy_blocks_kernel<<<wgs, 256, 0, static_cast<hipStream_t>(stream)>>>(p);
        if (hipGetLastError() != hipSuccess) return FASTLSTM_ERR_HIP;
    }
    return FASTLSTM_OK;
}

int fastlstm_upload_ints(const int *host, int n, int *dev, void *stream) {
    if (n < 0) return FASTLSTM_ERR_DIM;
    if (n && (!host || !dev)) return FASTLSTM_ERR_NULL;
    for (int base = 0; base < n; base += kUploadInts) {
        UploadParams p;
        p.n = std::min(kUploadInts, n - base);
        std::copy(host + base, host + base + p.n, p.v);
        upload_ints_kernel<<<1, 256, 0, static_cast<hipStream_t>(stream)>>>(p, dev + base);
        if (hipGetLastError() != hipSuccess) return FASTLSTM_ERR_HIP;
    }
    return FASTLSTM_OK;
}

}  // extern "C"
