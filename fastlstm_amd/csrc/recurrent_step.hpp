// A few timesteps of inference without a persistent launch: one kernel per timestep computes the gates of a whole
// cell, ifgo = x_t.Wx^T + bx + bh + h.Wh^T, and updates c and h (the maths of fastlstm/lstm.py:66-68 and
// kernels.py:414-663 for one step).  A step of one to a few rows is bound by latency: the chain of dependent
// loads, the launch, and for large layers the one pass over the weights.  The persistent path needs, per layer, a launch
// that prepares the workspace, the projection, the time loop (with a barrier before the first step) and the status
// collection; here there is no workspace, no barrier between workgroups, hence nothing to prepare, no status.
//
// Split: a workgroup owns four hidden units, whose 16 weight rows (unit, gate) are one MFMA operand, times all
// batch rows (16 NT <= 64 per blockIdx.y); its eight waves split K = I + H into eight contiguous runs of k-steps (whole
// cache lines of a weight row stay with one wave), request a batch of operand blocks before the first product,
// and add their sums through LDS.  H / 4 workgroups per layer: 128 at H = 512.  Every workgroup reads all of x_t and h
// through the L2, so with more than 32 rows and at least two workgroups per CU (the jobs of a launch together) a
// workgroup takes eight units (MT = 2).
// One step, state carried, per call of the module: 2 layers, B = 4, I = H = 512 fp16 112 -> 18 us; 3 layers, B = 1,
// I = 123, H = 213 fp32 165 -> 22; 1 layer, B = 32, I = 1024, H = 1536 fp16 53 -> 19.
//
// The step t of layer l needs layer l - 1's step t and its own step t - 1, so launch k runs step k - l of every layer l:
// T + L - 1 launches.  c is carried in fp32 between the steps of a call, as the persistent kernels carry it.
#pragma once
#include "common.hpp"

namespace fastlstm {

constexpr int kStepJobs = 4;   // cells of one launch

struct StepJob {
    const void *x, *h;         // [B,K], [B,H]; h null: zero state
    const void *Wx, *Wh;       // [4H,K], [4H,H]
    const void *bx, *bh;       // [4H] or null
    const void *c_in;          // [B,H] in T, or null
    float *c_run;              // [B,H]: c between the steps of a call, or null
    void *h_out, *h_out2;      // [B,H]; h_out2 may be null
    void *c_out;               // [B,H] in T (last step), or null
    int K;                     // input size of the layer
    int first;                 // 1: c comes from c_in (zero when null), 0: from c_run
};
struct StepParams {
    StepJob job[kStepJobs];
    int B, H, tiles;           // tiles: workgroups per job
};

// One operand fragment: EPL elements row[k .. k + EPL), zeros past `lim` or when the row does not exist.  VEC: rows start
// on 16 bytes and hold whole pieces; otherwise a piece inside the row is one load on any byte boundary all the same, and
// only the piece that the end of the row cuts is read by elements.
template <typename T, bool VEC> __device__ __forceinline__ u32x4 step_frag(const T *row, int k, int lim, bool ok) {
    using E = Elem<T>;
    if constexpr (VEC) {
        const bool in = ok && k < lim;
        const u32x4 v = *reinterpret_cast<const u32x4 *>(row + (in ? k : 0));
        return in ? v : u32x4{0u, 0u, 0u, 0u};
    } else {
        typedef u32x4 __attribute__((aligned(2))) piece;
        u32x4 v = {0u, 0u, 0u, 0u};
        if (ok && k + E::EPL <= lim) {
            v = *reinterpret_cast<const piece *>(row + k);
        } else if (ok && k < lim) {
            T tmp[E::EPL];
#pragma unroll
            for (int e = 0; e < E::EPL; ++e) tmp[e] = k + e < lim ? row[k + e] : E::from_f32(0.f);
            v = *reinterpret_cast<u32x4 *>(tmp);
        }
        return v;
    }
}

// 4 MT hidden units x 16 NT batch rows per workgroup.
template <typename T, int MT, int NT, bool VEC>
__global__ __launch_bounds__(kWave * 8) void lstm_step_kernel(const StepParams p) {
    using E = Elem<T>;
    constexpr bool ACC = (E::DT == FASTLSTM_FP32);
    constexpr int NWV = 8, U = NT == 4 ? 4 : 8;   // k-steps requested at a time
    constexpr int ITEMS = MT * NT;                // waves that finish a (unit tile, batch tile) each
    static_assert(ITEMS <= NWV, "one tile per wave");
    __shared__ f32x4 red[NWV][ITEMS][kWave];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int q = lane >> 4, n = lane & 15;
    const int which = blockIdx.x / p.tiles;
    // (constant indices: a run-time index would move the kernel's arguments to scratch memory)
    const StepJob &j = which == 0 ? p.job[0] : which == 1 ? p.job[1] : which == 2 ? p.job[2] : p.job[3];
    const int u0 = (blockIdx.x % p.tiles) * 4 * MT, b0 = blockIdx.y * 16 * NT, H = p.H, B = p.B;

    const int KX = (j.K + E::KSTEP - 1) / E::KSTEP, KH = j.h ? (H + E::KSTEP - 1) / E::KSTEP : 0;
    const int per = (KX + KH + NWV - 1) / NWV;
    const int k_end = min(KX + KH, (wave + 1) * per);
    f32x4 acc[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int i = 0; i < NT; ++i) acc[m][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int k0 = wave * per; k0 < k_end; k0 += U) {
        u32x4 a[U][MT], b[U][NT];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int ks = k0 + u;
            const bool in_x = ks < KX, live = ks < k_end;
            const int K = in_x ? j.K : H, k = (in_x ? ks : ks - KX) * E::KSTEP + q * E::EPL;
            const T *W = static_cast<const T *>(in_x ? j.Wx : j.Wh), *V = static_cast<const T *>(in_x ? j.x : j.h);
#pragma unroll
            for (int m = 0; m < MT; ++m) a[u][m] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
            for (int i = 0; i < NT; ++i) b[u][i] = u32x4{0u, 0u, 0u, 0u};
            if (live) {
#pragma unroll
                for (int m = 0; m < MT; ++m) {   // operand row n = (unit n / 4, gate n % 4)
                    const int unit = u0 + 4 * m + (n >> 2);
                    a[u][m] = step_frag<T, VEC>(W + ((size_t)(n & 3) * H + (unit < H ? unit : 0)) * K, k, K, unit < H);
                }
#pragma unroll
                for (int i = 0; i < NT; ++i) {
                    const int row = b0 + i * 16 + n;
                    b[u][i] = step_frag<T, VEC>(V + (size_t)(row < B ? row : 0) * K, k, K, row < B);
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);   // one round trip per batch of loads
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int i = 0; i < NT; ++i) acc[m][i] = mfma_kstep<T>(a[u][m], b[u][i], acc[m][i]);
    }
    // what the cell needs besides the sums: requested before the sums are exchanged
    const int unit = u0 + 4 * (wave / NT) + q, row = b0 + (wave % NT) * 16 + n;
    const bool mine = wave < ITEMS && unit < H && row < B;
    const size_t at = (size_t)row * H + unit;
    float bias[4] = {0.f, 0.f, 0.f, 0.f}, c0 = 0.f;
    if (mine) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            if (j.bx) bias[g] += E::to_f32(static_cast<const T *>(j.bx)[g * H + unit]);
            if (j.bh) bias[g] += E::to_f32(static_cast<const T *>(j.bh)[g * H + unit]);
        }
        if (!j.first) c0 = j.c_run[at];
        else if (j.c_in) c0 = E::to_f32(static_cast<const T *>(j.c_in)[at]);
    }
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int i = 0; i < NT; ++i) red[wave][m * NT + i][lane] = acc[m][i];
    __syncthreads();
    if (!mine) return;
    f32x4 s = red[0][wave][lane];
#pragma unroll
    for (int w = 1; w < NWV; ++w) s += red[w][wave][lane];
    const float c1 = sigmoidf_<ACC>(s[1] + bias[1]) * c0 + sigmoidf_<ACC>(s[0] + bias[0]) * tanhf_<ACC>(s[2] + bias[2]);
    const T h1 = E::from_f32(sigmoidf_<ACC>(s[3] + bias[3]) * tanhf_<ACC>(c1));
    static_cast<T *>(j.h_out)[at] = h1;
    if (j.h_out2) static_cast<T *>(j.h_out2)[at] = h1;
    if (j.c_run) j.c_run[at] = c1;
    if (j.c_out) static_cast<T *>(j.c_out)[at] = E::from_f32(c1);
}

// jobs <= kStepJobs; p.tiles is set here
hipError_t launch_step(int dtype, StepParams &p, int jobs, bool vec, hipStream_t s);

}  // namespace fastlstm
