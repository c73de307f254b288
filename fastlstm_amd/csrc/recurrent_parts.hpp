// fp32 numbers as sums of three bf16 numbers, for the recurrent products on the bf16 matrix units: of at least 64 terms, so that six of
// the nine products of two such sums (three roundings per 32 terms) are nearer to 64 bits than the fp32 matrix instructions are, though the
// parts are cut off and not rounded (gemm_f32.hpp, where that counts).
#pragma once
#include <type_traits>

#include "recurrent_common.hpp"

namespace fastlstm {

// A value with its lower 16 bits cut off.  (By value: a bit cast of an element of a vector takes the vector's first element.)
__device__ __forceinline__ float upper_half(float v) { return __builtin_bit_cast(float, __builtin_bit_cast(unsigned, v) & 0xffff0000u); }
__device__ __forceinline__ unsigned upper_halves(float a, float b) {
    return __builtin_amdgcn_perm(__builtin_bit_cast(unsigned, b), __builtin_bit_cast(unsigned, a), 0x07060302u);
}

// The three bf16 parts of a factor of a recurrent product.  A part that is zero where the number is not becomes the least bf16 number of
// its sign, 2^-133, and those of an infinity too: infinity times zero would be no number.  Zero stays zero.  (The matrix units take numbers
// below the least normal one as they are.)
// What a number is off by for that, 2^-132, is nothing beside the gates that h and the weights make.  The gate gradients of the reverse pass
// stand alone, and over a sequence they may fade through all magnitudes: the fp32 kernels carry all gradients times 2^16, by which every
// number's last bit is a bf16 number, and store them times 2^-16.  (Scaled where they are split, and the sums back, a step of H = 256 took 0.15
// us more.)  Relative error of dx where |dx| is about 1e-33, 1e-36, 1e-38 (fp32 matrix instructions: 2e-6 at
// all): 1e-5, 2e-3, 2e-1 without, 2e-6 with it.  A gate gradient beyond 2^112 overflows.
struct ThreeParts {
    float hi, mid, lo, least;   // (least: that number, for the last four columns)
    __device__ __forceinline__ explicit ThreeParts(float x) {
        const float tiny = fminf(fabsf(x), 0x1p-133f), r = x - upper_half(x);
        least = __builtin_copysignf(tiny, x);
        hi = __builtin_canonicalizef(x);
        mid = __builtin_copysignf(fmaxf(fabsf(r), tiny), x);
        lo = __builtin_copysignf(fmaxf(fabsf(r - upper_half(mid)), tiny), x);
    }
    __device__ __forceinline__ float part(int i) const { return i == 0 ? hi : i == 1 ? mid : i == 2 ? lo : least; }
};

constexpr float kGradScale = 0x1p16f, kGradUnscale = 0x1p-16f;   // (see above)

// 16 bytes of operand block: 8 consecutive elements of k -> the 16-bit fragment of part i
template <typename T, typename Get> __device__ __forceinline__ void operand_parts(Get get, u32x4 (&out)[sizeof(T) == 4 ? 3 : 1]) {
    if constexpr (sizeof(T) == 4) {
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            const ThreeParts a(get(2 * d)), b(get(2 * d + 1));
#pragma unroll
            for (int i = 0; i < 3; ++i) out[i][d] = upper_halves(a.part(i), b.part(i));
        }
    } else {
        T t[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) t[e] = get(e);
        __builtin_memcpy(&out[0], t, 16);
    }
}

// the 16-bit type whose MFMAs multiply
template <typename T> using OperandType = typename std::conditional<sizeof(T) == 4, __bf16, T>::type;

// acc + small += a . b by the products of the parts that count: the largest in a sum of its own (rounded once per 32 k), the five others
// (those left out are below 2^-22 of it) in `small`.  16-bit types: the one product, in acc.
template <typename T, int P> __device__ __forceinline__ void mfma_parts(const u32x4 (&a)[P], const u32x4 (&b)[P], f32x4 &acc, f32x4 &small) {
    using O = OperandType<T>;
    if constexpr (P == 3) {
        small = mfma_kstep<O>(a[2], b[0], small);
        small = mfma_kstep<O>(a[0], b[2], small);
        small = mfma_kstep<O>(a[1], b[1], small);
        small = mfma_kstep<O>(a[1], b[0], small);
        small = mfma_kstep<O>(a[0], b[1], small);
    }
    acc = mfma_kstep<O>(a[0], b[0], acc);
}

// Operand blocks of the XCD-local kernels: 16 rows x 32 k of 16-bit elements, fp32 one such block per part.
template <typename T> struct OperandBlocks {
    static constexpr int P = sizeof(T) == 4 ? 3 : 1, KSTEP = 32, BYTES = P * kFragBytes;   // of a k-step
    // byte offset of element k of row r (part 0)
    static __device__ __forceinline__ int offset(int r, int k) { return k / 32 * BYTES + frag_offset<OperandType<T>>(r, k % 32); }
};

}  // namespace fastlstm
