// fp32 values as sums of bf16 terms, for products on the bf16 matrix core that keep every bit of the fp32 operand.
#pragma once
#include "common.h"

#include <type_traits>

namespace axhip {

// fp32 x int8 products on the bf16 matrix core, with fp32 accuracy.  Every int8 value is a bf16 exactly.  An fp32
// value a is cut into three bf16 terms: hi = a with its low 16 bits cleared, mid = (a - hi) with its low 16 bits
// cleared, lo = a - hi - mid; both subtractions are exact and lo has at most 8 significant bits, so
// a = hi + mid + lo exactly, every term times an int8 value is exact in fp32, and only the accumulation rounds —
// as in the fp32 product, at a sixteenth of its matrix-core time per term.  An infinite a keeps hi = a and
// mid = lo = 0 (a - hi would be NaN), so infinities and NaNs come out as the fp32 product gives them.
// Cost per fp32 value: canonical form, and, subtract, median (the NaN filter), and, subtract, and half of each of three
// packs: 7.5 vector instructions; per int8 value one conversion and half a pack.
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
struct Bf16x3 {
    v4i hi, mid, lo;     // 8 k values each: a k-block's four, then the next k-block's four
};
__device__ __forceinline__ unsigned top_halves(unsigned second, unsigned first) {   // bf16 of two fp32, by truncation
    return __builtin_amdgcn_perm(second, first, 0x07060302);
}
__device__ __forceinline__ Bf16x3 bf16x3_of(const v4f &p, const v4f &q) {
    unsigned h[8], m[8], l[8];
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const float a = e < 4 ? p[e] : q[e - 4];
        // a signalling NaN whose payload sits in the low 16 bits only would be cut to an infinity: the canonical form has a
        // quiet bit, which the cut keeps (one instruction; other values pass unchanged)
        h[e] = __float_as_uint(__builtin_canonicalizef(a));
        float r = a - __uint_as_float(h[e] & 0xffff0000u);
        r = __builtin_amdgcn_fmed3f(r, r, 0.0f);     // NaN (a infinite or NaN) -> 0, anything else unchanged
        m[e] = __float_as_uint(r);
        l[e] = __float_as_uint(r - __uint_as_float(m[e] & 0xffff0000u));
    }
    Bf16x3 o;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        o.hi[e] = (int)top_halves(h[2 * e + 1], h[2 * e]);
        o.mid[e] = (int)top_halves(m[2 * e + 1], m[2 * e]);
        o.lo[e] = (int)top_halves(l[2 * e + 1], l[2 * e]);
    }
    return o;
}
// fp32 x fp32 products in bf16 terms: each operand is taken times 2^24 and cut into three terms rounded to nearest, hi + mid + lo = a
// exactly (hi keeps 8 significant bits, a - hi at most 16, a - hi - mid at most 8), and the product is formed of six products of
// terms on the bf16 matrix core and taken times 2^-48.  (Henry, Tang and Heinecke, "Leveraging the bfloat16 Artificial Intelligence
// Datatype For Higher-Precision Computations", 2019, describe such splits.)  Of the nine products of terms mid lo, lo mid and lo lo
// are left out: together at most 2^-24 of the product, of either sign.
// The factor 2^24: the bf16 matrix core takes denormal operands as zero.  Every finite float times 2^24 is a multiple of 2^-125, and so
// are its terms: none of them is denormal, whatever the float.  Without it the cut loses bits below 2^-102, which GELU and softmax
// produce in ordinary use; sending tiles that hold such values through fp32 instructions cost a feed-forward block on trained-like
// activations (2048 x 1024 x 4096, pre-activations of standard deviation 2) 329 us where it takes 203.
// What the terms cannot hold shows in the sums: operands from about 2^104 up, infinities and NaNs, and sums past 2^80 leave an infinity or a
// NaN in every sum they enter.  The kernels look at their sums (look_at, any_wave) and form such tiles again with fp32 instructions.
// Per pair of values: two products, three conversions, four shifts or masks, four subtractions.
typedef int v2i __attribute__((ext_vector_type(2)));
constexpr float TERMS_UP = 16777216.0f, TERMS_DOWN = 1.0f / (TERMS_UP * TERMS_UP);
__device__ __forceinline__ void bf16x3_nearest(float a, float b, int &hi, int &mid, int &lo) {
    typedef float v2f __attribute__((ext_vector_type(2)));
    typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
    auto two = [](float x, float y) { return __builtin_bit_cast(int, __builtin_convertvector(v2f{x, y}, v2bf)); };
    auto first = [](int p) { return __uint_as_float((unsigned)p << 16); };
    auto second = [](int p) { return __uint_as_float((unsigned)p & 0xffff0000u); };
    hi = two(a, b);
    const float ra = a - first(hi), rb = b - second(hi);
    mid = two(ra, rb);
    lo = two(ra - first(mid), rb - second(mid));
}
template <int E> using Term = std::conditional_t<E == 8, v4i, v2i>;      // E bf16 values: 8 or 4
template <int E>
__device__ __forceinline__ void cut(const float (&x)[E], float up, Term<E> (&t)[3]) {
#pragma unroll
    for (int e = 0; e < E; e += 2) {
        int hi, mid, lo;
        bf16x3_nearest(x[e] * up, x[e + 1] * up, hi, mid, lo);
        t[0][e / 2] = hi;
        t[1][e / 2] = mid;
        t[2][e / 2] = lo;
    }
}
__device__ __forceinline__ v16f mfma_terms(const v4i &a, const v4i &b, const v16f &c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
}
// seen, starting at zero, stays zero while every sum looked at is finite
__device__ __forceinline__ void look_at(const v16f &sum, float &seen) {
#pragma unroll
    for (int v = 0; v < 16; v++) seen = __builtin_fmaf(sum[v], 0.0f, seen);
}
// Whether any lane of the workgroup's WAVES waves (a multiple of four) says so, through a word of LDS per wave.  Every wave calls it; it holds a barrier.
template <int WAVES>
__device__ __forceinline__ bool any_wave(bool says, unsigned char *words, int wave) {
    int *word = reinterpret_cast<int *>(words);
    const bool mine = __builtin_amdgcn_ballot_w64(says) != 0;
    if ((threadIdx.x & 63) == 0) word[wave] = mine;
    __syncthreads();
    int any = 0;
#pragma unroll
    for (int w = 0; w < WAVES; w += 4) {
        const v4i four = *reinterpret_cast<const v4i *>(word + w);
        any |= four[0] | four[1] | four[2] | four[3];
    }
    return __builtin_amdgcn_readfirstlane(any) != 0;
}
__device__ __forceinline__ v4i bf16_of_i8(int first, int second) {   // two k-blocks of four int8 -> 8 bf16
    unsigned f[8];
#pragma unroll
    for (int e = 0; e < 8; e++) f[e] = __float_as_uint((float)(signed char)((e < 4 ? first : second) >> (8 * (e & 3))));
    v4i o;
#pragma unroll
    for (int e = 0; e < 4; e++) o[e] = (int)top_halves(f[2 * e + 1], f[2 * e]);
    return o;
}

}  // namespace axhip
