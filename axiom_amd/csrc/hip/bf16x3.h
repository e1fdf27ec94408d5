// fp32 values as sums of bf16 terms, for products on the bf16 matrix core that keep every bit of the fp32 operand.
#pragma once
#include "common.h"

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
// fp32 x fp32 products in bf16 terms: each operand cut into three terms rounded to nearest, hi + mid + lo = a exactly (hi keeps 8
// significant bits, a - hi at most 16, a - hi - mid at most 8).  Of the nine products of terms the three smallest (mid lo,
// lo mid, lo lo: below 2^-25 of the product, of either sign) are left out.  Exact for magnitudes from 2^-102 up to where
// rounding to bf16 overflows; the caller looks after the others.  Per pair: three conversions, four shifts or masks, four
// subtractions.
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
