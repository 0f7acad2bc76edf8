// Base-conversion sums shared by the plain and the fused conversion kernels.
#pragma once
#include "engine.hpp"

namespace fides {

__device__ __forceinline__ int num_digits(const DevTables& T, int nl) {
    const int n = (nl + T.alpha - 1) / T.alpha;
    return n < T.dnum ? n : T.dnum;
}

// Two adjacent coefficients per thread through 16-byte accesses.
struct u64x2 {
    uint64_t x, y;
};
typedef uint64_t v2u64 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(1))) v2u64 gv2u64;
__device__ __forceinline__ u64x2 ld2(const uint64_t* p) {
    const v2u64 v = *(const gv2u64*)p;
    return u64x2{v.x, v.y};
}
__device__ __forceinline__ void st2(uint64_t* p, uint64_t a, uint64_t b) { *(gv2u64*)p = v2u64{a, b}; }

// Carry-free sum of products: residues (< 2^60) are split into 30-bit halves,
// so every partial product is below 2^60 and up to 16 terms accumulate in four
// 64-bit registers with one v_mad_u64_u32 each and no carry handling;
// combine() forms the exact 128-bit sum once.
struct Acc4 {
    uint64_t s00 = 0, s01 = 0, s10 = 0, s11 = 0;
};
struct Half2 {
    uint32_t lo, hi;  // x = hi * 2^30 + lo
};
__device__ __forceinline__ Half2 split30(uint64_t x) { return Half2{(uint32_t)(x & 0x3fffffffu), (uint32_t)(x >> 30)}; }
// The halves of a value that stays in registers through a kernel: as words of
// their own, or the compiler keeps the 64-bit values that they were cut from.
__device__ __forceinline__ Half2 split30_held(uint64_t x) {
    Half2 h = split30(x);
    asm("" : "+v"(h.lo), "+v"(h.hi));
    return h;
}
__device__ __forceinline__ void mac_split(Acc4& a, Half2 x, Half2 y) {
    a.s00 = (uint64_t)x.lo * y.lo + a.s00;
    a.s01 = (uint64_t)x.lo * y.hi + a.s01;
    a.s10 = (uint64_t)x.hi * y.lo + a.s10;
    a.s11 = (uint64_t)x.hi * y.hi + a.s11;
}
// X = s11 2^60 + (s01 + s10) 2^30 + s00 as (lo, hi)
__device__ __forceinline__ void combine(const Acc4& a, uint64_t& lo, uint64_t& hi) {
    lo = a.s00;
    hi = 0;
    uint64_t t = a.s01 << 30;
    lo += t;
    hi += (a.s01 >> 34) + (lo < t);
    t = a.s10 << 30;
    lo += t;
    hi += (a.s10 >> 34) + (lo < t);
    t = a.s11 << 60;
    lo += t;
    hi += (a.s11 >> 4) + (lo < t);
}

template <int A>
struct MatRow {
    uint64_t v[A];
};

// sum x_i m_i mod p as a double of at most (1/2 + 2^-15) p, exact, for p < 2^50, A <= 12
// and x_i < 2^60.  The halves of x_i take constants of their own, so that two
// signed sums are enough, U of lo and V of hi parts: |U| < 24 2^58, |V| <= 24 2^50, and
// U with the low word of V on top stays below 2^63.
// V 2^29 + U is regrouped as D 2^32 + l, D an integer below 2^53 and l one word,
// and is at most 12 2^30 p, so its rounded quotient is off by little and what is
// left after it a small integer.  11 operations follow the sums, where four
// unsigned sums and a 128-bit reduction took 45.
template <int A>
struct MatRowFp {
    ConvFp v[A];
};
template <int A>
__device__ __forceinline__ double conv_fp(const Half2* x, const MatRowFp<A>& row, const PrimeInfo& P) {
    int64_t u = 0, v = 0;
#pragma unroll
    for (int i = 0; i < A; ++i) {
        const int64_t xl = (int32_t)x[i].lo, xh = (int32_t)x[i].hi;
        u = xl * row.v[i].lo + u;
        v = xl * row.v[i].hi + v;
        u = xh * row.v[i].lo30 + u;
        v = xh * row.v[i].hi30 + v;
    }
    u = (int64_t)((uint64_t)(uint32_t)v * 0x20000000u + (uint64_t)u);
    const double h = __builtin_fma((double)(int32_t)(v >> 32), 0x1p29, (double)(int32_t)(u >> 32)) * 0x1p32;
    const double l = (double)(uint32_t)u;
    return __builtin_fma(-__builtin_rint((h + l) * P.pinv), P.pd, h) + l;
}

}  // namespace fides
