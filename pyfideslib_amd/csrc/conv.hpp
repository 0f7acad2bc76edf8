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

}  // namespace fides
