// 64-bit modular arithmetic for CDNA4 (gfx950), built from 32-bit multiplies.
//
// CDNA4 has no 64x64-bit integer multiply; the compiler lowers the pieces
// below to v_mul_hi_u32 / v_mul_lo_u32 / v_mad_u64_u32.  Every routine returns
// the exact residue (or an exact residue plus a stated multiple of p when
// named *_lazy).  Moduli below 2^50 have a second, equally exact form on
// the FP64 units (fp_mul): every value is an integer below 2^53 in magnitude,
// every product the exact pair (rounded product, fma remainder), so rounding
// only ever picks the multiple of p that is taken off, never a residue's digit.
//
// Reference counterparts: FIDESlib src/ModMult.cuh:46-74 (Barrett),
// :96-102 (Shoup), :288-313 (128-bit reduce), src/AddSub.cuh:37-50.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace fides {

// Per-prime constants used by the kernels.
struct PrimeInfo {
    uint64_t p;      // modulus, < 2^60
    uint64_t mu;     // floor(2^(n+63) / p), n = bit length of p
    uint32_t nbits;  // n
    uint32_t fp;     // 1: p < 2^FP_BITS, the transforms run in FP64 (FpArith)
    uint64_t p2;     // 2p
    double pd, pinv; // p and 1/p, rounded to nearest
};

// Largest modulus of the exact FP64 transforms: every intermediate is an
// integer of magnitude below 8p <= 2^53.
constexpr int FP_BITS = 50;

// Pair (w, floor(w * 2^64 / p)) for Shoup multiplication by the constant w.
struct ShoupConst {
    uint64_t w, wp;
};

__device__ __forceinline__ uint64_t mulhi64(uint64_t a, uint64_t b) { return __umul64hi(a, b); }

// Full 128-bit product with four 32x32->64 multiply-adds.
__device__ __forceinline__ void mul128(uint64_t a, uint64_t b, uint64_t& lo, uint64_t& hi) {
    const uint32_t a0 = (uint32_t)a, a1 = (uint32_t)(a >> 32);
    const uint32_t b0 = (uint32_t)b, b1 = (uint32_t)(b >> 32);
    const uint64_t p00 = (uint64_t)a0 * b0;
    const uint64_t p01 = (uint64_t)a0 * b1 + (p00 >> 32);
    const uint64_t p10 = (uint64_t)a1 * b0 + (uint32_t)p01;
    hi = (uint64_t)a1 * b1 + (p01 >> 32) + (p10 >> 32);
    lo = (p10 << 32) | (uint32_t)p00;
}

// (lo, hi) += a * b   (caller guarantees no overflow of the 128-bit sum)
__device__ __forceinline__ void mac128(uint64_t& lo, uint64_t& hi, uint64_t a, uint64_t b) {
    uint64_t pl, ph;
    mul128(a, b, pl, ph);
    lo += pl;
    hi += ph + (lo < pl);
}

// Barrett reduction of X = hi*2^64 + lo, valid for X < 2^(n+63):
// qhat = floor((X >> (n-1)) * mu / 2^64) is within 2 of floor(X/p).
__device__ __forceinline__ uint64_t reduce128(uint64_t lo, uint64_t hi, const PrimeInfo& P) {
    const uint32_t s = P.nbits - 1;
    const uint64_t xs = (lo >> s) | (hi << (64 - s));
    const uint64_t q = mulhi64(xs, P.mu);
    uint64_t r = lo - q * P.p;
    r = r >= P.p2 ? r - P.p2 : r;
    return r >= P.p ? r - P.p : r;
}

// The same before its last subtractions: in [0, 3p).
__device__ __forceinline__ uint64_t reduce128_lazy(uint64_t lo, uint64_t hi, const PrimeInfo& P) {
    const uint32_t s = P.nbits - 1;
    const uint64_t xs = (lo >> s) | (hi << (64 - s));
    return lo - mulhi64(xs, P.mu) * P.p;
}

// Reduce a single 64-bit value (< 2^64) modulo p.
__device__ __forceinline__ uint64_t reduce64(uint64_t x, const PrimeInfo& P) { return reduce128(x, 0, P); }

__device__ __forceinline__ uint64_t mulmod(uint64_t a, uint64_t b, const PrimeInfo& P) {
    uint64_t lo, hi;
    mul128(a, b, lo, hi);
    return reduce128(lo, hi, P);
}

// x w - q p for a quotient q of x w / p that is off by little
__device__ __forceinline__ uint64_t shoup_rest(uint64_t x, uint64_t w, uint64_t q, uint64_t p) {
    // x w + q (-p): both low products accumulate into one pair of registers
    const uint64_t n = 0 - p;
    const uint32_t x0 = (uint32_t)x, x1 = (uint32_t)(x >> 32), w0 = (uint32_t)w, w1 = (uint32_t)(w >> 32);
    const uint32_t q0 = (uint32_t)q, q1 = (uint32_t)(q >> 32), n0 = (uint32_t)n, n1 = (uint32_t)(n >> 32);
    const uint64_t t = (uint64_t)q0 * n0 + (uint64_t)x0 * w0;
    const uint32_t h = (uint32_t)(t >> 32) + x0 * w1 + x1 * w0 + q0 * n1 + q1 * n0;
    return ((uint64_t)h << 32) | (uint32_t)t;
}
// Shoup: x * w mod p with x < 2^64, w < p; lazy result in [0, 2p).
__device__ __forceinline__ uint64_t mul_shoup_lazy(uint64_t x, uint64_t w, uint64_t wp, uint64_t p) {
    return shoup_rest(x, w, mulhi64(x, wp), p);
}
// The same in [0, 4p): of the quotient's four partial products the lowest is left
// out and the two middle ones enter by their upper words, each less than 1 off.  12
// instructions against 17, which leaves 22 a forward butterfly against 27 also with the
// reduction that the wider bound asks for every two stages instead of every four: a product
// at N = 2^16, level 24 (its special primes' transforms) 183.6 -> 181.4 us.
__device__ __forceinline__ uint64_t mul_shoup_lazy4(uint64_t x, uint64_t w, uint64_t wp, uint64_t p) {
    const uint32_t x0 = (uint32_t)x, x1 = (uint32_t)(x >> 32), p0 = (uint32_t)wp, p1 = (uint32_t)(wp >> 32);
    const uint64_t q = (uint64_t)x1 * p1 + __umulhi(x0, p1) + __umulhi(x1, p0);
    return shoup_rest(x, w, q, p);
}
__device__ __forceinline__ uint64_t mul_shoup(uint64_t x, uint64_t w, uint64_t wp, uint64_t p) {
    const uint64_t r = mul_shoup_lazy(x, w, wp, p);
    return r >= p ? r - p : r;
}

// x or x - m, whichever is in [0, m) for x < 2m
__device__ __forceinline__ uint64_t csub(uint64_t x, uint64_t m) { return x >= m ? x - m : x; }

__device__ __forceinline__ uint64_t addmod(uint64_t a, uint64_t b, uint64_t p) {
    const uint64_t s = a + b;
    return s >= p ? s - p : s;
}
__device__ __forceinline__ uint64_t submod(uint64_t a, uint64_t b, uint64_t p) {
    return a >= b ? a - b : a + p - b;
}

// ---- exact FP64 residues (p < 2^50) ----
// x w mod p as a signed integer: x w = h + l exactly, q is within 1/2 + 3 2^-53
// |x w| / p of x w / p, and h - q p is an integer below 2^53, so the fma and
// the sum are exact.  With |x| <= B p (B <= 8) and |w| <= p / 2 the result is at
// most (1/2 + 3 B / 16) p in magnitude; |w| < p doubles the second term.  6
// instructions at the rate of one 32-bit multiply each (a Shoup product: 9
// multiplies and 3 adds in mul_shoup_lazy4's form).
__device__ __forceinline__ double fp_mul(double x, double w, double p, double pinv) {
    const double h = x * w;
    const double l = __builtin_fma(x, w, -h);
    const double q = __builtin_rint(h * pinv);
    return __builtin_fma(-q, p, h) + l;
}
// x mod p, centered: |result| <= p / 2 + 1 for |x| <= 8p
__device__ __forceinline__ double fp_reduce(double x, double p, double pinv) {
    return __builtin_fma(-__builtin_rint(x * pinv), p, x);
}
// an integer below 2^52 as a double, and a non-negative one back
__device__ __forceinline__ double fp_from(uint64_t x) {
    return __longlong_as_double((long long)(x | 0x4330000000000000ull)) - 0x1p52;
}
__device__ __forceinline__ uint64_t fp_to(double x) {
    return (uint64_t)__double_as_longlong(x + 0x1p52) & 0x000fffffffffffffull;
}
// the residue in [0, p) of |x| <= 8p
__device__ __forceinline__ uint64_t fp_canon(double x, double p, double pinv) {
    const double r = fp_reduce(x, p, pinv);
    return fp_to(r < 0 ? r + p : r);
}

__device__ __forceinline__ uint32_t brev_bits(uint32_t x, int bits) { return __brev(x) >> (32 - bits); }
// the same for bits >= 0
__device__ __forceinline__ uint32_t brev_low(uint32_t x, int bits) { return bits ? brev_bits(x, bits) : 0u; }

}  // namespace fides
