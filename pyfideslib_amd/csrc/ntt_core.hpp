// Device code shared by the transform kernels: the two arithmetics, the phase
// machinery of one sub-transform (registers + LDS exchanges) and job lookup.
#pragma once
#include <type_traits>

#include "engine.hpp"

namespace fides {

__device__ __forceinline__ uint32_t lds_off(uint32_t e) { return e + (e >> 4); }

// Arithmetic of one limb's transform, picked per block by the limb's prime
// (wave-uniform): IntArith (any p < 2^60; Harvey-lazy Shoup butterflies on
// 64-bit words) or FpArith (p < 2^50; exact FP64 butterflies, modarith.hpp's
// fp_mul).  An FP64 butterfly is 8 to 9 instructions against about 22, and its
// twiddles are 8 bytes against 16.
//
// Bounds of the FP64 values, in units of p (every step must stay below 8):
// fp_mul of a value B returns at most 1/2 + 3B/16.  Forward: U +- V grows B to
// 19B/16 + 1/2 per stage -- 1, 1.69, 2.50, 3.47, 4.62 over four stages from a
// residue -- so U is reduced (to 1/2) in the first stage of every phase that
// starts a multiple of 4 stages into the pass (every phase of 3 stages), a
// residue's first phase excepted; entering with B <= 5.1 four stages end at
// 1.96, 2.83, 3.86, 5.08.  Inverse: a sum doubles B, so the sums of every
// second stage, and of a pass's last, are reduced: two stages take B to at most
// max(1/2, 1/2 + 3B/4) < 2, with no value above 4B < 8 on the way.
struct IntArith {
    using V = uint64_t;
    using W = ShoupConst;
    uint64_t p;
    __device__ __forceinline__ explicit IntArith(const PrimeInfo& P) : p(P.p) {}
    static __device__ __forceinline__ const W* fwd(const DevTables& T) { return T.tw_fwd; }
    static __device__ __forceinline__ const W* inv(const DevTables& T) { return T.tw_inv; }
    __device__ __forceinline__ V from(uint64_t x) const { return x; }
    static __device__ __forceinline__ V unpack(uint64_t m) { return m; }
    static __device__ __forceinline__ uint64_t pack(V v) { return v; }
    // every stage adds 4p to the bound (any 64-bit b will do): U is brought below
    // 8p at the start of every phase of two stages, and below 4p at that of
    // three (RED 2), so what a phase leaves is below 16p < 2^64
    static constexpr bool EACH_PHASE = true;
    template <int RED>
    __device__ __forceinline__ void fwd_bf(V& a, V& b, const W& w) const {
        const uint64_t U = RED == 2 ? csub(csub(a, 8 * p), 4 * p) : RED == 1 ? csub(a, 8 * p) : a;
        const uint64_t X = mul_shoup_lazy4(b, w.w, w.wp, p);
        a = U + X;
        b = U - X + 4 * p;
    }
    // inputs in [0, 4p), outputs in [0, 4p)
    template <bool RED>
    __device__ __forceinline__ void inv_bf(V& a, V& b, const W& w) const {
        const uint64_t U = a;
        a = csub(U + b, 4 * p);
        b = mul_shoup_lazy4(U - b + 4 * p, w.w, w.wp, p);
    }
    __device__ __forceinline__ void inv_last(V& a, V& b, const ShoupConst& s, const ShoupConst& ws) const {
        const uint64_t U = a, X = b;
        a = mul_shoup_lazy4(U + X, s.w, s.wp, p);
        b = mul_shoup_lazy4(U - X + 4 * p, ws.w, ws.wp, p);
    }
    // the residue of a forward output in [0, 16p), of an inverse one in [0, 4p)
    __device__ __forceinline__ uint64_t canon_fwd(V x) const { return csub(term_fwd(x), p); }
    __device__ __forceinline__ uint64_t canon_inv(V x) const { return csub(csub(x, 2 * p), p); }
    // a b, a b + c d as residues
    __device__ __forceinline__ uint64_t mul(uint64_t a, uint64_t b, const PrimeInfo& P) const { return mulmod(a, b, P); }
    __device__ __forceinline__ uint64_t mul2(uint64_t a, uint64_t b, uint64_t c, uint64_t d,
                                             const PrimeInfo& P) const {
        uint64_t lo, hi;
        mul128(a, b, lo, hi);
        mac128(lo, hi, c, d);
        return reduce128(lo, hi, P);
    }
    // the residue of a value below 3p (reduce128_lazy)
    __device__ __forceinline__ V from_lazy(uint64_t x) const { return csub(csub(x, 2 * p), p); }
    // a forward output as an inner product's term, in [0, 2p)
    __device__ __forceinline__ V term_fwd(V x) const { return csub(csub(csub(x, 8 * p), 4 * p), 2 * p); }
    // sum of at most 4 products x k with x < 2p, k < p (below 8p^2 < 2^(bits(p) +
    // 63), one reduction), as an inverse transform's input
    struct Sum {
        uint64_t lo = 0, hi = 0;
    };
    __device__ __forceinline__ void mac(Sum& s, V x, uint64_t k) const { mac128(s.lo, s.hi, x, k); }
    __device__ __forceinline__ V sum(const Sum& s, const PrimeInfo& P) const { return reduce128(s.lo, s.hi, P); }
    // the residue of an inverse transform's input
    __device__ __forceinline__ uint64_t canon_in(V x) const { return x; }
    // e c + f as an inverse transform's input
    __device__ __forceinline__ V mul_add(V e, const ShoupConst& c, uint64_t f) const {
        return addmod(mul_shoup(e, c.w, c.wp, p), f, p);
    }
    // y c + s for a conversion's sum y (from_lazy) and a residue s, as a forward input
    __device__ __forceinline__ V scale_add(V y, const ShoupConst& c, uint64_t s) const {
        return addmod(mul_shoup(y, c.w, c.wp, p), s, p);
    }
    // (e - v) c,  (e - v) c + f,  (e c + f - v) d  for residues e, f, c, d
    __device__ __forceinline__ uint64_t sub_mul(uint64_t e, V v, const ShoupConst& c) const {
        return mul_shoup(e + 8 * p - csub(v, 8 * p), c.w, c.wp, p);
    }
    __device__ __forceinline__ uint64_t sub_mul_add(uint64_t e, V v, const ShoupConst& c, uint64_t f) const {
        return addmod(sub_mul(e, v, c), f, p);
    }
    __device__ __forceinline__ uint64_t prod_sub_mul(uint64_t e, uint64_t f, V v, const ShoupConst& d,
                                                     const PrimeInfo& P) const {
        return sub_mul(mul(e, f, P), v, d);
    }
    __device__ __forceinline__ uint64_t mul_add_sub_mul(uint64_t e, const ShoupConst& c, uint64_t f, V v,
                                                        const ShoupConst& d) const {
        return mul_shoup(mul_shoup_lazy(e, c.w, c.wp, p) + f + 8 * p - csub(v, 8 * p), d.w, d.wp, p);
    }
};
struct FpArith {
    using V = double;
    using W = double;
    double p, pinv;
    __device__ __forceinline__ explicit FpArith(const PrimeInfo& P) : p(P.pd), pinv(P.pinv) {}
    static __device__ __forceinline__ const W* fwd(const DevTables& T) { return T.twd_fwd; }
    static __device__ __forceinline__ const W* inv(const DevTables& T) { return T.twd_inv; }
    __device__ __forceinline__ V from(uint64_t x) const { return fp_from(x); }
    // between the two passes a limb holds the doubles themselves
    static __device__ __forceinline__ V unpack(uint64_t m) { return __longlong_as_double((long long)m); }
    static __device__ __forceinline__ uint64_t pack(V v) { return (uint64_t)__double_as_longlong(v); }
    static constexpr bool EACH_PHASE = false;
    template <int RED>
    __device__ __forceinline__ void fwd_bf(V& a, V& b, W w) const {
        const double U = RED ? fp_reduce(a, p, pinv) : a;
        const double X = fp_mul(b, w, p, pinv);
        a = U + X;
        b = U - X;
    }
    template <bool RED>
    __device__ __forceinline__ void inv_bf(V& a, V& b, W w) const {
        const double U = a, X = b;
        a = RED ? fp_reduce(U + X, p, pinv) : U + X;
        b = fp_mul(U - X, w, p, pinv);
    }
    __device__ __forceinline__ void inv_last(V& a, V& b, const ShoupConst& s, const ShoupConst& ws) const {
        const double U = a, X = b;
        a = fp_mul(U + X, fp_from(s.w), p, pinv);
        b = fp_mul(U - X, fp_from(ws.w), p, pinv);
    }
    __device__ __forceinline__ uint64_t canon_fwd(V x) const { return fp_canon(x, p, pinv); }
    __device__ __forceinline__ uint64_t canon_inv(V x) const { return fp_canon(x, p, pinv); }
    __device__ __forceinline__ uint64_t mul(uint64_t a, uint64_t b, const PrimeInfo&) const {
        return fp_canon(fp_mul(fp_from(a), fp_from(b), p, pinv), p, pinv);
    }
    __device__ __forceinline__ uint64_t mul2(uint64_t a, uint64_t b, uint64_t c, uint64_t d, const PrimeInfo&) const {
        return fp_canon(fp_mul(fp_from(a), fp_from(b), p, pinv) + fp_mul(fp_from(c), fp_from(d), p, pinv), p, pinv);
    }
    __device__ __forceinline__ V term_fwd(V x) const { return fp_reduce(x, p, pinv); }
    // |x| <= p, k < p: each product at most (1/2 + 3/8) p, four of them below 4p
    using Sum = double;
    __device__ __forceinline__ void mac(Sum& s, V x, uint64_t k) const { s += fp_mul(x, fp_from(k), p, pinv); }
    __device__ __forceinline__ V sum(Sum s, const PrimeInfo&) const { return fp_reduce(s, p, pinv); }
    __device__ __forceinline__ uint64_t canon_in(V x) const { return fp_to(x < 0 ? x + p : x); }  // reduced before
    __device__ __forceinline__ V mul_add(V e, const ShoupConst& c, uint64_t f) const {
        return fp_reduce(fp_mul(e, fp_from(c.w), p, pinv) + fp_from(f), p, pinv);
    }
    // at most (1/2 + 9/8 + 1) p, a first phase's bound
    __device__ __forceinline__ V scale_add(V y, const ShoupConst& c, double s) const {
        return fp_mul(y, fp_from(c.w), p, pinv) + s;
    }
    // uncentered constants: fp_mul of a value B returns at most 1/2 + 3B/8; no sum below exceeds 7.1
    __device__ __forceinline__ uint64_t sub_mul(uint64_t e, V v, const ShoupConst& c) const {
        return fp_canon(fp_mul(fp_from(e) - v, fp_from(c.w), p, pinv), p, pinv);
    }
    __device__ __forceinline__ uint64_t sub_mul_add(uint64_t e, V v, const ShoupConst& c, uint64_t f) const {
        return fp_canon(fp_mul(fp_from(e) - v, fp_from(c.w), p, pinv) + fp_from(f), p, pinv);
    }
    __device__ __forceinline__ uint64_t prod_sub_mul(uint64_t e, uint64_t f, V v, const ShoupConst& d,
                                                     const PrimeInfo&) const {
        return fp_canon(fp_mul(fp_mul(fp_from(e), fp_from(f), p, pinv) - v, fp_from(d.w), p, pinv), p, pinv);
    }
    __device__ __forceinline__ uint64_t mul_add_sub_mul(uint64_t e, const ShoupConst& c, uint64_t f, V v,
                                                        const ShoupConst& d) const {
        const double y = fp_mul(fp_from(e), fp_from(c.w), p, pinv) + (fp_from(f) - v);
        return fp_canon(fp_mul(y, fp_from(d.w), p, pinv), p, pinv);
    }
};
// f(IntArith or FpArith of the prime); the class comes from the kernel
// arguments, so neither twiddle nor tile loads wait for the prime's constants
__device__ __forceinline__ bool is_fp(const DevTables& T, int pid) {
    return ((pid & 64 ? T.fpmask[1] : T.fpmask[0]) >> (pid & 63)) & 1;
}
template <class F>
__device__ __forceinline__ void with_arith(const DevTables& T, int pid, const PrimeInfo& P, F&& f) {
    if (is_fp(T, pid))
        f(FpArith(P));
    else
        f(IntArith(P));
}

// Element index (within a 2^K sub-transform) of register j of thread t in a
// phase over bits [LO, LO+NB); the LR-NB spare register bits and the thread
// bits fill the remaining positions from the bottom up.
template <int LR, int LO, int NB>
__device__ __forceinline__ uint32_t elem(uint32_t t, uint32_t j) {
    constexpr uint32_t EX = LR - NB;
    const uint32_t jlo = j & ((1u << NB) - 1);
    const uint32_t other = (t << EX) | (j >> NB);
    return (other & ((1u << LO) - 1)) | (jlo << LO) | ((other >> LO) << (LO + NB));
}

// Index of butterfly (j, j | 1<<bb) among the R/2 butterflies of a stage.
__device__ __forceinline__ constexpr int bfly(int j, int bb) { return ((j >> (bb + 1)) << bb) | (j & ((1 << bb) - 1)); }

// Twiddle slot of a butterfly: phases visit the K bits in a fixed order (top
// down for the forward transform, bottom up for the inverse); `done` bits
// precede the phase, s is the stage's rank inside the phase.
template <int LR>
__device__ __forceinline__ constexpr int slot(int done, int s, int j, int bb) {
    return (done + s) * (1 << (LR - 1)) + bfly(j, bb);
}

// ---- LDS exchange between phases ----
template <int LR, int LO, int NB, class V>
__device__ __forceinline__ void lds_get(const V* sub, uint32_t t, V* v) {
#pragma unroll
    for (int j = 0; j < (1 << LR); ++j) v[j] = sub[lds_off(elem<LR, LO, NB>(t, j))];
}
template <int LR, int LO, int NB, class V>
__device__ __forceinline__ void lds_put(V* sub, uint32_t t, const V* v) {
#pragma unroll
    for (int j = 0; j < (1 << LR); ++j) sub[lds_off(elem<LR, LO, NB>(t, j))] = v[j];
}

// Phase boundaries of a K-bit sub-transform with up to LR bits per phase.
// Forward phases run from the top bit down: the first covers bits
// [K - NB, K), the last [0, fwd_last_nb).  Inverse phases run from bit 0 up:
// the first covers [0, NB), the last [inv_last_lo, K).
template <int LR, int K>
constexpr int first_nb() { return K < LR ? K : LR; }
template <int LR, int K>
constexpr int fwd_last_nb() { return K % LR == 0 ? LR : K % LR; }
template <int LR, int K>
constexpr int inv_last_lo() { return LR * ((K - 1) / LR); }

// ---- forward (Cooley-Tukey), bits processed from the top down ----
// RED: the first stage of the phase reduces its U (the arithmetic's bound).
template <int LR, int K, int LO, int NB, int RED, class A, class TW>
__device__ __forceinline__ void fwd_bfly(const A& ar, typename A::V* v, uint32_t t, const TW& tw) {
    constexpr int R = 1 << LR;
#pragma unroll
    for (int bb = NB - 1; bb >= 0; --bb) {
#pragma unroll
        for (int j = 0; j < R; ++j) {
            if (j & (1 << bb)) continue;
            const auto w = tw(slot<LR>(K - LO - NB, NB - 1 - bb, j, bb), LO + bb, elem<LR, LO, NB>(t, j));
            if (bb == NB - 1)
                ar.template fwd_bf<RED>(v[j], v[j | (1 << bb)], w);
            else
                ar.template fwd_bf<0>(v[j], v[j | (1 << bb)], w);
        }
    }
}

// Forward phases from bit HI down to 0.  On entry v holds the elements of the
// phase that starts at HI (the caller loads them straight from global memory
// for the first phase); phases exchange through LDS; on exit v holds the
// elements of the last phase (bits [0, fwd_last_nb)), which the caller stores
// straight to global memory.  One barrier per exchange: a thread writes back
// exactly the elements it read, so reads and writes of one phase never race.
// That holds within a pass: whoever runs another pass on the same LDS waits first
// (lds_sync).
// hook(integral_constant<HI>) runs at the start of each phase (the row pass
// issues later phases' twiddle loads there).
template <bool WAVE>
__device__ __forceinline__ void lds_sync() {
    if constexpr (WAVE) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    } else {
        __syncthreads();
    }
}
struct NoHook {
    template <class X>
    __device__ __forceinline__ void operator()(X) const {}
};
// FRESH: the pass starts from residues in [0, p).
template <int LR, int K, int HI, bool FRESH, bool WAVE = false, class A, class TW, class HOOK = NoHook>
__device__ __forceinline__ void fwd_run(const A& ar, typename A::V* sub, typename A::V* v, uint32_t t, const TW& tw,
                                        const HOOK& hook = HOOK{}) {
    constexpr int NB = HI < LR ? HI : LR;
    constexpr int LO = HI - NB;
    constexpr int RED = FRESH && HI == K   ? 0
                        : A::EACH_PHASE    ? (LR == 3 ? 2 : 1)
                        : (K - HI) % 4 == 0 || LR == 3 ? 1
                                                       : 0;
    hook(std::integral_constant<int, HI>{});
    fwd_bfly<LR, K, LO, NB, RED>(ar, v, t, tw);
    if constexpr (LO > 0) {
        constexpr int NB2 = LO < LR ? LO : LR;
        lds_put<LR, LO, NB>(sub, t, v);
        lds_sync<WAVE>();
        lds_get<LR, LO - NB2, NB2>(sub, t, v);
        fwd_run<LR, K, LO, FRESH, WAVE>(ar, sub, v, t, tw, hook);
    }
}

// Prefetch of the forward twiddles into twr[] in slot order; IDX(b, e) gives
// the table index of the twiddle of stage bit b at lower element e.
// The twiddles of the one phase that starts at bit HI (none when HI <= 0).
template <int LR, int K, int HI, class W, class IDX>
__device__ __forceinline__ void fwd_prefetch(W* twr, const W* tab, uint32_t t, const IDX& idx) {
    if constexpr (HI > 0) {
        constexpr int NB = HI < LR ? HI : LR;
        constexpr int LO = HI - NB;
#pragma unroll
        for (int bb = NB - 1; bb >= 0; --bb)
#pragma unroll
            for (int j = 0; j < (1 << LR); ++j)
                if (!(j & (1 << bb))) twr[slot<LR>(K - HI, NB - 1 - bb, j, bb)] = tab[idx(LO + bb, elem<LR, LO, NB>(t, j))];
    }
}

// ---- inverse (Gentleman-Sande), bits processed from the bottom up ----
// When SCALE, the stage on bit K-1 multiplies both outputs by the limb scale s
// (sum by s, difference by w*s).
template <int LR, int K, int LO, int NB, bool SCALE, class A, class TW>
__device__ __forceinline__ void inv_bfly(const A& ar, typename A::V* v, uint32_t t, const TW& tw, const ShoupConst& s,
                                         const ShoupConst& ws) {
    constexpr int R = 1 << LR;
#pragma unroll
    for (int bb = 0; bb < NB; ++bb) {
#pragma unroll
        for (int j = 0; j < R; ++j) {
            if (j & (1 << bb)) continue;
            const int j2 = j | (1 << bb);
            if (SCALE && LO + bb == K - 1) {
                ar.inv_last(v[j], v[j2], s, ws);
            } else {
                const auto w = tw(slot<LR>(LO, bb, j, bb), LO + bb, elem<LR, LO, NB>(t, j));
                if ((LO + bb) % 2 == 1 || LO + bb == K - 1)
                    ar.template inv_bf<true>(v[j], v[j2], w);
                else
                    ar.template inv_bf<false>(v[j], v[j2], w);
            }
        }
    }
}

// Inverse phases from bit LO up to K, register/LDS discipline as fwd_run: v
// enters with the elements of the phase starting at LO and leaves with those
// of the last phase (bits [inv_last_lo, K)).
template <int LR, int K, int LO, bool SCALE, bool WAVE = false, class A, class TW, class HOOK = NoHook>
__device__ __forceinline__ void inv_run(const A& ar, typename A::V* sub, typename A::V* v, uint32_t t, const TW& tw,
                                        const ShoupConst& s, const ShoupConst& ws, const HOOK& hook = HOOK{}) {
    constexpr int NB = (K - LO) < LR ? (K - LO) : LR;
    hook(std::integral_constant<int, LO>{});
    inv_bfly<LR, K, LO, NB, SCALE>(ar, v, t, tw, s, ws);
    if constexpr (LO + NB < K) {
        constexpr int LO2 = LO + NB;
        constexpr int NB2 = (K - LO2) < LR ? (K - LO2) : LR;
        lds_put<LR, LO, NB>(sub, t, v);
        lds_sync<WAVE>();
        lds_get<LR, LO2, NB2>(sub, t, v);
        inv_run<LR, K, LO2, SCALE, WAVE>(ar, sub, v, t, tw, s, ws, hook);
    }
}

// The twiddles of the one phase that starts at bit LO (none when LO >= K).
template <int LR, int K, int LO, class W, class IDX>
__device__ __forceinline__ void inv_prefetch(W* twr, const W* tab, uint32_t t, const IDX& idx) {
    if constexpr (LO < K) {
        constexpr int NB = (K - LO) < LR ? (K - LO) : LR;
#pragma unroll
        for (int bb = 0; bb < NB; ++bb)
#pragma unroll
            for (int j = 0; j < (1 << LR); ++j)
                if (!(j & (1 << bb))) twr[slot<LR>(LO, bb, j, bb)] = tab[idx(LO + bb, elem<LR, LO, NB>(t, j))];
    }
}


// ---- a "row": a sub-transform of K2 bits on contiguous words ----
// The second pass of a transform (row r of N1 = 2^K1).  RR rows per block of TR
// threads each, 2^LR values per thread.
template <int K1_, int K2_, int LR_, int W>
struct RowGeom {
    static constexpr int K1 = K1_, K2 = K2_, LR = LR_, R = 1 << LR_;
    static constexpr int N1 = 1 << K1_, N2 = 1 << K2_, N = N1 * N2;
    static constexpr int TR = N2 / R;
    static constexpr int RR = N1 < W ? N1 : W;
    static constexpr int NTR = TR * RR;
    static constexpr int SR = N2 + N2 / 16 + 1;
    // twiddle slots per thread: K2 stages x R/2 butterflies
    static constexpr int NS = K2 * (R / 2);
    // the threads of one row share a wave: its exchanges need no block barrier
    static constexpr bool WAVE = TR <= 64 && 64 % TR == 0;
    // first / last phase of the forward transform, and of the inverse
    static constexpr int NB1 = first_nb<LR, K2>(), LO1 = K2 - NB1, NBL = fwd_last_nb<LR, K2>();
    static constexpr int LOL = inv_last_lo<LR, K2>(), NBI = K2 - LOL;
    // word of the evaluation-form row held in slot j by thread t
    static __device__ __forceinline__ uint32_t mem(uint32_t t, int j) {
        return elem<LR, 0, NBL>(t, j);
    }
};

// Forward transform of one row: v enters with the elements of the first phase
// (elem<LR, LO1, NB1>) and leaves with the words mem(t, j).  hook runs at the
// start of each phase; each phase's twiddles are issued one phase early.
template <class G, bool FRESH, class A, class HOOK = NoHook>
__device__ __forceinline__ void fwd_row(const A& ar, typename A::V* sub, typename A::V* v, uint32_t t, uint32_t row,
                                        const typename A::W* tab, const HOOK& hook = HOOK{}) {
    auto idx = [&](int b, uint32_t e) { return (row << (G::K2 - 1 - b)) + (e >> (b + 1)); };
    typename A::W twr[G::NS];
    fwd_prefetch<G::LR, G::K2, G::K2>(twr, tab, t, idx);
    auto hk = [&](auto hi) {
        fwd_prefetch<G::LR, G::K2, decltype(hi)::value - G::LR>(twr, tab, t, idx);
        hook(hi);
    };
    auto twf = [&](int s, int, uint32_t) { return twr[s]; };
    fwd_run<G::LR, G::K2, G::K2, FRESH, G::WAVE>(ar, sub, v, t, twf, hk);
}

// Inverse transform of one row: v enters with the words mem(t, j) and leaves
// with the elements of the last phase (elem<LR, LOL, NBI>).
template <class G, class A>
__device__ __forceinline__ void inv_row(const A& ar, typename A::V* sub, typename A::V* v, uint32_t t, uint32_t row,
                                        const typename A::W* tab) {
    auto idx = [&](int b, uint32_t e) { return (row << (G::K2 - 1 - b)) + (e >> (b + 1)); };
    typename A::W twr[G::NS];
    inv_prefetch<G::LR, G::K2, 0>(twr, tab, t, idx);
    auto hk = [&](auto lo) { inv_prefetch<G::LR, G::K2, decltype(lo)::value + G::LR>(twr, tab, t, idx); };
    auto twf = [&](int k, int, uint32_t) { return twr[k]; };
    inv_run<G::LR, G::K2, 0, false, G::WAVE>(ar, sub, v, t, twf, ShoupConst{0, 0}, ShoupConst{0, 0}, hk);
}

// The epilogue operands of thread t's words (STORE_* of a forward transform).
template <class G, int STORE>
struct Epilogue {
    uint64_t e0[G::R], e1[G::R];
    // limb: the limb's first word within the polynomial (uniform), row: the row's within the limb
    __device__ __forceinline__ void load(const NttJob& J, size_t limb, uint32_t row, uint32_t t) {
        if constexpr (STORE == STORE_MODDOWN || STORE == STORE_MODDOWN_RESCALE || STORE == STORE_MODDOWN_AUTO ||
                      STORE == STORE_MODDOWN_INV) {
            const gu64* aux = gp(J.aux) + limb;
#pragma unroll
            for (int j = 0; j < G::R; ++j) e0[j] = aux[row + G::mem(t, j)];
            if (J.add) {
                const gu64* add = gp(J.add) + limb;
#pragma unroll
                for (int j = 0; j < G::R; ++j) e1[j] = add[row + G::mem(t, j)];
            } else {  // no addend: adding 0 is a no-op
#pragma unroll
                for (int j = 0; j < G::R; ++j) e1[j] = 0;
            }
        } else if constexpr (STORE == STORE_RESCALE) {
            const gu64* dst = gp(J.dst) + limb;
#pragma unroll
            for (int j = 0; j < G::R; ++j) e0[j] = dst[row + G::mem(t, j)];
        } else if constexpr (STORE == STORE_MUL_RESCALE) {
            const gu64 *a = gp(J.aux) + limb, *w = gp(J.add) + limb;
#pragma unroll
            for (int j = 0; j < G::R; ++j) e0[j] = a[row + G::mem(t, j)], e1[j] = w[row + G::mem(t, j)];
        }
    }
    // row r of the transform; sub: the row's LDS
    template <class A>
    __device__ __forceinline__ void store(const DevTables& T, const NttJob& J, int pos, int pid, const A& ar,
                                          uint64_t* sub, uint32_t t, uint32_t r, const typename A::V* v) const {
        gu64* dst = gp(J.dst) + (size_t)pos * G::N;
        const uint32_t row = r * G::N2;
        if constexpr (STORE == STORE_PLAIN) {
#pragma unroll
            for (int j = 0; j < G::R; ++j) dst[row + G::mem(t, j)] = ar.canon_fwd(v[j]);
        } else if constexpr (STORE == STORE_MODDOWN) {
            const ShoupConst pinv = cld(T.pinv + pid);
#pragma unroll
            for (int j = 0; j < G::R; ++j) dst[row + G::mem(t, j)] = ar.sub_mul_add(e0[j], v[j], pinv, e1[j]);
        } else if constexpr (STORE == STORE_MODDOWN_INV) {
            using V = typename A::V;
            const ShoupConst pinv = cld(T.pinv + pid);
            V u[G::R];
#pragma unroll
            for (int j = 0; j < G::R; ++j) {
                const uint64_t w = ar.sub_mul_add(e0[j], v[j], pinv, e1[j]);
                dst[row + G::mem(t, j)] = w;
                u[j] = ar.from(w);
            }
            lds_sync<G::WAVE>();  // the LDS reads before are done
            inv_row<G>(ar, reinterpret_cast<V*>(sub), u, t, G::N1 + r, A::inv(T) + (size_t)pid * G::N);
            gu64* mid = gp(J.mid) + (size_t)pos * G::N;
#pragma unroll
            for (int j = 0; j < G::R; ++j) mid[row + elem<G::LR, G::LOL, G::NBI>(t, j)] = A::pack(u[j]);
        } else if constexpr (STORE == STORE_MODDOWN_AUTO) {
            // Element jg = r N2 + e sits at exponent 2 brev(jg) + 1 =
            // 2 N1 brev(e) + 2 brev(r) + 1; times k (mod 2N) it lands at
            // row brev(((c mod 2N1) - 1) / 2), column brev((brev(e) k + (c >> (K1+1))) mod N2)
            // with c = (2 brev(r) + 1) k mod 2N: one destination row per row.
            const ShoupConst pinv = cld(T.pinv + pid);
            const uint32_t k = J.autok;
            const uint32_t cx = (uint32_t)(((2ull * brev_bits(r, G::K1) + 1) * k) & (2ull * G::N - 1));
            const uint32_t rdst = brev_bits((cx & (2u * G::N1 - 1)) >> 1, G::K1);
            const uint32_t coff = cx >> (G::K1 + 1);
            lds_sync<G::WAVE>();  // the LDS reads before are done
#pragma unroll
            for (int j = 0; j < G::R; ++j) {
                const uint32_t e2 = brev_bits((brev_bits(G::mem(t, j), G::K2) * k + coff) & (G::N2 - 1), G::K2);
                sub[lds_off(e2)] = ar.sub_mul_add(e0[j], v[j], pinv, e1[j]);
            }
            lds_sync<G::WAVE>();
            const uint32_t out = rdst * G::N2;
#pragma unroll
            for (int j = 0; j < G::R; ++j) dst[out + G::mem(t, j)] = sub[lds_off(G::mem(t, j))];
        } else if constexpr (STORE == STORE_MODDOWN_RESCALE) {
            // r = (acc P^-1 + add - v) q_l^-1  (see k_moddown_conv)
            const ShoupConst pinv = cld(T.pinv + pid);
            const ShoupConst qi = cld(T.qlinv + (size_t)J.level * (T.L + 1) + pid);
#pragma unroll
            for (int j = 0; j < G::R; ++j) dst[row + G::mem(t, j)] = ar.mul_add_sub_mul(e0[j], pinv, e1[j], v[j], qi);
        } else if constexpr (STORE == STORE_MUL_RESCALE) {
            const ShoupConst qi = cld(T.qlinv + (size_t)J.level * (T.L + 1) + pid);
            const PrimeInfo P = cld(T.primes + pid);
#pragma unroll
            for (int j = 0; j < G::R; ++j) dst[row + G::mem(t, j)] = ar.prod_sub_mul(e0[j], e1[j], v[j], qi, P);
        } else {  // STORE_RESCALE
            const ShoupConst qi = cld(T.qlinv + (size_t)J.level * (T.L + 1) + pid);
#pragma unroll
            for (int j = 0; j < G::R; ++j) dst[row + G::mem(t, j)] = ar.sub_mul(e0[j], v[j], qi);
        }
    }
};

// The limb scale of an inverse transform: N^-1, times a base-conversion factor.
__device__ __forceinline__ const ShoupConst* inv_scale(const DevTables& T, const NttJob& J, int pos, int pid) {
    if (J.scale_sel == ISCALE_MODUP) return T.iscale_modup + ((size_t)J.level * (T.L + 1) + pos) * 2;
    if (J.scale_sel == ISCALE_MODDOWN && pos >= J.nq) return T.iscale_moddown + (size_t)(pos - J.nq) * 2;
    return T.iscale_plain + (size_t)pid * 2;
}

// A q_l coefficient lifted centered into prime P (OpenFHE SwitchModulus).
struct SwitchLift {
    uint64_t half, qlmod;
    __device__ __forceinline__ SwitchLift(const DevTables& T, int level, int pid)
        : half(cld(T.primes + level).p >> 1), qlmod(cld(T.qlmodq + (size_t)level * (T.L + 1) + pid)) {}
    __device__ __forceinline__ uint64_t operator()(uint64_t x, const PrimeInfo& P) const {
        const uint64_t m = reduce64(x, P);
        return x > half ? submod(m, qlmod, P.p) : m;
    }
};

// Blocks are dealt to the 8 XCDs in turn (block i to XCD i mod 8).  Taking
// tile i in block i puts every 8th column tile of a limb on one XCD: a few of
// its L2 channels carry everything, and the second pass finds nothing of what
// the first one wrote.  So an XCD takes chunks of neighbouring tiles in turn:
// half a limb, or one eighth of the launch while the whole of it fits the L2s
// (up to 32 limbs of 512 KB; longer contiguous runs put the slower 64-bit limbs of
// a launch on one or two XCDs).  Forward transform at N = 2^16, 50-bit
// primes: 25 limbs 23.6 -> 17.0 us, 50 limbs 30.1 -> 28.9, 74 limbs 37.8 -> 37.6.
__device__ __forceinline__ uint32_t xcd_item(uint32_t chunk) {
    const uint32_t x = blockIdx.x & 7, i = blockIdx.x >> 3;
    return (i / chunk * 8 + x) * chunk + i % chunk;
}
struct XcdGrid {
    uint32_t chunk;
    dim3 grid;  // a whole number of rounds of chunks: items beyond the real ones return
};
inline XcdGrid xcd_chunks(size_t items, size_t c) {
    const size_t each = (items + 7) / 8;
    c = c < each ? c : each;
    c = c ? c : 1;
    return XcdGrid{(uint32_t)c, dim3((unsigned)((items + 8 * c - 1) / (8 * c) * (8 * c)))};
}
// items tiles, per of them to a limb
inline XcdGrid xcd_grid(size_t items, int per) {
    return xcd_chunks(items, items <= (size_t)32 * per ? items : (size_t)(per > 1 ? per / 2 : 1));
}
// Kernels with arithmetic of their own between the passes (the inner product,
// the tensor, small conversions): what is slow about a 64-bit limb, and the end of
// the launch, have to be spread over the XCDs more than the passes' tiles have
// to stay on one; 2 to 12 tiles take the same time.  At N = 2^16, against xcd_grid:
// inner product of 25 + 8 limbs 53.9 -> 50.0 us, of 6 + 8 19.6 -> 15.6, for 9 keys
// at 18 + 8 197 -> 165; tensor 26.1 -> 24.7; conversions 41.6 -> 40.3 and
// 30.8 -> 28.4.  The transforms are the other way round (25 limbs inverse: 21.3 -> 22.5).
constexpr int XCD_TILES = 8;

// The job and position of flattened limb a: a device list is walked through
// its limb map; an inline list has `most` limbs per job.  False: nothing to do.
struct NttGrid {
    int limbs;  // device list: flattened limbs; inline list: n most
    int most;
    uint32_t chunk;  // xcd_item
    dim3 grid;
};
__device__ __forceinline__ bool block_job(const NttJobs& L, const NttGrid& g, int a, NttJob& J, int& pos) {
    if (a >= g.limbs) return false;
    if (L.dev) {
        J = get_job(L, ((const __attribute__((address_space(1))) int*)L.limbmap)[a]);
        a -= J.first;
    } else {
        int j = 0;
        for (; a >= g.most; a -= g.most) ++j;
        J = get_inline(L, j);
        if (a >= J.npos - (J.skip_hi - J.skip_lo)) return false;
    }
    pos = a < J.skip_lo ? a : a + (J.skip_hi - J.skip_lo);
    return true;
}
// tpl blocks per limb
inline NttGrid ntt_grid(const NttJobs& L, int limbs, int tpl) {
    int most = limbs;
    if (!L.dev) {
        most = 1;
        for (int i = 0; i < L.n; ++i) {
            const int a = L.inl[i].npos - (L.inl[i].skip_hi - L.inl[i].skip_lo);
            most = a > most ? a : most;
        }
        limbs = L.n * most;
    }
    const XcdGrid x = xcd_grid((size_t)limbs * tpl, tpl);
    return NttGrid{limbs, most, x.chunk, x.grid};
}

}  // namespace fides
