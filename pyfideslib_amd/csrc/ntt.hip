// Negacyclic NTT / INTT for gfx950.
//
// Transform (OpenFHE ForwardTransformToBitReverseInPlace, FIDESlib
// src/NTT.cu:292-659): a_eval[j] = a(psi^(2 brev(j) + 1)) mod q, bit-reversed
// output; the inverse (src/NTT.cu:43-233) includes N^-1.
//
// Structure: N = N1 * N2 (N1 = 2^ceil(logN/2)).  The Cooley-Tukey stages that
// pair elements more than N2 apart act along "columns" (stride N2), the rest
// along contiguous "rows".  Forward = column pass then row pass; inverse
// (Gentleman-Sande) = row pass then column pass.  Each pass is one launch: a
// workgroup stages a tile of W columns or W rows in LDS (16 columns or 4
// rows; see rule_pick), each
// thread keeps 4 values in registers and runs two radix-2 stages on them
// between LDS exchanges.  Short per-wave instruction streams and many waves
// matter more than register blocking here: a pass is latency-bound (a tile's
// load -> phases -> store chain), not VALU-bound.  A ring
// of 2^14 would fit one block's LDS, but one CU alone needs 9 us for its
// butterflies (29 us measured, against 10 us for two launches over many CUs).
//
// Twiddles psi^brev(k) come from the bit-reversed tables: centered doubles for
// the primes below 2^50, whose butterflies run on the FP64 units, 64-bit words
// with their Shoup companions for the others (ntt_core.hpp).  Column-pass
// twiddles (the first N1 table entries, shared by all columns) are staged in
// LDS; row-pass twiddles (distinct per row) are prefetched into registers
// before the data load so their latency overlaps it.  Values
// stay lazily reduced between stages and are reduced once at the final store.
//
// Fusions (FIDESlib src/NTTfusions.cuh:218-262):
//   LOAD_SWITCH   (forward, pass 1): read the q_l coefficient limb and lift it
//                 centered into q_i (OpenFHE SwitchModulus) -- rescale.
//   STORE_MODDOWN (forward, pass 2): y = (acc - v) P^-1 (+ addend) -- ModDown.
//   STORE_MODDOWN_INV (forward, pass 2): STORE_MODDOWN, then the inverse's first
//                 pass on the row just stored -- the ModDown of what is switched
//                 next (25 limbs at N = 2^16: 12.4 + 10.9 us in two launches).
//   STORE_RESCALE (forward, pass 2): y = (x - v) q_l^-1 -- rescale.
//   STORE_MUL_RESCALE (forward, pass 2): y = (x w - v) q_l^-1 -- rescale of a
//                 product with a plaintext, which is not written out before.
//   STORE_MODDOWN_RESCALE (forward, pass 2): y = (acc P^-1 + add - v) q_l^-1 --
//                 ModDown and rescale merged (k_moddown_conv explains the form).
//   STORE_MODDOWN_AUTO (forward, pass 2): STORE_MODDOWN, then the automorphism
//                 X -> X^k (rotation: ModDown, add c0, automorphism -- the
//                 k_automorph gather, FIDESlib src/Rotation.cuh:14-36) as a
//                 scatter through LDS; every row of the output is one row of
//                 the input, permuted.
//   inverse pass 2 folds N^-1 (times an optional per-limb base-conversion
//   factor) into its last stage.
#include <cstdlib>

#include "ntt_core.hpp"

namespace fides {

// Column pass: CC columns of N1 rows per block, TC threads per column, 2^LRC
// values per thread (2, or 3 for radix-8 phases; logN = 17 only 3, as 16
// columns of 4-value threads would exceed 1024 threads).
template <int LOGN, int W, int LRC>
struct ColGeom {
    static constexpr int K1 = (LOGN + 1) / 2, K2 = LOGN / 2;
    static constexpr int N1 = 1 << K1, N2 = 1 << K2, N = 1 << LOGN;
    static constexpr int RC = 1 << LRC;
    static constexpr int TC = N1 / RC;
    static constexpr int CC = N2 < W ? N2 : W;
    static constexpr int NTC = TC * CC;
    static constexpr int SC = N1 + N1 / 16 + 1;
    static constexpr int TPL = N2 / CC;                  // tiles per limb
    static constexpr int NTW = (N1 + NTC - 1) / NTC;     // column twiddles a thread stages
};
template <int LOGN>
constexpr int min_lrc() { return ((1 << ((LOGN + 1) / 2)) / 4) * 16 > 1024 ? 3 : 2; }
template <int LOGN, int W>
using Rows = RowGeom<(LOGN + 1) / 2, LOGN / 2, 2, W>;

// The first N1 twiddles, shared by all columns: loaded with the tile, written
// to LDS after it (so neither waits for the other).
template <class G, class W>
__device__ __forceinline__ void stage_load(const W* tab, W* r) {
#pragma unroll
    for (int i = 0; i < G::NTW; ++i) r[i] = tab[(threadIdx.x + i * G::NTC) & (G::N1 - 1)];
}
template <class G, class W>
__device__ __forceinline__ void stage_put(W* twl, const W* r) {
#pragma unroll
    for (int i = 0; i < G::NTW; ++i) twl[(threadIdx.x + i * G::NTC) & (G::N1 - 1)] = r[i];
}

// Forward pass 1: column sub-transforms (global stages 0..K1-1).
template <int LOGN, int W, int LRC, int LOAD>
__global__ void __launch_bounds__((ColGeom<LOGN, W, LRC>::NTC)) k_ntt_fwd_cols(DevTables T, NttJobs L, NttGrid g) {
    using G = ColGeom<LOGN, W, LRC>;
    constexpr int R = G::RC, NB1 = first_nb<LRC, G::K1>(), LO1 = G::K1 - NB1, NBL = fwd_last_nb<LRC, G::K1>();
    __shared__ uint64_t lds[G::CC * G::SC];
    __shared__ ShoupConst twlds[G::N1];
    const uint32_t item = xcd_item(g.chunk);
    NttJob J;
    int pos;
    if (!block_job(L, g, item / G::TPL, J, pos)) return;
    const int pid = pos_pid(pos, J.nq, J.q0, T.L + 1);
    const int cc = threadIdx.x % G::CC, t = threadIdx.x / G::CC;
    const uint32_t col = (item % G::TPL) * G::CC + cc;
    uint64_t x[R];
    {
        const gu64* src = gp(J.src) + (LOAD == LOAD_SWITCH ? (size_t)0 : (size_t)pos * G::N);
#pragma unroll
        for (int j = 0; j < R; ++j) x[j] = src[col + elem<LRC, LO1, NB1>(t, j) * G::N2];
    }
    const PrimeInfo P = cld(T.primes + pid);
    with_arith(T, pid, P, [&](const auto& ar) {
        using A = std::decay_t<decltype(ar)>;
        using V = typename A::V;
        typename A::W tw[G::NTW];
        auto* twl = reinterpret_cast<typename A::W*>(twlds);
        stage_load<G>(A::fwd(T) + (size_t)pid * G::N, tw);
        V v[R];
        if constexpr (LOAD == LOAD_SWITCH) {
            const SwitchLift lift(T, J.level, pid);
#pragma unroll
            for (int j = 0; j < R; ++j) v[j] = ar.from(lift(x[j], P));
        } else {
#pragma unroll
            for (int j = 0; j < R; ++j) v[j] = ar.from(x[j]);
        }
        stage_put<G>(twl, tw);
        __syncthreads();
        auto twf = [&](int, int b, uint32_t e) { return twl[(1u << (G::K1 - 1 - b)) + (e >> (b + 1))]; };
        fwd_run<LRC, G::K1, G::K1, true>(ar, reinterpret_cast<V*>(lds) + cc * G::SC, v, t, twf);
        gu64* mid = gp(J.mid) + (size_t)pos * G::N;
#pragma unroll
        for (int j = 0; j < R; ++j) mid[col + elem<LRC, 0, NBL>(t, j) * G::N2] = A::pack(v[j]);
    });
}

// Forward pass 2: row sub-transforms (global stages K1..logN-1) + epilogue.
template <int LOGN, int W, int STORE>
__global__ void __launch_bounds__((Rows<LOGN, W>::NTR)) k_ntt_fwd_rows(DevTables T, NttJobs L, NttGrid g) {
    using G = Rows<LOGN, W>;
    __shared__ uint64_t lds[G::RR * G::SR];
    constexpr int TPL = G::N1 / G::RR;  // tiles per limb
    const uint32_t item = xcd_item(g.chunk);
    NttJob J;
    int pos;
    if (!block_job(L, g, item / TPL, J, pos)) return;
    const int pid = pos_pid(pos, J.nq, J.q0, T.L + 1);
    const int t = threadIdx.x % G::TR, rr = threadIdx.x / G::TR;
    const uint32_t r = (item % TPL) * G::RR + rr;
    const size_t limb = (size_t)pos * G::N;
    const uint32_t row = r * G::N2;
    uint64_t x[G::R];
    {
        const gu64* mid = gp(J.mid) + limb;
#pragma unroll
        for (int j = 0; j < G::R; ++j) x[j] = mid[row + elem<G::LR, G::LO1, G::NB1>(t, j)];
    }
    const PrimeInfo P = cld(T.primes + pid);
    uint64_t* sub = lds + rr * G::SR;
    with_arith(T, pid, P, [&](const auto& ar) {
        using A = std::decay_t<decltype(ar)>;
        using V = typename A::V;
        V v[G::R];
#pragma unroll
        for (int j = 0; j < G::R; ++j) v[j] = A::unpack(x[j]);
        Epilogue<G, STORE> epi;
        // the epilogue's operands are issued at the start of the phase before the last
        constexpr int EPI_HI = G::NBL + G::LR < G::K2 ? G::NBL + G::LR : G::K2;
        fwd_row<G, false>(ar, reinterpret_cast<V*>(sub), v, t, G::N1 + r, A::fwd(T) + (size_t)pid * G::N,
                          [&](auto hi) {
                              if constexpr (decltype(hi)::value == EPI_HI) epi.load(J, limb, row, t);
                          });
        epi.store(T, J, pos, pid, ar, sub, t, r, v);
    });
}

// Inverse pass 1: row sub-transforms (global stages on bits 0..K2-1).
template <int LOGN, int W>
__global__ void __launch_bounds__((Rows<LOGN, W>::NTR)) k_ntt_inv_rows(DevTables T, NttJobs L, NttGrid g) {
    using G = Rows<LOGN, W>;
    __shared__ uint64_t lds[G::RR * G::SR];
    constexpr int TPL = G::N1 / G::RR;  // tiles per limb
    const uint32_t item = xcd_item(g.chunk);
    NttJob J;
    int pos;
    if (!block_job(L, g, item / TPL, J, pos)) return;
    const int pid = pos_pid(pos, J.nq, J.q0, T.L + 1);
    const int t = threadIdx.x % G::TR, rr = threadIdx.x / G::TR;
    const uint32_t r = (item % TPL) * G::RR + rr;
    const size_t limb = (size_t)pos * G::N;
    const uint32_t row = r * G::N2;
    uint64_t x[G::R];
    {
        const gu64* src = gp(J.src) + limb;
#pragma unroll
        for (int j = 0; j < G::R; ++j) x[j] = src[row + G::mem(t, j)];
    }
    const PrimeInfo P = cld(T.primes + pid);
    with_arith(T, pid, P, [&](const auto& ar) {
        using A = std::decay_t<decltype(ar)>;
        using V = typename A::V;
        V v[G::R];
#pragma unroll
        for (int j = 0; j < G::R; ++j) v[j] = ar.from(x[j]);
        inv_row<G>(ar, reinterpret_cast<V*>(lds) + rr * G::SR, v, t, G::N1 + r,
                          A::inv(T) + (size_t)pid * G::N);
        gu64* mid = gp(J.mid) + limb;
#pragma unroll
        for (int j = 0; j < G::R; ++j) mid[row + elem<G::LR, G::LOL, G::NBI>(t, j)] = A::pack(v[j]);
    });
}

// Inverse pass 2: column sub-transforms, last stage scaled by N^-1 (x factor).
template <int LOGN, int W, int LRC>
__global__ void __launch_bounds__((ColGeom<LOGN, W, LRC>::NTC)) k_ntt_inv_cols(DevTables T, NttJobs L, NttGrid g) {
    using G = ColGeom<LOGN, W, LRC>;
    constexpr int R = G::RC, NB1 = first_nb<LRC, G::K1>(), LOL = inv_last_lo<LRC, G::K1>(), NBL = G::K1 - LOL;
    __shared__ uint64_t lds[G::CC * G::SC];
    __shared__ ShoupConst twlds[G::N1];
    const uint32_t item = xcd_item(g.chunk);
    NttJob J;
    int pos;
    if (!block_job(L, g, item / G::TPL, J, pos)) return;
    const int pid = pos_pid(pos, J.nq, J.q0, T.L + 1);
    const int cc = threadIdx.x % G::CC, t = threadIdx.x / G::CC;
    const uint32_t col = (item % G::TPL) * G::CC + cc;
    uint64_t x[R];
    {
        const gu64* mid = gp(J.mid) + (size_t)pos * G::N;
#pragma unroll
        for (int j = 0; j < R; ++j) x[j] = mid[col + elem<LRC, 0, NB1>(t, j) * G::N2];
    }
    const PrimeInfo P = cld(T.primes + pid);
    const ShoupConst* sc = inv_scale(T, J, pos, pid);
    const ShoupConst s = cld(sc), ws = cld(sc + 1);
    with_arith(T, pid, P, [&](const auto& ar) {
        using A = std::decay_t<decltype(ar)>;
        using V = typename A::V;
        typename A::W tw[G::NTW];
        auto* twl = reinterpret_cast<typename A::W*>(twlds);
        stage_load<G>(A::inv(T) + (size_t)pid * G::N, tw);
        V v[R];
#pragma unroll
        for (int j = 0; j < R; ++j) v[j] = A::unpack(x[j]);
        stage_put<G>(twl, tw);
        __syncthreads();
        auto twf = [&](int, int b, uint32_t e) { return twl[(1u << (G::K1 - 1 - b)) + (e >> (b + 1))]; };
        inv_run<LRC, G::K1, 0, true>(ar, reinterpret_cast<V*>(lds) + cc * G::SC, v, t, twf, s, ws);
        gu64* dst = gp(J.dst) + (size_t)pos * G::N;
#pragma unroll
        for (int j = 0; j < R; ++j) dst[col + elem<LRC, LOL, NBL>(t, j) * G::N2] = ar.canon_inv(v[j]);
    });
}

// Centered FP64 twiddles of the primes that use them.
__global__ void k_fp_twiddles(DevTables T, const ShoupConst* tw, double* out) {
    const PrimeInfo P = cld(T.primes + blockIdx.y);
    if (!P.fp) return;
    const size_t i = (size_t)blockIdx.y * T.N + blockIdx.x * blockDim.x + threadIdx.x;
    const uint64_t w = tw[i].w;
    out[i] = w > (P.p >> 1) ? fp_from(w) - P.pd : fp_from(w);
}

// ---------------------------------------------------------- launchers ----

// Launch configuration of a transform: column tile width, log2 values per
// column thread, row tile height (the fourth entry of a tuning configuration is
// read and has no effect).
struct NttPick {
    int cc, lrc, rr;
};
// Fixed rules: column tiles are 16 wide (128-byte row segments) except for
// launches of under 64 tiles, row tiles 4 rows (256 threads), 8 values per column
// thread (radix-8 phases, one LDS exchange fewer) from 40 limbs up.  They were
// measured at N = 2^16 with integer butterflies in every limb.  With the present ones
// they hold at 1, 2 and 25 limbs, and tiles of 4 or 8 columns are ahead elsewhere: forward
// (inverse) at 4 limbs 12.8 -> 11.4 us (13.3 -> 11.5), at 8 13.5 -> 12.0 (13.5 -> 12.1), at 74
// 44.1 -> 41.3 (45.2 -> 42.9).  The table holds that for N = 2^16 and 2^13; the other rings
// have not been measured again and keep the rules.
// FIDES_NTT_COLS / FIDES_NTT_ROWS (4, 8 or 16) and FIDES_NTT_LRC (2 or 3)
// force a value.
static int env_int(const char* name) {
    const char* e = std::getenv(name);
    return e ? std::atoi(e) : -1;
}
static NttPick rule_pick(int logN, int limbs) {
    static const int ov_c = env_int("FIDES_NTT_COLS"), ov_r = env_int("FIDES_NTT_ROWS");
    static const int ov_l = env_int("FIDES_NTT_LRC");
    auto width = [](int w) { return w == 4 || w == 8 ? w : 16; };
    const int n2 = 1 << (logN / 2);
    const int tiles16 = limbs * (n2 < 16 ? 1 : n2 / 16);
    NttPick p;
    p.cc = ov_c > 0 ? width(ov_c) : (tiles16 < 64 ? 4 : 16);
    p.rr = ov_r > 0 ? width(ov_r) : 4;
    p.lrc = ov_l > 0 ? (ov_l == 3 ? 3 : 2) : (limbs >= 40 ? 3 : 2);
    return p;
}

// The measured table's entry for this launch (pyfideslib_amd/tune.py), else
// the fixed rules.
static NttPick ntt_pick(bool forward, int logN, int limbs) {
    TuneCfg c;
    if (tune_get(forward ? TUNE_NTT_FWD : TUNE_NTT_INV, logN, limbs, c)) return NttPick{c.v[0], c.v[1], c.v[2]};
    return rule_pick(logN, limbs);
}

TuneCfg ntt_rule_cfg(bool, int logN, int limbs) {
    const NttPick p = rule_pick(logN, limbs);
    return TuneCfg{{p.cc, p.lrc, p.rr, 0}};
}

template <int LOGN, int W, int LRC>
static void fwd_cols(const DevTables& T, const NttJobs& L, int limbs, int load, hipStream_t s) {
    using G = ColGeom<LOGN, W, LRC>;
    const NttGrid n = ntt_grid(L, limbs, G::TPL);
    const dim3 g = n.grid;
    if (load == LOAD_SWITCH)
        hipLaunchKernelGGL((k_ntt_fwd_cols<LOGN, W, LRC, LOAD_SWITCH>), g, dim3(G::NTC), 0, s, T, L, n);
    else
        hipLaunchKernelGGL((k_ntt_fwd_cols<LOGN, W, LRC, LOAD_PLAIN>), g, dim3(G::NTC), 0, s, T, L, n);
}

template <int LOGN, int W, int LRC>
static void inv_cols(const DevTables& T, const NttJobs& L, int limbs, hipStream_t s) {
    using G = ColGeom<LOGN, W, LRC>;
    const NttGrid n = ntt_grid(L, limbs, G::TPL);
    hipLaunchKernelGGL((k_ntt_inv_cols<LOGN, W, LRC>), n.grid, dim3(G::NTC), 0, s, T, L, n);
}

template <int LOGN, int W>
static void fwd_rows(const DevTables& T, const NttJobs& L, int limbs, int store, hipStream_t s) {
    using G = Rows<LOGN, W>;
    const NttGrid n = ntt_grid(L, limbs, G::N1 / G::RR);
    const dim3 g = n.grid, b(G::NTR);
    if (store == STORE_MODDOWN)
        hipLaunchKernelGGL((k_ntt_fwd_rows<LOGN, W, STORE_MODDOWN>), g, b, 0, s, T, L, n);
    else if (store == STORE_MODDOWN_INV)
        hipLaunchKernelGGL((k_ntt_fwd_rows<LOGN, W, STORE_MODDOWN_INV>), g, b, 0, s, T, L, n);
    else if (store == STORE_MODDOWN_AUTO)
        hipLaunchKernelGGL((k_ntt_fwd_rows<LOGN, W, STORE_MODDOWN_AUTO>), g, b, 0, s, T, L, n);
    else if (store == STORE_MODDOWN_RESCALE)
        hipLaunchKernelGGL((k_ntt_fwd_rows<LOGN, W, STORE_MODDOWN_RESCALE>), g, b, 0, s, T, L, n);
    else if (store == STORE_MUL_RESCALE)
        hipLaunchKernelGGL((k_ntt_fwd_rows<LOGN, W, STORE_MUL_RESCALE>), g, b, 0, s, T, L, n);
    else if (store == STORE_RESCALE)
        hipLaunchKernelGGL((k_ntt_fwd_rows<LOGN, W, STORE_RESCALE>), g, b, 0, s, T, L, n);
    else
        hipLaunchKernelGGL((k_ntt_fwd_rows<LOGN, W, STORE_PLAIN>), g, b, 0, s, T, L, n);
}

template <int LOGN, int W>
static void inv_rows(const DevTables& T, const NttJobs& L, int limbs, hipStream_t s) {
    using G = Rows<LOGN, W>;
    const NttGrid n = ntt_grid(L, limbs, G::N1 / G::RR);
    hipLaunchKernelGGL((k_ntt_inv_rows<LOGN, W>), n.grid, dim3(G::NTR), 0, s, T, L, n);
}

template <class F>
static void by_width(int w, F&& f) {
    if (w == 4)
        f(std::integral_constant<int, 4>{});
    else if (w == 8)
        f(std::integral_constant<int, 8>{});
    else
        f(std::integral_constant<int, 16>{});
}

// Column-pass dispatch over (tile width, values per thread).
template <int LOGN, bool FWD>
static void cols_dispatch(const DevTables& T, const NttJobs& L, int limbs, int load, const NttPick& pk,
                          hipStream_t s) {
    by_width(pk.cc, [&](auto wv) {
        constexpr int WW = decltype(wv)::value;
        auto go = [&](auto lv) {
            constexpr int LL = decltype(lv)::value;
            if constexpr (FWD)
                fwd_cols<LOGN, WW, LL>(T, L, limbs, load, s);
            else
                inv_cols<LOGN, WW, LL>(T, L, limbs, s);
        };
        if (pk.lrc == 3)
            go(std::integral_constant<int, 3>{});
        else
            go(std::integral_constant<int, min_lrc<LOGN>()>{});
    });
}

template <int LOGN>
static hipError_t fwd_impl(const DevTables& T, const NttJobs& L, int limbs, int load, int store, hipStream_t s,
                           int passes) {
    const NttPick pk = ntt_pick(true, LOGN, limbs);
    if (passes & NTT_PASS1) cols_dispatch<LOGN, true>(T, L, limbs, load, pk, s);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || !(passes & NTT_PASS2)) return e;
    by_width(pk.rr, [&](auto wr) { fwd_rows<LOGN, decltype(wr)::value>(T, L, limbs, store, s); });
    return hipGetLastError();
}

template <int LOGN>
static hipError_t inv_impl(const DevTables& T, const NttJobs& L, int limbs, hipStream_t s, int passes) {
    const NttPick pk = ntt_pick(false, LOGN, limbs);
    if (passes & NTT_PASS1)
        by_width(pk.rr, [&](auto wr) { inv_rows<LOGN, decltype(wr)::value>(T, L, limbs, s); });
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || !(passes & NTT_PASS2)) return e;
    cols_dispatch<LOGN, false>(T, L, limbs, 0, pk, s);
    return hipGetLastError();
}

hipError_t launch_fp_twiddles(const DevTables& T, const ShoupConst* tw, double* out, hipStream_t s) {
    hipLaunchKernelGGL(k_fp_twiddles, dim3(T.N / 256, T.np), dim3(256), 0, s, T, tw, out);  // N >= 2^10
    return hipGetLastError();
}

hipError_t launch_ntt_fwd(const DevTables& T, const NttJobs& L, int limbs, int load, int store, hipStream_t s,
                          int passes) {
    if (limbs <= 0) return hipSuccess;
    switch (T.logN) {
        case 10: return fwd_impl<10>(T, L, limbs, load, store, s, passes);
        case 11: return fwd_impl<11>(T, L, limbs, load, store, s, passes);
        case 12: return fwd_impl<12>(T, L, limbs, load, store, s, passes);
        case 13: return fwd_impl<13>(T, L, limbs, load, store, s, passes);
        case 14: return fwd_impl<14>(T, L, limbs, load, store, s, passes);
        case 15: return fwd_impl<15>(T, L, limbs, load, store, s, passes);
        case 16: return fwd_impl<16>(T, L, limbs, load, store, s, passes);
        case 17: return fwd_impl<17>(T, L, limbs, load, store, s, passes);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_ntt_inv(const DevTables& T, const NttJobs& L, int limbs, hipStream_t s, int passes) {
    if (limbs <= 0) return hipSuccess;
    switch (T.logN) {
        case 10: return inv_impl<10>(T, L, limbs, s, passes);
        case 11: return inv_impl<11>(T, L, limbs, s, passes);
        case 12: return inv_impl<12>(T, L, limbs, s, passes);
        case 13: return inv_impl<13>(T, L, limbs, s, passes);
        case 14: return inv_impl<14>(T, L, limbs, s, passes);
        case 15: return inv_impl<15>(T, L, limbs, s, passes);
        case 16: return inv_impl<16>(T, L, limbs, s, passes);
        case 17: return inv_impl<17>(T, L, limbs, s, passes);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace fides
