// Geometry and grids of the fused key-switch kernels (fused.hip, fused_down.hip).
#pragma once
#include "conv.hpp"
#include "ntt_core.hpp"

namespace fides {

constexpr int FUSED_LOGN_MIN = 12, FUSED_LOGN_MAX = 16;
// Source limbs of a conversion (11 as 12, conv_bound), where their sums fit one
// reduction (fused_ok): with 60-bit special primes that holds up to 8, with shorter ones
// up to 12.  At 12 the ModDown with a rescale spills 38 registers and is still ahead of
// the separate kernels: 20 limbs and 11 special primes of 59 bits, separate -> fused, N = 2^16
// a product 182 -> 182 us, a rotation 155 -> 150, at half the limbs 114 -> 111 and 97 -> 94;
// N = 2^15 116 -> 110, 99 -> 92, 83 -> 78, 72 -> 66.  Past it sources would not fit.
// At N = 2^14 a ModDown from more than 9 primes repeats their column pass (conv_inv) at a
// cost that hoisted sets and large batches do not win back: 10 primes, 5 rotations 127 -> 138 us;
// 11, 32 products 896 -> 974.
constexpr int FUSED_CONV_MAX = 12;
constexpr int fused_down_max(int logN) { return logN == 14 ? 9 : FUSED_CONV_MAX; }
constexpr int FUSED_DIGITS = 4;
constexpr int CONV_INV_LOGN = 14;

// Rows of the second pass: as many per block as fill one wave or four.
template <int LOGN>
using FRows = RowGeom<(LOGN + 1) / 2, LOGN / 2, 2, (LOGN >= 15 ? 256 : 64) / ((1 << (LOGN / 2)) / 4)>;

template <class F>
static hipError_t by_logn(int logN, F&& f) {
    switch (logN) {
        case 12: f(std::integral_constant<int, 12>{}); break;
        case 13: f(std::integral_constant<int, 13>{}); break;
        case 14: f(std::integral_constant<int, 14>{}); break;
        case 15: f(std::integral_constant<int, 15>{}); break;
        case 16: f(std::integral_constant<int, 16>{}); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// Unsigned division by a launch constant d of values up to most: one multiply
// where it is exact (most d < 2^32), else the division itself.
struct FastDiv {
    uint32_t d, m;
    FastDiv(size_t d_, size_t most)
        : d((uint32_t)d_), m(most * d_ < 0x100000000ull && d_ > 1 ? (uint32_t)(0x100000000ull / d_ + 1) : 0u) {}
    __device__ __forceinline__ uint32_t div(uint32_t n) const { return m ? __umulhi(n, m) : d == 1 ? n : n / d; }
};

// Tiles of the conversion kernels: 4 columns of N1 rows, 512 threads, TB
// target limbs at a time (2048 outputs, 4 a thread).  The conversion and the
// column pass use different thread layouts and meet in LDS:
//   convert  a thread holds its CPT coefficients of every source limb in
//            registers (30-bit halves, 2 A CPT of them) and computes 4 sums, CPT
//            coefficients of TPT targets each;
//   columns  a wave runs whole columns of one target (4 values per thread), so
//            its LDS exchanges need no block barrier and the waves of 64-bit
//            and FP64 limbs go their own ways;
//   store    4 neighbouring columns a row.
// Two barriers per TB targets, LDS double-buffered.  Holding 4 coefficients per
// thread and running the column pass in the same layout took 176 registers (2
// waves per SIMD) and measured 51.8 us against the 45.6 us of separate kernels.
template <int LOGN>
struct ConvCols {
    static constexpr int K1 = (LOGN + 1) / 2, K2 = LOGN / 2;
    static constexpr int N1 = 1 << K1, N2 = 1 << K2, N = 1 << LOGN;
    static constexpr int NT = 512, CC = 4, COEF = CC * N1;
    static constexpr int TPC = N1 / 4;                   // threads per column
    static constexpr int TB = 2048 / COEF;               // targets at a time
    static constexpr int CPT = COEF > NT ? COEF / NT : 1;  // coefficients and
    static constexpr int TPT = 4 / CPT;                  // targets of a thread's sums
    static constexpr int SC = N1 + N1 / 16 + 1;
    static constexpr int TPL = N2 / CC;
    static constexpr int LO1 = K1 - 2, NBL = fwd_last_nb<2, K1>();
    static_assert(COEF * TB == 4 * NT && TB * N1 == NT && CPT <= 2, "four sums and one twiddle per thread");
    // the coefficients of thread tid: row, first column (CPT neighbouring columns), first target
    static __device__ __forceinline__ uint32_t c_row(uint32_t tid) { return (tid * CPT / CC) % N1; }
    static __device__ __forceinline__ uint32_t c_col(uint32_t tid) { return tid * CPT % CC; }
    static __device__ __forceinline__ uint32_t c_tgt(uint32_t tid) { return tid * CPT / COEF * TPT; }
    // column pass: target (wave-uniform), column and thread within the column
    static __device__ __forceinline__ uint32_t n_tgt(uint32_t tid) { return tid / (CC * TPC); }
    static __device__ __forceinline__ uint32_t n_col(uint32_t tid) { return tid / TPC % CC; }
    static __device__ __forceinline__ uint32_t n_t(uint32_t tid) { return tid % TPC; }
};
// Rings up to 2^CONV_INV_LOGN are bound by launches: there the conversion
// kernels also run the column pass of their sources' inverse transform (once
// per target group, which costs arithmetic that the idle CUs have to spare).
template <int LOGN>
constexpr bool conv_inv() { return LOGN <= CONV_INV_LOGN; }
template <int LOGN, int SOURCES, bool INV = conv_inv<LOGN>()>
struct ConvLds {
    using G = ConvCols<LOGN>;
    struct Targets {
        uint64_t tile[2][G::TB][G::CC][G::SC];
        ShoupConst tw[2][G::TB][G::N1];
    };
    struct Sources {
        uint64_t tile[SOURCES][G::CC][G::SC];
        ShoupConst tw[SOURCES][G::N1];
    };
    struct None {};
    union {
        Targets t;
        std::conditional_t<INV, Sources, None> s;  // before the first target
    };
};

// The column pass of the inverse transform of n source limbs (limb(i): what the
// row pass left, pid(i), scale(i): the limb's last-stage pair) on the block's
// columns; coefficient (row, column) of limb i ends at S.s.tile[i][column][row].
template <int LOGN, int SOURCES, bool INV, class LIMB, class PID, class SCALE>
__device__ __forceinline__ void conv_sources(const DevTables& T, ConvLds<LOGN, SOURCES, INV>& S, int n, uint32_t col0,
                                             const LIMB& limb, const PID& pid_of, const SCALE& scale) {
    using G = ConvCols<LOGN>;
    constexpr int LOL = inv_last_lo<2, G::K1>(), NBI = G::K1 - LOL, PAIRS = G::COEF / 2;
    for (int w = threadIdx.x; w < n * PAIRS; w += G::NT) {
        const int i = __builtin_amdgcn_readfirstlane(w / PAIRS);  // PAIRS is a multiple of the wave
        const uint32_t e = (w % PAIRS) * 2, row = e / G::CC, cc = e % G::CC;
        const u64x2 v = ld2(limb(i) + row * G::N2 + col0 + cc);
        S.s.tile[i][cc][lds_off(row)] = v.x;
        S.s.tile[i][cc + 1][lds_off(row)] = v.y;
    }
    for (int w = threadIdx.x; w < n * G::N1; w += G::NT) {
        const int i = __builtin_amdgcn_readfirstlane(w / G::N1), r = w % G::N1;
        const size_t at = (size_t)pid_of(i) * G::N + r;
        if (is_fp(T, pid_of(i)))
            reinterpret_cast<double*>(S.s.tw[i])[r] = T.twd_inv[at];
        else
            S.s.tw[i][r] = T.tw_inv[at];
    }
    __syncthreads();
    const uint32_t t = G::n_t(threadIdx.x);
    for (int ci = threadIdx.x / G::TPC; ci < n * G::CC; ci += G::NT / G::TPC) {
        const int i = __builtin_amdgcn_readfirstlane(ci / G::CC);  // a wave's columns are of one limb
        const uint32_t cc = ci % G::CC;
        const int pid = pid_of(i);
        const PrimeInfo P = cld(T.primes + pid);
        const ShoupConst* sc = scale(i);
        const ShoupConst s = cld(sc), ws = cld(sc + 1);
        with_arith(T, pid, P, [&](const auto& ar) {
            using A = std::decay_t<decltype(ar)>;
            using V = typename A::V;
            const auto* twl = reinterpret_cast<const typename A::W*>(S.s.tw[i]);
            V* sub = reinterpret_cast<V*>(S.s.tile[i][cc]);
            V v[4];
            lds_get<2, 0, first_nb<2, G::K1>()>(sub, t, v);  // the words as the row pass packed them
            auto twf = [&](int, int b, uint32_t e) { return twl[(1u << (G::K1 - 1 - b)) + (e >> (b + 1))]; };
            inv_run<2, G::K1, 0, true, true>(ar, sub, v, t, twf, s, ws);
#pragma unroll
            for (int j = 0; j < 4; ++j) S.s.tile[i][cc][lds_off(elem<2, LOL, NBI>(t, j))] = ar.canon_inv(v[j]);
        });
    }
    __syncthreads();
}

// The column pass of a wave's target (prime pid) on the buffer's tile.
template <int LOGN, int SOURCES, bool INV>
__device__ __forceinline__ void conv_columns(const DevTables& T, int pid, ConvLds<LOGN, SOURCES, INV>& S, int buf, int i) {
    using G = ConvCols<LOGN>;
    const uint32_t t = G::n_t(threadIdx.x), cc = G::n_col(threadIdx.x);
    const PrimeInfo P = cld(T.primes + pid);
    with_arith(T, pid, P, [&](const auto& ar) {
        using A = std::decay_t<decltype(ar)>;
        using V = typename A::V;
        const auto* twl = reinterpret_cast<const typename A::W*>(S.t.tw[buf][i]);
        V* sub = reinterpret_cast<V*>(S.t.tile[buf][i][cc]);
        V v[4];
        lds_get<2, G::LO1, 2>(sub, t, v);
        auto twf = [&](int, int b, uint32_t e) { return twl[(1u << (G::K1 - 1 - b)) + (e >> (b + 1))]; };
        fwd_run<2, G::K1, G::K1, false, true>(ar, sub, v, t, twf);
        lds_put<2, 0, G::NBL>(sub, t, v);
    });
}
// One twiddle of a target (row r of its table) per thread: read ahead of the
// conversion, put in LDS after it.
struct ConvTw {
    bool fp;
    ShoupConst w;
    __device__ __forceinline__ void load(const DevTables& T, int pid, int r) {
        fp = is_fp(T, pid);
        if (fp)
            w.w = (uint64_t)__double_as_longlong(T.twd_fwd[(size_t)pid * T.N + r]);
        else
            w = T.tw_fwd[(size_t)pid * T.N + r];
    }
    template <int LOGN, int SOURCES, bool INV>
    __device__ __forceinline__ void put(ConvLds<LOGN, SOURCES, INV>& S, int buf, int i, int r) const {
        if (fp)
            reinterpret_cast<uint64_t*>(S.t.tw[buf][i])[r] = w.w;
        else
            S.t.tw[buf][i][r] = w;
    }
};
// The tile's rows to limb `out`: 2048 words of TB targets, 4 a thread.
template <int LOGN, int SOURCES, bool INV, class F>
__device__ __forceinline__ void conv_store(const ConvLds<LOGN, SOURCES, INV>& S, int buf, uint32_t col0, const F& limb) {
    using G = ConvCols<LOGN>;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const uint32_t w = (threadIdx.x + q * G::NT) * 2;
        const uint32_t i = w / G::COEF, row = w / G::CC % G::N1, cc = w % G::CC;
        uint64_t* o = limb((int)i);
        if (o) st2(o + row * G::N2 + col0 + cc, S.t.tile[buf][i][cc][lds_off(row)],
                   S.t.tile[buf][i][cc + 1][lds_off(row)]);
    }
}

// Grid of a conversion kernel: items (job, [digit,] target group, tile).
struct ConvGrid {
    uint32_t items, chunk;
    FastDiv tg, nd;
};
// Past 32 limbs of tiles half a limb to an XCD (24 products at 25 limbs: 410 us for the
// ModUp against 438 with XCD_TILES).
inline XcdGrid conv_grid(size_t items, int per) {
    return items <= (size_t)32 * per ? xcd_chunks(items, XCD_TILES) : xcd_grid(items, per);
}
// Blocks of a conversion's launch.  Where each group runs the sources' column
// pass again, groups past one round of what is resident cost more than they
// give: two blocks a CU, one where the sources' tiles take more than half of its
// LDS.  Against 1024 blocks, N = 2^13, 59-bit limbs (separate kernels in brackets): 10 special
// primes, 5 hoisted rotations 96 -> 87 us (87), 8 products 162 -> 143 (156); 11 special primes
// 105 -> 93 (90) and 192 -> 156 (167).
constexpr size_t conv_most_blocks(int logN, int sources) {
    const size_t n1 = (size_t)1 << ((logN + 1) / 2), bytes = sources * (4 * (n1 + n1 / 16 + 1) * 8 + n1 * 16);
    return logN > CONV_INV_LOGN ? 1024 : bytes > (80 << 10) ? 256 : 512;
}
// Target groups, of whole rounds of tb targets: up to 1024 blocks in all, two
// rounds of what is resident (ModUp at N = 2^16, level 24: 40.3 us with 768 blocks, 45 with
// 384, 47 with 1536; ModDown 28.4 with 768, 27.5 with 512, 33 with 256 or 1024).
// Where whole rounds leave less than half of the CUs with a block, single targets up
// to 192 blocks: a thread then forms one sum instead of TPT in turn (N = 2^13, 4
// limbs: ModDown 9.2 -> 8.2 us, ModUp 8.2 -> 7.4; at 128 blocks, N = 2^14, no gain).
inline int fused_groups(size_t base_blocks, int targets, int tb, size_t most = 1024) {
    const int rounds = (targets + tb - 1) / tb;
    if (base_blocks && base_blocks * rounds < 128) {
        const int g = (int)(192 / base_blocks);
        return g < 1 ? 1 : g < targets ? g : targets;
    }
    size_t g = most / (base_blocks ? base_blocks : 1);
    if (g < 1) g = 1;
    if (g > (size_t)rounds) g = rounds;
    const size_t each = (rounds + g - 1) / g;  // rounds per group, evened out
    return (int)((rounds + each - 1) / each);
}

// The groups of a launch of `convs` conversions.
inline int conv_launch_groups(int kind, int logN, int convs, size_t base_blocks, int targets, int tb, int sources) {
    const int tg = conv_set_tg(kind, logN, convs, targets);
    return tg ? tg : fused_groups(base_blocks, targets, tb, conv_most_blocks(logN, sources));
}

// The exact sum over the A sources of x_i m_i (m: one matrix row, scalar
// loads), before its reduction.
template <int A>
__device__ __forceinline__ void conv_acc(const Half2* x, const MatRow<A>& row, uint64_t& lo, uint64_t& hi) {
    Acc4 acc;
#pragma unroll
    for (int i = 0; i < A; ++i) mac_split(acc, x[i], split30(row.v[i]));
    combine(acc, lo, hi);
}

// The conversion sums of CPT coefficients at a (wave-uniform) target prime, in
// its arithmetic, to tile[c][at]; mat, fp: the matrices' rows of all primes.
// These kernels are bound by instruction issue: with conv_fp in place of four
// unsigned sums, a 128-bit reduction and the way to a double, 85 -> 48 vector
// instructions an output, and at N = 2^16 with 25 limbs and 50-bit primes the ModDown
// took 37 -> 30.8 us and the ModUp 44 -> 41.6.
template <int A, int CPT, int SC>
__device__ __forceinline__ void conv_tile(const DevTables& T, int pid, const PrimeInfo& P, const Half2 (&x)[CPT][A],
                                          const uint64_t* mat, const ConvFp* fp, uint64_t (*tile)[SC], uint32_t at) {
    if (is_fp(T, pid)) {
        const MatRowFp<A> row = cld(reinterpret_cast<const MatRowFp<A>*>(fp + (size_t)pid * A));
#pragma unroll
        for (int c = 0; c < CPT; ++c) tile[c][at] = FpArith::pack(conv_fp<A>(x[c], row, P));
    } else {
        const MatRow<A> row = cld(reinterpret_cast<const MatRow<A>*>(mat + (size_t)pid * A));
        const IntArith ar(P);
#pragma unroll
        for (int c = 0; c < CPT; ++c) {
            uint64_t lo, hi;
            conv_acc<A>(x[c], row, lo, hi);
            tile[c][at] = ar.from_lazy(reduce128_lazy(lo, hi, P));
        }
    }
}

}  // namespace fides
