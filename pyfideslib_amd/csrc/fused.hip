// The key switch's ModUp half in three launches where the plain form takes
// six: the conversion and the column pass of its outputs' transform in one
// kernel, their row pass and the inner product with the key in another (which
// also begins the inverse transforms of what ModDown brings down), and the
// tensor product with the row pass of its third part's inverse transform.
//
// At N = 2^16 a pass over the 25 to 74 limbs of a key switch is bound by memory
// and by the latency of a launch's chain, the conversions apart, which are bound by
// instruction issue: what is fused away is the write and read of every limb in between.
#include "fused.hpp"

namespace fides {

// ------------------------------------------------ tensor + inverse rows ----
struct RowsGrid {
    uint32_t items, chunk;
    FastDiv npos;
};

template <int LOGN>
__global__ void __launch_bounds__(FRows<LOGN>::NTR) k_tensor_rows(DevTables T, TensorJobs L, RowsGrid g) {
    using G = FRows<LOGN>;
    constexpr int TPL = G::N1 / G::RR;
    __shared__ uint64_t lds[G::RR * G::SR];
    const uint32_t item = xcd_item(g.chunk);
    if (item >= g.items) return;
    const uint32_t lim = item / TPL, z = g.npos.div(lim);
    const int i = (int)(lim - z * g.npos.d);
    const TensorJob J = L.dev ? get_job(L, (int)z) : get_inline(L, (int)z);
    if (i >= J.nl) return;
    const int t = threadIdx.x % G::TR, rr = threadIdx.x / G::TR;
    const uint32_t r = (item % TPL) * G::RR + rr;
    const size_t limb = (size_t)i * G::N;
    const uint32_t x = r * G::N2 + G::mem(t, 0);  // 4 neighbouring words
    const u64x2 a0 = ld2(J.c0 + limb + x), a0h = ld2(J.c0 + limb + x + 2);
    const u64x2 a1 = ld2(J.c1 + limb + x), a1h = ld2(J.c1 + limb + x + 2);
    const u64x2 b0 = ld2(J.d0 + limb + x), b0h = ld2(J.d0 + limb + x + 2);
    const u64x2 b1 = ld2(J.d1 + limb + x), b1h = ld2(J.d1 + limb + x + 2);
    const PrimeInfo P = cld(T.primes + i);
    with_arith(T, i, P, [&](const auto& ar) {
        using A = std::decay_t<decltype(ar)>;
        using V = typename A::V;
        const uint64_t p0[4] = {a0.x, a0.y, a0h.x, a0h.y}, p1[4] = {a1.x, a1.y, a1h.x, a1h.y};
        const uint64_t q0[4] = {b0.x, b0.y, b0h.x, b0h.y}, q1[4] = {b1.x, b1.y, b1h.x, b1h.y};
        uint64_t o0[4], o1[4], o2[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            o0[j] = ar.mul(p0[j], q0[j], P);
            o1[j] = ar.mul2(p0[j], q1[j], p1[j], q0[j], P);
            o2[j] = ar.mul(p1[j], q1[j], P);
        }
        st2(J.o0 + limb + x, o0[0], o0[1]);
        st2(J.o0 + limb + x + 2, o0[2], o0[3]);
        st2(J.o1 + limb + x, o1[0], o1[1]);
        st2(J.o1 + limb + x + 2, o1[2], o1[3]);
        st2(J.o2 + limb + x, o2[0], o2[1]);
        st2(J.o2 + limb + x + 2, o2[2], o2[3]);
        V v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = ar.from(o2[j]);
        inv_row<G>(ar, reinterpret_cast<V*>(lds) + rr * G::SR, v, t, G::N1 + r, A::inv(T) + (size_t)i * G::N);
        gu64* mid = gp(J.t) + limb;
#pragma unroll
        for (int j = 0; j < 4; ++j) mid[r * G::N2 + elem<2, G::LOL, G::NBI>(t, j)] = A::pack(v[j]);
    });
}

// --------------------------------------------- ModUp conversion + columns ----
template <int LOGN, int A>
__global__ void __launch_bounds__(512, 4) k_modup_cols(DevTables T, ModUpJobs L, ConvGrid g) {
    using G = ConvCols<LOGN>;
    __shared__ ConvLds<LOGN, A> S;
    const uint32_t item = xcd_item(g.chunk);
    if (item >= g.items) return;
    const uint32_t u = item / G::TPL, u2 = g.tg.div(u), z = g.nd.div(u2);
    const int tg = (int)(u - u2 * g.tg.d), d = (int)(u2 - z * g.nd.d);
    const ModUpJob J = L.dev ? get_job(L, (int)z) : get_inline(L, (int)z);
    const int nl = __builtin_amdgcn_readfirstlane(J.level) + 1;
    if (d >= num_digits(T, nl)) return;
    const int start = d * T.alpha;
    const int size = (nl - start) < T.alpha ? (nl - start) : T.alpha;
    const int ntarget = nl - size + T.K;
    // targets tg, tg + TG, ..: the 64-bit ones come last and are dealt out evenly
    const int TG = (int)g.tg.d, k1 = (ntarget - tg + TG - 1) / TG;
    if (k1 <= 0) return;
    const uint32_t tid = threadIdx.x;
    const uint32_t col0 = (item % G::TPL) * G::CC;
    const uint32_t c_at = G::c_row(tid) * G::N2 + col0 + G::c_col(tid);
    const int c_tgt = __builtin_amdgcn_readfirstlane(G::c_tgt(tid));
    const int n_tgt = __builtin_amdgcn_readfirstlane(G::n_tgt(tid));
    // the digit's limbs; rows beyond its size are zero
    Half2 x[G::CPT][A];
    if constexpr (conv_inv<LOGN>()) {
        conv_sources(
            T, S, size, col0, [&](int i) { return J.t + (size_t)(start + i) * G::N; },
            [&](int i) { return start + i; },
            [&](int i) { return T.iscale_modup + ((size_t)(nl - 1) * (T.L + 1) + start + i) * 2; });
#pragma unroll
        for (int i = 0; i < A; ++i)
#pragma unroll
            for (int c = 0; c < G::CPT; ++c)
                x[c][i] = split30_held(i < size ? S.s.tile[i][G::c_col(tid) + c][lds_off(G::c_row(tid))] : 0);
        __syncthreads();  // the targets take over the LDS
    } else {
        uint64_t v[A][G::CPT];
#pragma unroll
        for (int i = 0; i < A; ++i) {
            const uint64_t* src = J.t + (size_t)(start + (i < size ? i : size - 1)) * G::N + c_at;
            if constexpr (G::CPT == 2) {
                const u64x2 w = ld2(src);
                v[i][0] = w.x, v[i][1] = w.y;
            } else {
                v[i][0] = gp(src)[0];
            }
        }
#pragma unroll
        for (int i = 0; i < A; ++i)
#pragma unroll
            for (int c = 0; c < G::CPT; ++c) x[c][i] = split30_held(i < size ? v[i][c] : 0);
    }
    const size_t m_at = (size_t)(d * T.alpha + size - 1) * T.np * A;
    uint64_t* out = J.ext + (size_t)d * (nl + T.K) * G::N;
    auto pos_of = [&](int m) { const int k = m * TG + tg; return k < start ? k : k + size; };
    auto pid_of = [&](int k) { return pos_pid(pos_of(k), nl, 0, T.L + 1); };
    int buf = 0;
    const int s_tgt = __builtin_amdgcn_readfirstlane((int)(tid / G::N1)), s_row = (int)(tid % G::N1);
    auto s_pid = [&](int k) { const int i = k + s_tgt < k1 ? k + s_tgt : k1 - 1; return pid_of(i); };
    ConvTw tw;
    tw.load(T, s_pid(0), s_row);
    for (int k = 0; k < k1; k += G::TB, buf ^= 1) {
#pragma unroll
        for (int q = 0; q < G::TPT; ++q) {
            const int i = c_tgt + q;
            if (k + i >= k1) continue;
            const int pid = pid_of(k + i);
            const PrimeInfo P = cld(T.primes + pid);
            conv_tile<A>(T, pid, P, x, T.modup_mat + m_at, T.modup_fp + m_at, &S.t.tile[buf][i][G::c_col(tid)],
                         lds_off(G::c_row(tid)));
        }
        tw.put(S, buf, s_tgt, s_row);
        if (k + G::TB < k1) tw.load(T, s_pid(k + G::TB), s_row);
        __syncthreads();
        if (k + n_tgt < k1) conv_columns(T, pid_of(k + n_tgt), S, buf, n_tgt);
        __syncthreads();
        conv_store(S, buf, col0, [&](int i) -> uint64_t* {
            return k + i < k1 ? out + (size_t)pos_of(k + i) * G::N : nullptr;
        });
    }
}

// ------------------------------------------------- rows + inner product ----
// One tile of rows at one prime: the digits' row passes (a digit's own
// positions come from the evaluation-form source), the inner product with both
// key parts, and the inverse transform's row pass where the limb goes down.
// Items (job, prime, tile); with several jobs the job runs fastest, so that
// the jobs of one key (they are sorted by key), or of one source, read its rows
// from the XCD's L2.  EVAL: the digits are in evaluation form already (a hoisted
// set runs their row pass once for all its keys; doing it per key, or keeping
// three digits in registers through a loop over the keys, spilled at 128
// registers and took 348 us for 9 keys at level 17).
struct KskGrid {
    uint32_t items, chunk;
    FastDiv n;
    int q_primes;  // primes below q_primes are the Q primes of the list's top level
};

template <int LOGN, bool EVAL, bool ROT>
__global__ void __launch_bounds__(FRows<LOGN>::NTR, 4) k_rows_ksk(DevTables T, KskJobs L, KskGrid g) {
    using G = FRows<LOGN>;
    constexpr int TPL = G::N1 / G::RR;
    __shared__ uint64_t lds[G::RR * G::SR];
    const uint32_t item = xcd_item(g.chunk);
    if (item >= g.items) return;
    const uint32_t u = g.n.div(item), z = item - u * g.n.d;
    const int py = (int)(u / TPL);
    const int pid = py < g.q_primes ? py : T.L + 1 + (py - g.q_primes);
    const int t = threadIdx.x % G::TR, rr = threadIdx.x / G::TR;
    const uint32_t r = (u % TPL) * G::RR + rr;
    const uint32_t in0 = r * G::N2, x0 = r * G::N2 + G::mem(t, 0);
    const KskJob J = L.dev ? get_job(L, (int)z) : get_inline(L, (int)z);
    const int nl = __builtin_amdgcn_readfirstlane(J.level) + 1;
    if (pid <= T.L && pid >= nl) return;  // a Q prime above this job's level
    const int pos = pid <= T.L ? pid : nl + (pid - (T.L + 1));
    const PrimeInfo P = cld(T.primes + pid);
    const int npos = nl + T.K, nd = num_digits(T, nl);
    const int own_d = pos < nl ? pos / T.alpha : -1;
    const bool special = pos >= nl;
    const size_t limb = (size_t)pos * G::N;
    with_arith(T, pid, P, [&](const auto& ar) {
        using A = std::decay_t<decltype(ar)>;
        using V = typename A::V;
        V* sub = reinterpret_cast<V*>(lds) + rr * G::SR;
        const auto* tf = A::fwd(T) + (size_t)pid * G::N;
        // digit d's row in evaluation form
        auto digit = [&](int d, V* v) {
            if (d == own_d) {
                const u64x2 a = ld2(J.own + limb + x0), b = ld2(J.own + limb + x0 + 2);
                v[0] = ar.from(a.x), v[1] = ar.from(a.y), v[2] = ar.from(b.x), v[3] = ar.from(b.y);
                return;
            }
            if constexpr (EVAL) {
                const uint64_t* e = J.ext + ((size_t)d * npos + pos) * G::N;
                const u64x2 a = ld2(e + x0), b = ld2(e + x0 + 2);
                v[0] = ar.from(a.x), v[1] = ar.from(a.y), v[2] = ar.from(b.x), v[3] = ar.from(b.y);
                return;
            }
            const gu64* e = gp(J.ext) + ((size_t)d * npos + pos) * G::N;
            uint64_t m[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) m[k] = e[in0 + elem<2, G::LO1, G::NB1>(t, k)];
#pragma unroll
            for (int k = 0; k < 4; ++k) v[k] = A::unpack(m[k]);
            lds_sync<G::WAVE>();  // the row pass before has read its words
            fwd_row<G, false>(ar, sub, v, t, G::N1 + r, tf);
#pragma unroll
            for (int k = 0; k < 4; ++k) v[k] = ar.term_fwd(v[k]);
        };
        auto mac = [&](typename A::Sum* sa, typename A::Sum* sb, int d, const V* v) {
            const size_t kx = ((size_t)d * T.np + pid) * G::N + x0;
            const u64x2 a = ld2(J.ka + kx), ah = ld2(J.ka + kx + 2), b = ld2(J.kb + kx), bh = ld2(J.kb + kx + 2);
            ar.mac(sa[0], v[0], a.x), ar.mac(sa[1], v[1], a.y), ar.mac(sa[2], v[2], ah.x), ar.mac(sa[3], v[3], ah.y);
            ar.mac(sb[0], v[0], b.x), ar.mac(sb[1], v[1], b.y), ar.mac(sb[2], v[2], bh.x), ar.mac(sb[3], v[3], bh.y);
        };
        // sigma(sum + c0') + base: sigma sends a row to one row (its columns are scattered
        // in LDS, the index map is STORE_MODDOWN_AUTO's), so what goes out is whole rows
        // and the kernel that gathered (23 us a giant step of 25 + 8 limbs) is not run
        auto rotate = [&](typename A::Sum* sums, uint64_t* out, const uint64_t* base, const uint64_t* add0,
                          uint64_t* rdown) {
            uint64_t u[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) u[k] = ar.canon_in(ar.sum(sums[k], P));
            if (add0 && (!J.scale_p || !special)) {
                const u64x2 f0 = ld2(add0 + limb + x0), f1 = ld2(add0 + limb + x0 + 2);
                uint64_t f[4] = {f0.x, f0.y, f1.x, f1.y};
                if (J.scale_p) {
                    const ShoupConst pm = cld(T.pmodq + pid);
#pragma unroll
                    for (int k = 0; k < 4; ++k) f[k] = mul_shoup(f[k], pm.w, pm.wp, P.p);
                }
#pragma unroll
                for (int k = 0; k < 4; ++k) u[k] = addmod(u[k], f[k], P.p);
            }
            const uint32_t cx = (uint32_t)(((2ull * brev_bits(r, G::K1) + 1) * J.autok) & (2ull * G::N - 1));
            const uint32_t rdst = brev_bits((cx & (2u * G::N1 - 1)) >> 1, G::K1), coff = cx >> (G::K1 + 1);
            uint64_t* words = reinterpret_cast<uint64_t*>(sub);
            lds_sync<G::WAVE>();
#pragma unroll
            for (int k = 0; k < 4; ++k)
                words[lds_off(brev_bits((brev_bits(G::mem(t, k), G::K2) * J.autok + coff) & (G::N2 - 1), G::K2))] = u[k];
            lds_sync<G::WAVE>();
#pragma unroll
            for (int k = 0; k < 4; ++k) u[k] = words[lds_off(G::mem(t, k))];
            const uint32_t y0 = rdst * G::N2 + G::mem(t, 0);
            if (base) {
                const u64x2 f0 = ld2(base + limb + y0), f1 = ld2(base + limb + y0 + 2);
                u[0] = addmod(u[0], f0.x, P.p), u[1] = addmod(u[1], f0.y, P.p);
                u[2] = addmod(u[2], f1.x, P.p), u[3] = addmod(u[3], f1.y, P.p);
            }
            st2(out + limb + y0, u[0], u[1]);
            st2(out + limb + y0 + 2, u[2], u[3]);
            if (rdown && special) {
                V a[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) a[k] = ar.from(u[k]);
                lds_sync<G::WAVE>();  // the words are read
                inv_row<G>(ar, sub, a, t, G::N1 + rdst, A::inv(T) + (size_t)pid * G::N);
                gu64* o = gp(rdown) + (size_t)(pos - nl) * G::N;
#pragma unroll
                for (int k = 0; k < 4; ++k) o[rdst * G::N2 + elem<2, G::LOL, G::NBI>(t, k)] = A::pack(a[k]);
            }
        };
        auto finish = [&](typename A::Sum* sums, uint64_t* acc, uint64_t* down, const uint64_t* add) {
            V a[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) a[k] = ar.sum(sums[k], P);
            if (down == nullptr || !(special || (add != nullptr && pos == nl - 1))) {
                st2(acc + limb + x0, ar.canon_in(a[0]), ar.canon_in(a[1]));
                st2(acc + limb + x0 + 2, ar.canon_in(a[2]), ar.canon_in(a[3]));
                return;
            }
            if (!special) {
                const ShoupConst pinv = cld(T.pinv + pid);
                const u64x2 f0 = ld2(add + limb + x0), f1 = ld2(add + limb + x0 + 2);
                a[0] = ar.mul_add(a[0], pinv, f0.x);
                a[1] = ar.mul_add(a[1], pinv, f0.y);
                a[2] = ar.mul_add(a[2], pinv, f1.x);
                a[3] = ar.mul_add(a[3], pinv, f1.y);
            }
            lds_sync<G::WAVE>();  // the row pass before has read its words
            inv_row<G>(ar, sub, a, t, G::N1 + r, A::inv(T) + (size_t)pid * G::N);
            gu64* o = gp(down) + (special ? (size_t)(1 + pos - nl) * G::N : (size_t)0);
#pragma unroll
            for (int k = 0; k < 4; ++k) o[in0 + elem<2, G::LOL, G::NBI>(t, k)] = A::pack(a[k]);
        };
        typename A::Sum sa[4] = {}, sb[4] = {};
#pragma unroll 1
        for (int d = 0; d < nd; ++d) {
            V v[4];
            digit(d, v);
            mac(sa, sb, d, v);
        }
        if constexpr (ROT) {
            rotate(sa, J.rot_a, J.base_a, nullptr, J.rot_down);
            rotate(sb, J.rot_b, J.base_b, J.add0, nullptr);
        } else {
            finish(sa, J.acc_a, J.down_a, J.add_a);
            finish(sb, J.acc_b, J.down_b, J.add_b);
        }
    });
}

// ---------------------------------------------------------- launchers ----
bool fused_ok(const DevTables& T) {
    return T.logN >= FUSED_LOGN_MIN && T.logN <= FUSED_LOGN_MAX && T.dnum <= FUSED_DIGITS &&
           T.alpha <= FUSED_CONV_MAX && T.K <= fused_down_max(T.logN) && T.modup_one_reduce && T.moddown_one_reduce;
}

bool fused_inv_cols(const DevTables& T) { return fused_ok(T) && T.logN <= CONV_INV_LOGN; }

hipError_t launch_tensor_rows(const DevTables& T, const TensorJobs& L, int max_nl, hipStream_t s) {
    if (L.n <= 0 || max_nl <= 0) return hipSuccess;
    return by_logn(T.logN, [&](auto ln) {
        using G = FRows<decltype(ln)::value>;
        constexpr int TPL = G::N1 / G::RR;
        const size_t items = (size_t)L.n * max_nl * TPL;
        const XcdGrid x = xcd_chunks(items, XCD_TILES);
        const RowsGrid g{(uint32_t)items, x.chunk, FastDiv(max_nl, items)};
        hipLaunchKernelGGL((k_tensor_rows<decltype(ln)::value>), x.grid, dim3(G::NTR), 0, s, T, L, g);
    });
}

template <int LOGN, int A>
static void modup_cols(const DevTables& T, const ModUpJobs& L, int max_nd, int targets, hipStream_t s) {
    using G = ConvCols<LOGN>;
    const int tg = conv_launch_groups(TUNE_MODUP, LOGN, max_nd * L.n, (size_t)G::TPL * max_nd * L.n, targets, G::TB, A);
    const size_t items = (size_t)L.n * max_nd * tg * G::TPL;
    const XcdGrid x = conv_grid(items, G::TPL);
    const ConvGrid g{(uint32_t)items, x.chunk, FastDiv(tg, items), FastDiv(max_nd, items)};
    hipLaunchKernelGGL((k_modup_cols<LOGN, A>), x.grid, dim3(G::NT), 0, s, T, L, g);
}

template <int LOGN>
static void modup_cols_a(const DevTables& T, const ModUpJobs& L, int max_nd, int targets, hipStream_t s) {
    switch (T.alpha) {  // the template bound the matrix rows are padded to
        case 1: modup_cols<LOGN, 1>(T, L, max_nd, targets, s); break;
        case 2: modup_cols<LOGN, 2>(T, L, max_nd, targets, s); break;
        case 3: modup_cols<LOGN, 3>(T, L, max_nd, targets, s); break;
        case 4: modup_cols<LOGN, 4>(T, L, max_nd, targets, s); break;
        case 5: modup_cols<LOGN, 5>(T, L, max_nd, targets, s); break;
        case 6: modup_cols<LOGN, 6>(T, L, max_nd, targets, s); break;
        case 7: modup_cols<LOGN, 7>(T, L, max_nd, targets, s); break;
        case 8: modup_cols<LOGN, 8>(T, L, max_nd, targets, s); break;
        case 9: modup_cols<LOGN, 9>(T, L, max_nd, targets, s); break;
        case 10: modup_cols<LOGN, 10>(T, L, max_nd, targets, s); break;
        default: modup_cols<LOGN, 12>(T, L, max_nd, targets, s); break;
    }
}

// The most targets a digit of any level up to the list's top has: all
// positions but a full digit's (or all but the top level's, within one digit).
static int modup_targets(const DevTables& T, int max_nl) { return T.K + (max_nl > T.alpha ? max_nl - 1 : 0); }

hipError_t launch_modup_cols(const DevTables& T, const ModUpJobs& L, int max_nd, int max_nl, hipStream_t s) {
    if (L.n <= 0 || max_nd <= 0) return hipSuccess;
    if (!fused_ok(T)) return hipErrorInvalidValue;
    const int targets = modup_targets(T, max_nl);
    return by_logn(T.logN, [&](auto ln) { modup_cols_a<decltype(ln)::value>(T, L, max_nd, targets, s); });
}

int fused_conv_tg(const DevTables& T, int kind, int convs) {
    const int nl = kind == TUNE_MODUP && convs < T.dnum ? convs * T.alpha : T.L + 1;
    const int targets = kind == TUNE_MODUP ? modup_targets(T, nl) : nl;
    int tg = 0;
    (void)by_logn(T.logN, [&](auto ln) {
        using G = ConvCols<decltype(ln)::value>;
        const int sources = kind == TUNE_MODUP ? conv_bound(T.alpha) : conv_bound(T.K) + 1;  // of a product
        tg = conv_launch_groups(kind, T.logN, convs, (size_t)G::TPL * convs, targets, G::TB, sources);
    });
    return tg;
}

hipError_t launch_rows_ksk(const DevTables& T, const KskJobs& L, int max_npos, hipStream_t s, bool eval, bool rot) {
    if (L.n <= 0 || max_npos <= 0) return hipSuccess;
    if (!fused_ok(T)) return hipErrorInvalidValue;
    return by_logn(T.logN, [&](auto ln) {
        constexpr int LN = decltype(ln)::value;
        using G = FRows<LN>;
        constexpr int TPL = G::N1 / G::RR;
        const size_t items = (size_t)L.n * max_npos * TPL;
        const XcdGrid x = xcd_chunks(items, XCD_TILES);
        const KskGrid g{(uint32_t)items, x.chunk, FastDiv(L.n, items), max_npos - T.K};
        const dim3 b(G::NTR);
        if (eval && rot)
            hipLaunchKernelGGL((k_rows_ksk<LN, true, true>), x.grid, b, 0, s, T, L, g);
        else if (eval)
            hipLaunchKernelGGL((k_rows_ksk<LN, true, false>), x.grid, b, 0, s, T, L, g);
        else if (rot)
            hipLaunchKernelGGL((k_rows_ksk<LN, false, true>), x.grid, b, 0, s, T, L, g);
        else
            hipLaunchKernelGGL((k_rows_ksk<LN, false, false>), x.grid, b, 0, s, T, L, g);
    });
}

}  // namespace fides
