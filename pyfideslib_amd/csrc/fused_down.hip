// ModDown's conversion from the special primes (with the rescale that follows
// folded in, see k_moddown_conv) and the column pass of its outputs'
// transform in one kernel; layout and reasons as in fused.hip.
#include "fused.hpp"

namespace fides {

template <int LOGN, int KK, bool RESCALE>
__global__ void __launch_bounds__(512, 4) k_moddown_cols(DevTables T, ModDownJobs L, ConvGrid g) {
    using G = ConvCols<LOGN>;
    __shared__ ConvLds<LOGN, KK + (RESCALE ? 1 : 0)> S;
    const uint32_t item = xcd_item(g.chunk);
    if (item >= g.items) return;
    const uint32_t u = item / G::TPL, z = g.tg.div(u);
    const int tg = (int)(u - z * g.tg.d);
    const ModDownJob J = L.dev ? get_job(L, (int)z) : get_inline(L, (int)z);
    const int nl = __builtin_amdgcn_readfirstlane(J.level) + 1, l = nl - 1;
    const int ntarget = RESCALE ? l : nl;
    // targets tg, tg + TG, ..: the 64-bit ones come last and are dealt out evenly
    const int TG = (int)g.tg.d, k1 = (ntarget - tg + TG - 1) / TG;
    if (k1 <= 0) return;
    const uint32_t tid = threadIdx.x;
    const uint32_t col0 = (item % G::TPL) * G::CC;
    const uint32_t c_at = G::c_row(tid) * G::N2 + col0 + G::c_col(tid);
    const int c_tgt = __builtin_amdgcn_readfirstlane(G::c_tgt(tid));
    const int n_tgt = __builtin_amdgcn_readfirstlane(G::n_tgt(tid));
    const int K = KK > 10 ? T.K : KK;  // past 10 the matrix rows are padded with zeros
    Half2 x[G::CPT][KK];
    uint64_t top[G::CPT];
    if constexpr (conv_inv<LOGN>()) {
        // the special limbs, and the limb that a rescale drops
        conv_sources(
            T, S, K + (RESCALE ? 1 : 0), col0, [&](int i) { return i < K ? J.t + (size_t)i * G::N : J.top_acc; },
            [&](int i) { return i < K ? T.L + 1 + i : l; },
            [&](int i) { return i < K ? T.iscale_moddown + (size_t)i * 2 : T.iscale_plain + (size_t)l * 2; });
#pragma unroll
        for (int i = 0; i < KK; ++i)
#pragma unroll
            for (int c = 0; c < G::CPT; ++c)
                x[c][i] = split30_held(i < K ? S.s.tile[i][G::c_col(tid) + c][lds_off(G::c_row(tid))] : 0);
        if constexpr (RESCALE) {
#pragma unroll
            for (int c = 0; c < G::CPT; ++c) top[c] = S.s.tile[K][G::c_col(tid) + c][lds_off(G::c_row(tid))];
        }
        __syncthreads();  // the targets take over the LDS
    } else {
        uint64_t v[KK][G::CPT];
#pragma unroll
        for (int i = 0; i < KK; ++i) {
            const uint64_t* src = J.t + (size_t)(i < K ? i : K - 1) * G::N + c_at;
            if constexpr (G::CPT == 2) {
                const u64x2 w = ld2(src);
                v[i][0] = w.x, v[i][1] = w.y;
            } else {
                v[i][0] = gp(src)[0];
            }
        }
        if constexpr (RESCALE) {
#pragma unroll
            for (int c = 0; c < G::CPT; ++c) top[c] = gp(J.top_acc)[c_at + c];
        }
#pragma unroll
        for (int i = 0; i < KK; ++i)
#pragma unroll
            for (int c = 0; c < G::CPT; ++c) x[c][i] = split30_held(i < K ? v[i][c] : 0);
    }
    // the dropped limb less its converted part, centered on a rescale; as a double
    // where its prime is on the FP64 units, and else in [0, q_l)
    uint64_t half = 0;
    const bool l_fp = is_fp(T, l);
    if constexpr (RESCALE) {
        const PrimeInfo Pl = cld(T.primes + l);
        const ShoupConst pl = cld(T.pinv + l);
        const MatRow<KK> row = cld(reinterpret_cast<const MatRow<KK>*>(T.moddown_mat + (size_t)l * KK));
        half = Pl.p >> 1;
#pragma unroll
        for (int c = 0; c < G::CPT; ++c) {
            uint64_t lo, hi;
            conv_acc<KK>(x[c], row, lo, hi);
            top[c] = submod(top[c], mul_shoup(reduce128(lo, hi, Pl), pl.w, pl.wp, Pl.p), Pl.p);
            if (l_fp) top[c] = FpArith::pack(fp_from(top[c]) - (top[c] > half ? Pl.pd : 0.0));
        }
    }
    int buf = 0;
    const int s_tgt = __builtin_amdgcn_readfirstlane((int)(tid / G::N1)), s_row = (int)(tid % G::N1);
    auto s_pid = [&](int k) { const int i = k + s_tgt < k1 ? k + s_tgt : k1 - 1; return i * TG + tg; };
    ConvTw tw;
    tw.load(T, s_pid(0), s_row);
    for (int k = 0; k < k1; k += G::TB, buf ^= 1) {
#pragma unroll
        for (int q = 0; q < G::TPT; ++q) {
            const int i = c_tgt + q, pid = (k + i) * TG + tg;
            if (k + i >= k1) continue;
            const PrimeInfo P = cld(T.primes + pid);
            uint64_t(*tile)[G::SC] = &S.t.tile[buf][i][G::c_col(tid)];
            const uint32_t at = lds_off(G::c_row(tid));
            if constexpr (RESCALE) {
                const ShoupConst pi = cld(T.pinv + pid);
                // centered lift of the dropped limb into q_i
                auto lift = [&](uint64_t t) {
                    uint64_t sw = reduce64(t, P);
                    if (t > half) sw = submod(sw, cld(T.qlmodq + (size_t)l * (T.L + 1) + pid), P.p);
                    return sw;
                };
                if (is_fp(T, pid)) {
                    const FpArith ar(P);
                    const MatRowFp<KK> row = cld(reinterpret_cast<const MatRowFp<KK>*>(T.moddown_fp + (size_t)pid * KK));
#pragma unroll
                    for (int c = 0; c < G::CPT; ++c) {
                        const double s = l_fp ? ar.term_fwd(FpArith::unpack(top[c])) : fp_from(lift(top[c]));
                        tile[c][at] = FpArith::pack(ar.scale_add(conv_fp<KK>(x[c], row, P), pi, s));
                    }
                } else {
                    const IntArith ar(P);
                    const MatRow<KK> row = cld(reinterpret_cast<const MatRow<KK>*>(T.moddown_mat + (size_t)pid * KK));
                    const double ql = cld(T.primes + l).pd;
#pragma unroll
                    for (int c = 0; c < G::CPT; ++c) {
                        uint64_t lo, hi;
                        conv_acc<KK>(x[c], row, lo, hi);
                        uint64_t t = top[c];
                        if (l_fp) {
                            const double td = FpArith::unpack(t);
                            t = fp_to(td < 0 ? td + ql : td);
                        }
                        tile[c][at] = ar.scale_add(ar.from_lazy(reduce128_lazy(lo, hi, P)), pi, lift(t));
                    }
                }
            } else {
                conv_tile<KK>(T, pid, P, x, T.moddown_mat, T.moddown_fp, tile, at);
            }
        }
        tw.put(S, buf, s_tgt, s_row);
        if (k + G::TB < k1) tw.load(T, s_pid(k + G::TB), s_row);
        __syncthreads();
        if (k + n_tgt < k1) conv_columns(T, (k + n_tgt) * TG + tg, S, buf, n_tgt);
        __syncthreads();
        conv_store(S, buf, col0, [&](int i) -> uint64_t* {
            return k + i < k1 ? J.y + (size_t)((k + i) * TG + tg) * G::N : nullptr;
        });
    }
}

template <int LOGN, int KK>
static void moddown_cols(const DevTables& T, const ModDownJobs& L, int targets, bool rescale, hipStream_t s) {
    using G = ConvCols<LOGN>;
    const int tg = conv_launch_groups(TUNE_MODDOWN, LOGN, L.n, (size_t)G::TPL * L.n, targets, G::TB,
                                      KK + rescale);
    const size_t items = (size_t)L.n * tg * G::TPL;
    const XcdGrid x = conv_grid(items, G::TPL);
    const ConvGrid g{(uint32_t)items, x.chunk, FastDiv(tg, items), FastDiv(1, items)};
    if constexpr (KK <= fused_down_max(LOGN)) {
        if (rescale)
            hipLaunchKernelGGL((k_moddown_cols<LOGN, KK, true>), x.grid, dim3(G::NT), 0, s, T, L, g);
        else
            hipLaunchKernelGGL((k_moddown_cols<LOGN, KK, false>), x.grid, dim3(G::NT), 0, s, T, L, g);
    }
}

template <int LOGN>
static hipError_t moddown_cols_k(const DevTables& T, const ModDownJobs& L, int targets, bool rescale, hipStream_t s) {
    switch (T.K) {  // the template bound the matrix rows are padded to
        case 1: moddown_cols<LOGN, 1>(T, L, targets, rescale, s); break;
        case 2: moddown_cols<LOGN, 2>(T, L, targets, rescale, s); break;
        case 3: moddown_cols<LOGN, 3>(T, L, targets, rescale, s); break;
        case 4: moddown_cols<LOGN, 4>(T, L, targets, rescale, s); break;
        case 5: moddown_cols<LOGN, 5>(T, L, targets, rescale, s); break;
        case 6: moddown_cols<LOGN, 6>(T, L, targets, rescale, s); break;
        case 7: moddown_cols<LOGN, 7>(T, L, targets, rescale, s); break;
        case 8: moddown_cols<LOGN, 8>(T, L, targets, rescale, s); break;
        case 9: moddown_cols<LOGN, 9>(T, L, targets, rescale, s); break;
        case 10: moddown_cols<LOGN, 10>(T, L, targets, rescale, s); break;
        default: moddown_cols<LOGN, 12>(T, L, targets, rescale, s); break;
    }
    return hipGetLastError();
}

hipError_t launch_moddown_cols(const DevTables& T, const ModDownJobs& L, int max_nl, bool rescale, hipStream_t s) {
    if (L.n <= 0) return hipSuccess;
    if (!fused_ok(T)) return hipErrorInvalidValue;
    const int targets = rescale ? max_nl - 1 : max_nl;
    if (targets <= 0) return hipErrorInvalidValue;
    switch (T.logN) {
        case 12: return moddown_cols_k<12>(T, L, targets, rescale, s);
        case 13: return moddown_cols_k<13>(T, L, targets, rescale, s);
        case 14: return moddown_cols_k<14>(T, L, targets, rescale, s);
        case 15: return moddown_cols_k<15>(T, L, targets, rescale, s);
        case 16: return moddown_cols_k<16>(T, L, targets, rescale, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace fides
