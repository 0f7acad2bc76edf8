// Rescaling in three launches: the row pass of the dropped limb's inverse
// transform (of a product with a plaintext on the way: the other limbs of that
// product are formed in the last launch's epilogue, so it is never written),
// its column pass with the lifts into the limbs that stay and their column
// pass, and the transform's row pass (launch_ntt_fwd).
//
// Bound by launches and latency up to a few limbs and by memory past it.
#include "fused.hpp"

namespace fides {

// Items (job, tile of rows).
template <int LOGN>
__global__ void __launch_bounds__(FRows<LOGN>::NTR) k_top_rows(DevTables T, RescaleJobs L) {
    using G = FRows<LOGN>;
    constexpr int TPL = G::N1 / G::RR;
    __shared__ uint64_t lds[G::RR * G::SR];
    const int z = blockIdx.x / TPL;
    const RescaleJob J = L.dev ? get_job(L, z) : get_inline(L, z);
    const int t = threadIdx.x % G::TR, rr = threadIdx.x / G::TR;
    const uint32_t r = (blockIdx.x % TPL) * G::RR + rr;
    const size_t x = (size_t)J.level * G::N + r * G::N2 + G::mem(t, 0);  // 4 neighbouring words
    const u64x2 a0 = ld2(J.a + x), a1 = ld2(J.a + x + 2);
    u64x2 w0{0, 0}, w1{0, 0};
    if (J.w) w0 = ld2(J.w + x), w1 = ld2(J.w + x + 2);
    const PrimeInfo P = cld(T.primes + J.level);
    with_arith(T, J.level, P, [&](const auto& ar) {
        using A = std::decay_t<decltype(ar)>;
        using V = typename A::V;
        uint64_t u[4] = {a0.x, a0.y, a1.x, a1.y};
        if (J.w) {
            const uint64_t w[4] = {w0.x, w0.y, w1.x, w1.y};
#pragma unroll
            for (int j = 0; j < 4; ++j) u[j] = ar.mul(u[j], w[j], P);
        }
        V v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = ar.from(u[j]);
        inv_row<G>(ar, reinterpret_cast<V*>(lds) + rr * G::SR, v, t, G::N1 + r, A::inv(T) + (size_t)J.level * G::N);
        gu64* o = gp(J.top);
#pragma unroll
        for (int j = 0; j < 4; ++j) o[r * G::N2 + elem<2, G::LOL, G::NBI>(t, j)] = A::pack(v[j]);
    });
}

// Items (job, target group, tile), layout as the conversion kernels': the
// dropped limb's columns are transformed once per group and held, centered
// (as doubles where its prime is on the FP64 units), for its targets.
template <int LOGN>
__global__ void __launch_bounds__(512, 6) k_rescale_cols(DevTables T, RescaleJobs L, ConvGrid g) {
    using G = ConvCols<LOGN>;
    __shared__ ConvLds<LOGN, 1, true> S;
    const uint32_t item = xcd_item(g.chunk);
    if (item >= g.items) return;
    const uint32_t u = item / G::TPL, z = g.tg.div(u);
    const int tg = (int)(u - z * g.tg.d);
    const RescaleJob J = L.dev ? get_job(L, (int)z) : get_inline(L, (int)z);
    const int l = __builtin_amdgcn_readfirstlane(J.level);
    const int TG = (int)g.tg.d, k1 = (l - tg + TG - 1) / TG;
    if (k1 <= 0) return;
    const uint32_t tid = threadIdx.x;
    const uint32_t col0 = (item % G::TPL) * G::CC;
    const int c_tgt = __builtin_amdgcn_readfirstlane(G::c_tgt(tid));
    const int n_tgt = __builtin_amdgcn_readfirstlane(G::n_tgt(tid));
    conv_sources(
        T, S, 1, col0, [&](int) { return (const uint64_t*)J.top; }, [&](int) { return l; },
        [&](int) { return T.iscale_plain + (size_t)l * 2; });
    const bool l_fp = is_fp(T, l);
    const PrimeInfo Pl = cld(T.primes + l);
    uint64_t top[G::CPT];
#pragma unroll
    for (int c = 0; c < G::CPT; ++c) {
        top[c] = S.s.tile[0][G::c_col(tid) + c][lds_off(G::c_row(tid))];
        if (l_fp) top[c] = FpArith::pack(fp_from(top[c]) - (top[c] > (Pl.p >> 1) ? Pl.pd : 0.0));
    }
    __syncthreads();  // the targets take over the LDS
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
            if (is_fp(T, pid) && l_fp) {
                const FpArith ar(P);
#pragma unroll
                for (int c = 0; c < G::CPT; ++c) tile[c][at] = FpArith::pack(ar.term_fwd(FpArith::unpack(top[c])));
            } else {
                const SwitchLift lift(T, l, pid);
#pragma unroll
                for (int c = 0; c < G::CPT; ++c) {
                    uint64_t x = top[c];
                    if (l_fp) {
                        const double td = FpArith::unpack(x);
                        x = fp_to(td < 0 ? td + Pl.pd : td);
                    }
                    x = lift(x, P);
                    tile[c][at] = is_fp(T, pid) ? FpArith::pack(fp_from(x)) : x;
                }
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

bool rescale_ok(const DevTables& T) { return T.logN >= FUSED_LOGN_MIN && T.logN <= FUSED_LOGN_MAX; }

hipError_t launch_rescale_cols(const DevTables& T, const RescaleJobs& L, int max_level, hipStream_t s) {
    if (L.n <= 0) return hipSuccess;
    if (max_level <= 0 || !rescale_ok(T)) return hipErrorInvalidValue;
    return by_logn(T.logN, [&](auto ln) {
        constexpr int LN = decltype(ln)::value;
        using R = FRows<LN>;
        using G = ConvCols<LN>;
        hipLaunchKernelGGL((k_top_rows<LN>), dim3(R::N1 / R::RR * L.n), dim3(R::NTR), 0, s, T, L);
        const int tg = fused_groups((size_t)G::TPL * L.n, max_level, G::TB);
        const size_t items = (size_t)L.n * tg * G::TPL;
        const XcdGrid x = conv_grid(items, G::TPL);
        const ConvGrid g{(uint32_t)items, x.chunk, FastDiv(tg, items), FastDiv(1, items)};
        hipLaunchKernelGGL((k_rescale_cols<LN>), x.grid, dim3(G::NT), 0, s, T, L, g);
    });
}

}  // namespace fides
