// The fused kernels compiled for the host and run lane by lane: between two
// waits (of the wave or of the block) the lanes go one after the other, first
// in ascending order, then in descending order.  A kernel whose lanes exchange
// words without a wait between them gives different results in the two.
#include <ucontext.h>

#include <cstdio>
#include <functional>
#include <memory>
#include <random>
#include <type_traits>
#include <vector>

#include "../../pyfideslib_amd/csrc/fused.hip"
#include "../../pyfideslib_amd/csrc/fused_down.hip"
#include "../../pyfideslib_amd/csrc/rescale.hip"

// no tuning configuration: the launchers' rules
int fides::conv_set_tg(int, int, int, int) { return 0; }

dim3 threadIdx, blockIdx, blockDim, gridDim;

namespace {

enum State { READY, WAVE, BLOCK, DONE };
struct Lane {
    ucontext_t ctx;
    std::unique_ptr<char[]> stack;
    State state;
};
constexpr size_t STACK = 256 << 10;
std::vector<Lane> lanes(512);
ucontext_t scheduler;
std::function<void()> body;
bool descending = false;

void wait(State s) {
    Lane& l = lanes[threadIdx.x];
    l.state = s;
    swapcontext(&l.ctx, &scheduler);
}
void lane_main() {
    body();
    wait(DONE);
}
void run_lane(int i) {
    threadIdx.x = (unsigned)i;
    swapcontext(&scheduler, &lanes[i].ctx);
}
int count(int from, int to, State s) {
    int n = 0;
    for (int i = from; i < to; ++i) n += lanes[i].state == s;
    return n;
}
// One block of n lanes.
void run_block(int n) {
    for (int i = 0; i < n; ++i) {
        Lane& l = lanes[i];
        if (!l.stack) l.stack.reset(new char[STACK]);
        getcontext(&l.ctx);
        l.ctx.uc_stack.ss_sp = l.stack.get();
        l.ctx.uc_stack.ss_size = STACK;
        l.ctx.uc_link = nullptr;
        makecontext(&l.ctx, lane_main, 0);
        l.state = READY;
    }
    const int waves = n / 64;
    while (count(0, n, DONE) < n) {
        for (int k = 0; k < waves; ++k) {
            const int from = 64 * (descending ? waves - 1 - k : k), to = from + 64;
            while (count(from, to, READY)) {
                for (int j = 0; j < 64; ++j) {
                    const int i = descending ? to - 1 - j : from + j;
                    if (lanes[i].state == READY) run_lane(i);
                }
                if (count(from, to, WAVE) == 64)
                    for (int i = from; i < to; ++i) lanes[i].state = READY;
            }
            if (count(from, to, WAVE)) {
                std::printf("the lanes of a wave wait for different things\n");
                std::exit(1);
            }
        }
        for (int i = 0; i < n; ++i)
            if (lanes[i].state == BLOCK) lanes[i].state = READY;
    }
}

using namespace fides;
std::mt19937_64 rng(1);

struct Set {
    DevTables T;
    std::vector<uint64_t> p;
    std::vector<PrimeInfo> primes;
    std::vector<std::vector<uint64_t>> words;  // every table and buffer
    uint64_t* buf(size_t n) {
        words.emplace_back(n, 0);
        return words.back().data();
    }
    uint64_t below(int t) { return rng() % p[t]; }
    ShoupConst sc(int t) {
        const uint64_t w = below(t);
        return ShoupConst{w, (uint64_t)(((unsigned __int128)w << 64) / p[t])};
    }
    // n constants, entry i of prime t(i)
    const ShoupConst* consts(size_t n, const std::function<int(size_t)>& t) {
        ShoupConst* c = (ShoupConst*)buf(2 * n);
        for (size_t i = 0; i < n; ++i) c[i] = sc(t(i));
        return c;
    }
    const double* doubles(size_t per) {
        double* d = (double*)buf(p.size() * per);
        for (size_t i = 0; i < p.size() * per; ++i) d[i] = (double)(int64_t)(below((int)(i / per)) - p[i / per] / 2);
        return d;
    }
    // [rows][np][n] constants as residues and, for primes on the FP64 units, split in halves
    const uint64_t* matrix(size_t rows, int n, const ConvFp** fp) {
        const size_t size = rows * p.size() * n;
        uint64_t* m = buf(size);
        ConvFp* f = (ConvFp*)buf(2 * size);
        for (size_t i = 0; i < size; ++i) {
            m[i] = below((int)(i / n % p.size()));
            f[i] = ConvFp{(int32_t)(rng() >> 36), (int32_t)(rng() >> 45), (int32_t)(rng() >> 36), (int32_t)(rng() >> 45)};
        }
        *fp = f;
        return m;
    }
    uint64_t* limbs(const std::vector<int>& ids) {
        uint64_t* b = buf(ids.size() * T.N);
        for (size_t i = 0; i < ids.size() * T.N; ++i) b[i] = below(ids[i / T.N]);
        return b;
    }
    // limbs as a transform's first pass leaves them
    uint64_t* passed(const std::vector<int>& ids) {
        uint64_t* b = limbs(ids);
        for (size_t i = 0; i < ids.size() * T.N; ++i)
            if (is_fp(T, ids[i / T.N])) b[i] = FpArith::pack((double)b[i]);
        return b;
    }
    Set(int logN, int L, int dnum, int K) {
        std::memset(&T, 0, sizeof(T));
        T.logN = logN, T.N = 1 << logN, T.L = L, T.K = K, T.dnum = dnum, T.np = L + 1 + K;
        T.alpha = (L + dnum) / dnum;
        T.modup_one_reduce = T.moddown_one_reduce = 1;
        words.reserve(256);
        for (int i = 0; i < T.np; ++i) {  // the first prime and the special ones on 64-bit words
            const bool fp = i > 0 && i <= L;
            p.push_back((fp ? 1ull << 50 : 1ull << 60) - 2 * (rng() % 1000) - 1);
            const int n = fp ? 50 : 60;
            primes.push_back(PrimeInfo{p[i], (uint64_t)(((unsigned __int128)1 << (n + 63)) / p[i]), (uint32_t)n, fp,
                                       2 * p[i], (double)p[i], 1.0 / (double)p[i]});
            T.fpmask[i >> 6] |= (uint64_t)fp << (i & 63);
        }
        T.primes = primes.data();
        const size_t N = T.N, q = L + 1;
        T.tw_fwd = consts(T.np * N, [=](size_t i) { return (int)(i / N); });
        T.tw_inv = consts(T.np * N, [=](size_t i) { return (int)(i / N); });
        T.twd_fwd = doubles(N), T.twd_inv = doubles(N);
        T.iscale_plain = consts(2 * T.np, [](size_t i) { return (int)(i / 2); });
        T.iscale_modup = consts(2 * q * q, [=](size_t i) { return (int)(i / 2 % q); });
        T.iscale_moddown = consts(2 * K, [=](size_t i) { return (int)(q + i / 2); });
        T.modup_mat = matrix((size_t)dnum * T.alpha, conv_bound(T.alpha), &T.modup_fp);
        T.moddown_mat = matrix(1, conv_bound(K), &T.moddown_fp);
        T.pinv = consts(T.np, [](size_t i) { return (int)i; });
        T.pmodq = consts(T.np, [](size_t i) { return (int)i; });
        T.qlinv = consts(q * q, [=](size_t i) { return (int)(i % q); });
        uint64_t* m = buf(q * q);
        for (size_t i = 0; i < q * q; ++i) m[i] = below((int)(i % q));
        T.qlmodq = m;
    }
};

template <class Jobs, class J>
Jobs one(const J& j) {
    Jobs l;
    std::memset(&l, 0, sizeof(l));
    l.inl[0] = j;
    l.n = 1;
    return l;
}

// Runs launch in both orders and compares what it leaves in out.
int bad = 0;
void check(const char* name, Set& S, uint64_t* out, size_t n, const std::function<hipError_t()>& launch) {
    std::vector<uint64_t> got[2];
    for (int k = 0; k < 2; ++k) {
        descending = k;
        std::fill(out, out + n, 0);
        if (launch() != hipSuccess) std::exit(2);
        got[k].assign(out, out + n);
    }
    size_t diff = 0, set = 0;
    for (size_t i = 0; i < n; ++i) diff += got[0][i] != got[1][i], set += got[0][i] != 0;
    const bool ok = !diff && set > n / 2;
    bad += !ok;
    std::printf("logN %d %-24s %s (%zu of %zu words differ)\n", S.T.logN, name, ok ? "ok" : "WRONG", diff, n);
    std::fflush(stdout);
}

void run(int logN) {
    const int L = 3, K = 2, nl = L + 1;
    Set S(logN, L, 2, K);
    const DevTables& T = S.T;
    const size_t N = T.N;
    std::vector<int> q, pq, sp, top;
    for (int i = 0; i < nl; ++i) q.push_back(i);
    for (int i = 0; i < K; ++i) sp.push_back(nl + i);
    pq = q;
    pq.insert(pq.end(), sp.begin(), sp.end());
    std::vector<int> digits = pq;
    digits.insert(digits.end(), pq.begin(), pq.end());
    top = {L};
    top.insert(top.end(), sp.begin(), sp.end());

    uint64_t* out = S.buf(4 * (nl + K) * N);
    {
        TensorJob j{S.limbs(q), S.limbs(q), S.limbs(q), S.limbs(q), out, out + nl * N, out + 2 * nl * N, nl, 0,
                    out + 3 * nl * N};
        check("tensor", S, out, 4 * nl * N, [&] { return launch_tensor_rows(T, one<TensorJobs>(j), nl, nullptr); });
    }
    {
        ModUpJob j{fused_inv_cols(T) ? S.passed(q) : S.limbs(q), out, L};
        // a digit's own positions stay unwritten
        check("modup", S, out, 2 * (nl + K) * N, [&] { return launch_modup_cols(T, one<ModUpJobs>(j), 2, nl, nullptr); });
    }
    const uint64_t* key[2] = {S.limbs(digits), S.limbs(digits)};
    const uint64_t* add[2] = {S.limbs(q), S.limbs(q)};
    const uint64_t* own = S.limbs(q);
    uint64_t* ext = S.passed(digits);
    uint64_t* down = out + 2 * (nl + K) * N;
    KskJob k{};
    k.ext = ext, k.own = own, k.ka = key[0], k.kb = key[1], k.level = L;
    k.acc_a = out, k.acc_b = out + (nl + K) * N;
    check("inner product", S, out, 2 * (nl + K) * N, [&] { return launch_rows_ksk(T, one<KskJobs>(k), nl + K, nullptr); });
    k.down_a = down, k.down_b = down + (K + 1) * N, k.add_a = add[0], k.add_b = add[1];
    check("inner product, down", S, out, (2 * (nl + K) + 2 * (K + 1)) * N,
          [&] { return launch_rows_ksk(T, one<KskJobs>(k), nl + K, nullptr); });
    KskJob r{};
    r.ext = ext, r.own = own, r.ka = key[0], r.kb = key[1], r.level = L;
    r.rot_a = out, r.rot_b = out + (nl + K) * N, r.base_a = S.limbs(pq), r.add0 = add[0], r.scale_p = 1;
    r.rot_down = down, r.autok = 5;
    check("inner product, rotated", S, out, (2 * (nl + K) + K) * N,
          [&] { return launch_rows_ksk(T, one<KskJobs>(r), nl + K, nullptr, false, true); });
    {
        uint64_t* t = fused_inv_cols(T) ? S.passed(top) : S.limbs(top);
        ModDownJob j{t + N, out, nullptr, nullptr, L, 0};
        check("moddown", S, out, nl * N, [&] { return launch_moddown_cols(T, one<ModDownJobs>(j), nl, false, nullptr); });
        j.top_acc = t;
        check("moddown, rescale", S, out, (nl - 1) * N,
              [&] { return launch_moddown_cols(T, one<ModDownJobs>(j), nl, true, nullptr); });
    }
    {
        RescaleJob j{S.limbs(q), S.limbs(q), out + (nl - 1) * N, out, L, 0};
        check("rescale", S, out, nl * N, [&] { return launch_rescale_cols(T, one<RescaleJobs>(j), L, nullptr); });
    }
}

}  // namespace

void host_wave_wait() { wait(WAVE); }
void host_block_wait() { wait(BLOCK); }

template <class... P, class... A>
void host_launch(void (*kernel)(P...), dim3 grid, dim3 block, int, hipStream_t, A... args) {
    blockDim = block;
    gridDim = grid;
    body = [&] { kernel(args...); };
    for (unsigned b = 0; b < grid.x; ++b) {
        blockIdx = dim3(b, 0, 0);
        run_block((int)block.x);
    }
}

int main() {
    run(12);
    run(15);
    return bad ? 1 : 0;
}
