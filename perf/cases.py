"""The work a user of the engine has it do, as cases that can be timed.

Every case runs one call (or the few calls that belong together) of the public
Python surface on ciphertexts that are already on the GPU, at one parameter
set: ring size 2^logN, L scaling primes of `bits` bits (a 60-bit first prime
and 60-bit special primes), dnum key-switching digits.  Residues and keys are
uniform below their primes, as they are in any real ciphertext or key.

A program keeps one context per parameter set with its keys, its transform's
diagonals and its bootstrapping plan, and runs many ciphertexts through it;
`prepare` does the same: contexts, keys and plans are made once and shared,
the ciphertexts, plaintext vectors and polynomials come from the seed.
"""
import math
import random

import numpy as np
import torch

import pyfideslib_amd as F
from pyfideslib_amd import bootstrap as B
from pyfideslib_amd import params as PP

_RANGES = {"logN": (12, 16), "bits": (40, 50, 59)}
_MOST_OUT = 32  # ciphertexts one call of a batch or a rotation set returns


def listed():
    small = {"logN": 13, "L": 3, "bits": 40, "dnum": 2}
    top = {"logN": 16, "L": 24, "bits": 50, "dnum": 3}
    return [
        # the smallest parameter set: a single product, where launches and latency count
        dict(small, name="mult_n13", kind="mult", level=3),
        # a rotation at a middling ring size, one level below the top
        dict(logN=14, L=8, bits=50, dnum=3, name="rotate_n14", kind="rotate", level=7, step=3),
        # products with wide scaling primes (the usual choice where precision matters)
        dict(logN=15, L=11, bits=59, dnum=3, name="mult_n15_59", kind="mult", level=11),
        # forward and inverse transform of one full polynomial: the stage everything is made of
        dict(top, name="ntt_n16", kind="ntt", limbs=25),
        # the benchmark's headline call: a product at the top of the chain
        dict(top, name="mult_n16_top", kind="mult", level=24),
        # the same call deep in a circuit, where few limbs are left
        dict(top, name="mult_n16_low", kind="mult", level=5),
        # an affine layer on one ciphertext: weights times input, rescaled, plus a bias ciphertext
        dict(top, name="plain_n16", kind="plain", level=24),
        # the same with weights that arrive as numbers: encoded, then multiplied
        dict(top, name="encode_n16", kind="encode", level=23),
        # rotations of one ciphertext that share their decomposition (sums over windows)
        dict(top, name="hoisted_n16", kind="hoisted", level=17, count=9),
        # what a serving loop collects: independent products at whatever levels they are
        dict(top, name="batch_n16", kind="batch", op="mult", level=24, count=24),
        # a 64-diagonal matrix-vector product in the extended basis (a dense layer, a bootstrapping stage)
        dict(top, name="transform_n16", kind="transform", level=24, count=64, bstep=8),
        # a whole bootstrap: the largest single call
        dict(top, name="bootstrap_n16", kind="bootstrap", level=0),
    ]


def draw(rng):
    """One more case of the same ranges; a bootstrap is the largest call, so none is drawn."""
    kind = rng.choice(["ntt", "mult", "mult", "rotate", "plain", "encode", "hoisted", "batch", "batch", "transform",
                       "series"])
    logN = rng.randint(*_RANGES["logN"])
    c = {"logN": logN, "L": rng.randint(3, min(24, 3 + (1 << (logN - 12)) * 3)),
         "bits": rng.choice(_RANGES["bits"]), "dnum": rng.randint(2, 4), "kind": kind}
    if kind == "series":
        c.update(L=rng.randint(9, 16), bits=rng.choice((40, 50)), count=rng.randint(5, 31))
    L = c["L"]
    c["level"] = rng.randint(max(1, L - 3), L) if kind == "series" else rng.randint(1, L)
    if kind == "ntt":
        c["limbs"] = rng.randint(1, L + 1)
    elif kind == "rotate":
        c["step"] = rng.choice((1, -1)) * rng.randint(1, (1 << (logN - 1)) - 1)
    elif kind == "hoisted":
        c["count"] = rng.randint(2, 14)
    elif kind == "batch":
        c.update(op=rng.choice(("mult", "rotate")), count=int(round(math.exp(rng.uniform(math.log(2), math.log(32))))))
    elif kind == "transform":
        c["count"] = rng.randint(5, 40)
        c["bstep"] = 1 << rng.randint(1, 3)
    return c


# ------------------------------------------------------- parameters, inputs ----
_params, _handles = {}, {}


def _raw(case):
    k = (case["logN"], case["bits"], case["L"], case["dnum"])
    if k not in _params:
        _params[k] = PP.ckks_params(k[0], 60, k[1], k[2], 60, k[3])
    return k, _params[k]


def _uniform(moduli, N, seed):
    """[len(moduli), N] residues on the GPU, limb i below moduli[i]."""
    g = torch.Generator(device="cuda").manual_seed(seed & 0x7FFFFFFFFFFF)
    return torch.stack([torch.randint(0, int(p), (N,), dtype=torch.int64, device="cuda", generator=g) for p in moduli])


def _host(t):
    return t.cpu().numpy().view(np.uint64)


def _key(raw, index):
    mods = list(raw.moduli) + list(raw.special_moduli)
    t = _uniform(mods * (2 * raw.dnum), raw.N, 7_000_003 * (index + 1)).view(2, raw.dnum, len(mods), raw.N)
    return _host(t[0]), _host(t[1])


class _Handle:
    """One parameter set's context with what a program keeps in it."""

    def __init__(self, raw):
        self.raw, self.ctx, self.keys, self.plans = raw, F.Context(raw), set(), {}

    def need(self, relin=False, rotations=()):
        if relin and "relin" not in self.keys:
            self.ctx.load_eval_key(_key(self.raw, 0))
            self.keys.add("relin")
        half = self.raw.N // 2
        for r in rotations:
            if r % half and r not in self.keys:
                self.ctx.load_rotation_key(r, _key(self.raw, 1 + r % half))
                self.keys.add(r)

    def diagonals(self, level, count):
        k = ("diagonals", level, count)
        if k not in self.plans:
            mods = list(self.raw.moduli[: level + 1]) + list(self.raw.special_moduli)
            self.plans[k] = [self.ctx.plaintext_ext(_host(_uniform(mods, self.raw.N, 900_001 + i)),
                                                    noise=2.0 ** 50) for i in range(count)]
        return self.plans[k]

    def bootstrapper(self):
        if "bootstrap" not in self.plans:
            bs = B.Bootstrapper(self.ctx, 2.0 ** 50, level_budget=(3, 3), K=28, double_angle=3, degree=119,
                                sparse_encaps=True)
            self.need(relin=True, rotations=bs.rotations)
            self.ctx.load_switch_key(F.SSE_DENSE_TO_SPARSE, _key(self.raw, 100_001))
            self.ctx.load_switch_key(F.SSE_SPARSE_TO_DENSE, _key(self.raw, 100_002))
            self.ctx.load_automorph_key(2 * self.raw.N - 1, _key(self.raw, 100_003))
            self.plans["bootstrap"] = bs
        return self.plans["bootstrap"]


def _handle(case):
    k, raw = _raw(case)
    if k not in _handles:
        _handles[k] = _Handle(raw)
    return _handles[k]


def _parts(raw, seed, i, level):
    """(c0, c1) of input ciphertext i: limbs 0..level on the GPU."""
    mods = raw.moduli[: level + 1]
    return _uniform(mods, raw.N, seed * 4099 + 2 * i + 1), _uniform(mods, raw.N, seed * 4099 + 2 * i + 2)


def _load(h, case, seed, i, level):
    c0, c1 = _parts(h.raw, seed, i, level)
    torch.cuda.synchronize()
    ct = h.ctx.ciphertext()
    F._check(F.lib().fides_ct_load_device(h.ctx.h, ct.h, c0.data_ptr(), c1.data_ptr(), level + 1,
                                          2.0 ** case["bits"], 1, h.raw.N // 2))
    h.ctx.synchronize()
    return ct


def _steps(case):
    """Rotation steps of a hoisted set: 1, 2, 3, ... with the powers of two a rotate-and-sum uses."""
    return [i + 1 if i < 4 else 1 << (i - 1) for i in range(case["count"])][: max(1, case["logN"] - 1)]


def _batch(case):
    """(level, rotation step) of each member of a batch."""
    r = random.Random(case["count"] * 1009 + case["level"])
    lo = min(case["level"], 4)
    return [(r.randint(lo, case["level"]), 1 << r.randint(0, 4)) for _ in range(case["count"])]


def _slots(case, seed):
    return np.random.default_rng(seed).uniform(-1.0, 1.0, 1 << (case["logN"] - 1))


def _coeffs(case):
    n = case["count"] + 1
    return [float(v) for v in np.random.default_rng(n).normal(0, 1, n) / (np.arange(n) + 1.0) ** 2]


def prepare(case, seed):
    h = _handle(case)
    raw, ctx, kind, lv = h.raw, h.ctx, case["kind"], case["level"] if "level" in case else 0
    s = {"case": case, "h": h, "views": {}}
    if kind == "ntt":
        s["polys"] = [_uniform(raw.moduli[: case["limbs"]], raw.N, seed * 4099 + i) for i in (1, 2)]
    elif kind in ("mult", "batch") and case.get("op", "mult") == "mult":
        h.need(relin=True)
        levels = [lv] if kind == "mult" else [max(1, x) for x, _ in _batch(case)]
        s["a"] = [_load(h, case, seed, 2 * i, x) for i, x in enumerate(levels)]
        s["b"] = [_load(h, case, seed, 2 * i + 1, x) for i, x in enumerate(levels)]
        s["out"] = [ctx.ciphertext() for _ in levels]
    elif kind == "rotate":
        h.need(rotations=[case["step"]])
        s["a"], s["out"] = [_load(h, case, seed, 0, lv)], [ctx.ciphertext()]
    elif kind == "batch":
        members = _batch(case)
        s["steps"] = [r for _, r in members]
        h.need(rotations=s["steps"])
        s["a"] = [_load(h, case, seed, i, x) for i, (x, _) in enumerate(members)]
        s["out"] = [ctx.ciphertext() for _ in members]
    elif kind == "hoisted":
        h.need(rotations=_steps(case))
        s["a"], s["out"] = [_load(h, case, seed, 0, lv)], [ctx.ciphertext() for _ in _steps(case)]
    elif kind in ("plain", "encode"):
        s["a"], s["b"] = [_load(h, case, seed, 0, lv)], [_load(h, case, seed, 1, lv - 1)]
        s["out"] = [ctx.ciphertext()]
        s["z"] = _slots(case, seed)
        if kind == "plain":
            w = _uniform(raw.moduli[: lv + 1], raw.N, seed * 4099 + 900)
            s["w"] = ctx.plaintext(_host(w), noise=2.0 ** case["bits"])
    elif kind == "transform":
        n, b = case["count"], case["bstep"]
        h.need(rotations=list(range(1, b)) + [b])
        s["diag"] = h.diagonals(lv, n)
        s["a"], s["out"] = [_load(h, case, seed, 0, lv)], [ctx.ciphertext()]
    elif kind == "series":
        h.need(relin=True)
        s["a"], s["out"] = [_load(h, case, seed, 0, lv)], [ctx.ciphertext()]
        s["coeffs"] = _coeffs(case)
    elif kind == "bootstrap":
        s["bs"] = h.bootstrapper()
        s["a"], s["out"] = [_load(h, case, seed, 0, lv)], [ctx.ciphertext()]
    else:
        raise ValueError(kind)
    torch.cuda.synchronize()
    return s


class _Mem:
    """Both parts of a device-resident ciphertext, for torch.as_tensor (no copy)."""

    def __init__(self, p0, p1, limbs, N):
        self.__cuda_array_interface__ = {"shape": (2, limbs, N), "strides": (p1 - p0, 8 * N, 8), "typestr": "<i8",
                                         "data": (p0, False), "version": 2}


def _view(s, ct):
    key = ct.device_ptrs() + (ct.level,)
    if key not in s["views"]:
        s["views"][key] = torch.as_tensor(_Mem(*key[:2], key[2] + 1, s["h"].raw.N), device="cuda")
    return s["views"][key]


def run(s):
    case, ctx = s["case"], s["h"].ctx
    kind = case["kind"]
    if kind == "ntt":
        x, y = s["polys"]
        ctx.ntt(x.data_ptr(), case["limbs"])
        ctx.ntt(y.data_ptr(), case["limbs"], inverse=True)
        return [x, y]
    a, out = s["a"], s["out"]
    if kind == "mult":
        a[0].mult(s["b"][0], rescale=True, out=out[0])
    elif kind == "rotate":
        a[0].rotate(case["step"], out=out[0])
    elif kind == "hoisted":
        a[0].rotate_hoisted(_steps(case), out)
    elif kind == "batch" and case["op"] == "mult":
        ctx.mult_batch(a, s["b"], out, rescale=True)
    elif kind == "batch":
        ctx.rotate_batch(a, s["steps"], out)
    elif kind in ("plain", "encode"):
        w = s["w"] if kind == "plain" else ctx.encode(s["z"], case["level"], 2.0 ** case["bits"])
        a[0].mult_plain(w, rescale=True, out=out[0])
        out[0].add(s["b"][0], out=out[0])
    elif kind == "transform":
        a[0].linear_transform(s["diag"], case["bstep"], out=out[0])
    elif kind == "series":
        a[0].chebyshev_series(s["coeffs"], out=out[0])
    elif kind == "bootstrap":
        s["bs"].bootstrap(a[0], out=out[0])
    return [_view(s, o) for o in out]


# ------------------------------------------------------------------- work ----
def work(case):
    """Bytes: inputs, keys and plaintexts read once, outputs written once.  Operations: two per modular
    product and per butterfly sum, from the transforms, conversions and inner products a call is made of."""
    _, raw = _raw(case)
    N, K, dnum = raw.N, raw.K, raw.dnum
    alpha = -(-(raw.L + 1) // dnum)
    poly = lambda n: 8 * N * n  # noqa: E731
    ntt = lambda n: 4 * n * N // 2 * case["logN"]  # noqa: E731
    lv = case.get("level", 0)
    nd = lambda l: min(dnum, -(-(l + 1) // alpha))  # noqa: E731
    key = lambda l: poly(2 * nd(l) * (l + 1 + K))  # noqa: E731

    def keyswitch(l, rescale=False):
        nl, d = l + 1, nd(l)
        limbs = nl + d * (nl + K) - nl + 2 * K + 2 * nl + (4 if rescale else 0)
        conv = sum(min(alpha, nl - i * alpha) * (nl + K - min(alpha, nl - i * alpha)) for i in range(d)) + 2 * K * nl
        return ntt(limbs) + 2 * N * (conv + 2 * d * (nl + K))

    kind = case["kind"]
    if kind == "ntt":
        return {"bytes": 4 * poly(case["limbs"]), "flops": 2 * ntt(case["limbs"])}
    if kind == "mult" or (kind == "batch" and case["op"] == "mult"):
        levels = [lv] if kind == "mult" else [max(1, x) for x, _ in _batch(case)]
        by = sum(poly(4 * (x + 1) + 2 * x) for x in levels) + key(max(levels))
        return {"bytes": by, "flops": sum(keyswitch(x, True) + 8 * N * (x + 1) for x in levels)}
    if kind in ("rotate", "batch"):
        members = [(lv, case["step"])] if kind == "rotate" else _batch(case)
        by = sum(poly(4 * (x + 1)) for x, _ in members) + len({r for _, r in members}) * key(max(x for x, _ in members))
        return {"bytes": by, "flops": sum(keyswitch(x) for x, _ in members)}
    if kind in ("plain", "encode"):
        by = poly(2 * (lv + 1) + 4 * lv) + (poly(lv + 1) if kind == "plain" else 4 * N)
        return {"bytes": by, "flops": ntt(2 + 2 * lv) + 8 * N * (lv + 1)}
    n = {"hoisted": len(_steps(case)) if kind == "hoisted" else 0}.get(kind, case.get("count", 0))
    if kind == "hoisted":
        return {"bytes": poly(2 * (lv + 1) * (n + 1)) + n * key(lv), "flops": n * keyswitch(lv) // 2}
    if kind == "transform":
        b = case["bstep"]
        g = -(-n // b)
        by = poly(4 * (lv + 1) + n * (lv + 1 + K)) + min(b, n) * key(lv)
        return {"bytes": by, "flops": (g + b) * keyswitch(lv) // 2 + 4 * N * n * (lv + 1 + K)}
    if kind == "series":
        m = 2 * math.ceil(math.sqrt(n))
        return {"bytes": poly(4 * lv) + key(lv), "flops": m * keyswitch(max(1, lv - 2), True)}
    return {"bytes": 30 * key(raw.L // 2) + 158 * poly(raw.L // 2 + K),
            "flops": 90 * keyswitch(raw.L // 2, True)}


# ------------------------------------------------------------------ exact ----
def _mul(a, b, p):
    """a * b mod p for uint64 arrays below p < 2^62: the quotient in 64-bit-mantissa floats, one correction."""
    p = np.uint64(p)
    q = (a.astype(np.longdouble) * np.asarray(b, dtype=np.uint64).astype(np.longdouble) / np.longdouble(p)).astype(np.uint64)
    with np.errstate(over="ignore"):
        r = (a * np.asarray(b, dtype=np.uint64) - q * p).view(np.int64)
    r = np.where(r < 0, r + np.int64(p), r)
    return np.where(r >= np.int64(p), r - np.int64(p), r).view(np.uint64)


def _add(a, b, p):
    s = a + b
    return np.where(s >= np.uint64(p), s - np.uint64(p), s)


def _sub(a, b, p):
    return np.where(a >= b, a - b, a + np.uint64(p) - b)


def _twiddles(p, root, N):
    bits = N.bit_length() - 1
    w, x = np.empty(N, dtype=np.uint64), 1
    for i in range(N):
        w[int(format(i, "0%db" % bits)[::-1], 2)] = x
        x = x * root % p
    return w


def _ntt(x, p, root, inverse=False):
    """Negacyclic transform: value j of the output is x(root^(2 brev(j) + 1))."""
    N = len(x)
    w = _twiddles(p, pow(root, -1, p) if inverse else root, N)
    v, m = x.copy(), 1
    if not inverse:
        while m < N:
            v = v.reshape(m, 2, -1)
            t = _mul(v[:, 1], w[m: 2 * m, None], p)
            v = np.stack([_add(v[:, 0], t, p), _sub(v[:, 0], t, p)], axis=1)
            m *= 2
        return v.reshape(N)
    m = N // 2
    while m:
        v = v.reshape(m, 2, -1)
        v = np.stack([_add(v[:, 0], v[:, 1], p), _mul(_sub(v[:, 0], v[:, 1], p), w[m: 2 * m, None], p)], axis=1)
        m //= 2
    return _mul(v.reshape(N), pow(N, -1, p), p)


def _convert(limbs, primes, p):
    """sum_i [x_i (D / q_i)^-1]_(q_i) (D / q_i) mod p, the fast base conversion."""
    D = math.prod(primes)
    y = np.zeros(len(limbs[0]), dtype=np.uint64)
    for x, q in zip(limbs, primes):
        t = _mul(x, pow(D // q, -1, q), q)
        y = _add(y, _mul(t % np.uint64(p), D // q % p, p), p)
    return y


def _keyswitch(raw, x, key):
    """(b, a) parts of the key switch of x (evaluation form): hybrid decomposition, inner product, ModDown."""
    nl, K = len(x), raw.K
    Q, P = [int(q) for q in raw.moduli], [int(p) for p in raw.special_moduli]
    primes = Q[:nl] + P
    roots = list(raw.root_of_unity[:nl]) + list(raw.special_root_of_unity)
    ids = list(range(nl)) + [raw.L + 1 + k for k in range(K)]
    alpha = -(-(raw.L + 1) // raw.dnum)
    coef = [_ntt(x[i], Q[i], raw.root_of_unity[i], True) for i in range(nl)]
    acc = [[np.zeros(raw.N, dtype=np.uint64) for _ in primes] for _ in range(2)]
    for d in range(-(-nl // alpha)):
        own = range(d * alpha, min(nl, (d + 1) * alpha))
        for j, p in enumerate(primes):
            v = x[j] if j in own else _ntt(_convert([coef[i] for i in own], [Q[i] for i in own], p), p, roots[j])
            for h in range(2):
                acc[h][j] = _add(acc[h][j], _mul(v, key[1 - h][d, ids[j]], p), p)
    out, Pp = [], math.prod(P)
    for h in range(2):
        sp = [_ntt(acc[h][nl + k], P[k], roots[nl + k], True) for k in range(K)]
        out.append([_mul(_sub(acc[h][i], _ntt(_convert(sp, P, Q[i]), Q[i], roots[i]), Q[i]), pow(Pp, -1, Q[i]), Q[i])
                    for i in range(nl)])
    return out


def _rescale(raw, c):
    l = len(c) - 1
    ql = int(raw.moduli[l])
    top = _ntt(c[l], ql, raw.root_of_unity[l], True)
    out = []
    for i in range(l):
        q = int(raw.moduli[i])
        lift = top % np.uint64(q)
        lift = np.where(top > np.uint64(ql >> 1), _sub(lift, np.full_like(lift, ql % q), q), lift)
        out.append(_mul(_sub(c[i], _ntt(lift, q, raw.root_of_unity[i]), q), pow(ql, -1, q), q))
    return out


def _stacked(parts):
    return [np.stack([np.stack(c) for c in parts]).view(np.int64)]


def exact(case, seed):
    """The transforms, products, rotations and plaintext products, in plain numpy integers; the calls made of
    many of these are left out (they would take minutes)."""
    _, raw = _raw(case)
    kind, N, lv = case["kind"], raw.N, case.get("level", 0)
    Q = [int(q) for q in raw.moduli]
    if kind == "ntt":
        xs = [_host(_uniform(Q[: case["limbs"]], N, seed * 4099 + i)) for i in (1, 2)]
        return [np.stack([_ntt(x[i], Q[i], raw.root_of_unity[i], inv) for i in range(len(x))]).view(np.int64)
                for x, inv in zip(xs, (False, True))]
    if kind not in ("mult", "rotate", "plain"):
        return None
    if kind != "plain" and work(case)["flops"] > 4e8:  # about 15 seconds
        return None
    a = [_host(t) for t in _parts(raw, seed, 0, lv)]
    n = range(lv + 1)
    if kind == "rotate":
        kb, ka = _keyswitch(raw, a[1], _key(raw, 1 + case["step"] % (N // 2)))
        parts = [[_add(a[0][i], kb[i], Q[i]) for i in n], ka]
        k, bits = pow(5, case["step"] % (N // 2), 2 * N), case["logN"]
        rev = np.array([int(format(i, "0%db" % bits)[::-1], 2) for i in range(N)])
        src = rev[((2 * rev + 1) * k % (2 * N)) >> 1]
        return _stacked([[x[src] for x in c] for c in parts])
    if kind == "plain":
        b = [_host(t) for t in _parts(raw, seed, 1, lv - 1)]
        w = _host(_uniform(Q[: lv + 1], N, seed * 4099 + 900))
        parts = [_rescale(raw, [_mul(x[i], w[i], Q[i]) for i in n]) for x in a]
        return _stacked([[_add(x[i], y[i], Q[i]) for i in range(lv)] for x, y in zip(parts, b)])
    b = [_host(t) for t in _parts(raw, seed, 1, lv)]
    d0, d2 = ([_mul(a[h][i], b[h][i], Q[i]) for i in n] for h in (0, 1))
    d1 = [_add(_mul(a[0][i], b[1][i], Q[i]), _mul(a[1][i], b[0][i], Q[i]), Q[i]) for i in n]
    ks = _keyswitch(raw, d2, _key(raw, 0))
    return _stacked([_rescale(raw, [_add(d[i], k[i], Q[i]) for i in n]) for d, k in zip((d0, d1), ks)])
