"""Which contexts take the fused key switch, and what both sides of that line
compute (needs a GPU): counts of special primes and digit sizes up to the most
and one past it, the widths of special primes whose sums fit one reduction and
do not, per ring size.  Products, rotations, batches, hoisted sets, P*Q
rotations and giant steps are bit-exact against the oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.gpu_util import log, make_env

pytestmark = pytest.mark.gpu

# logN, L, dnum, K, bits of the scaling and of the special primes, fused
SHAPES = [
    # 8 special primes of 60 bits and 50-bit targets: the sums fit; 9 do not
    (12, 7, 1, 8, 50, 60, True), (12, 8, 1, 9, 50, 60, False), (13, 8, 1, 9, 50, 60, False),
    # of 59 and 50 bits: up to 12, past it by count
    (12, 8, 1, 9, 50, 59, True), (12, 9, 1, 10, 50, 59, True), (12, 10, 1, 11, 50, 59, True),
    (12, 11, 1, 12, 50, 59, True), (12, 12, 1, 13, 50, 59, False), (12, 11, 2, 13, 50, 50, False),
    # digits of 10, 11 and 12 limbs, of 13
    (12, 19, 2, 9, 40, 59, True), (12, 21, 2, 10, 40, 59, True), (12, 23, 2, 10, 40, 59, True),
    (12, 12, 1, 12, 40, 59, False),
    # the other rings
    (13, 10, 1, 11, 59, 59, True), (14, 8, 1, 9, 50, 59, True), (14, 9, 1, 10, 50, 59, False),
    (15, 10, 1, 11, 59, 59, True), (16, 11, 1, 12, 50, 59, True),
    # digits, rings past the line
    (12, 4, 5, 1, 50, 60, False), (11, 3, 2, 2, 50, 60, False), (17, 2, 3, 1, 50, 60, False),
]


def same(got, want):
    return all(np.array_equal(x, y) for x, y in zip(got, want))


@pytest.mark.parametrize("logN,L,dnum,K,bits,special,fused", SHAPES)
def test_line(logN, L, dnum, K, bits, special, fused):
    P = O.make_params(logN, 60, bits, L, special, dnum, K=K)
    o, ctx, keys = make_env(P, rotations=(1, 2, 3))
    assert ctx.fused == fused
    E = O.ExtBasis(o)
    for level in sorted({1, L}):
        log(f"logN={logN} L={L} dnum={dnum} K={K} {bits}/{special} level={level}")
        top = tuple(np.stack([np.full(P.N, int(P.moduli[i]) - 1, dtype=np.uint64) for i in range(level + 1)])
                    for _ in range(2))
        a = (o.random_poly(level + 1, 11), o.random_poly(level + 1, 12))
        ga, gt = ctx.load(*a, noise=2.0 ** bits), ctx.load(*top, noise=2.0 ** bits)
        want = o.mult(a, top, keys["relin"])
        full = o.mult(top, top, keys["relin"])
        assert same(ga.mult(gt, rescale=False).store(), want)
        assert same(gt.mult(gt, rescale=True).store(), o.rescale(full))
        outs = [ctx.ciphertext() for _ in range(2)]
        ctx.mult_batch([ga, gt], [gt, gt], outs, rescale=True)
        assert all(same(x.store(), o.rescale(w)) for x, w in zip(outs, (want, full))), "batch"
        rot = {r: o.rotate(a, r, keys[r]) for r in (1, 2, 3)}
        assert same(ga.rotate(3).store(), rot[3])
        assert all(same(x.store(), rot[r]) for r, x in zip((1, 2), ga.rotate_hoisted([1, 2]))), "hoisted"
        ext = [E.rotate(a[0], a[1], O.rot_index(logN, r), keys[r]) for r in (1, 2)]
        for idx in ((0,), (0, 1)):
            got = ga.rotate_hoisted([idx_ + 1 for idx_ in idx], ext=True)
            assert all(same(x.store_ext(), ext[i]) for i, x in zip(idx, got)), "P*Q rotations"
    pq = E.ids(L)
    diag = [o.random_poly(len(pq), 40 + i, primeids=pq) for i in range(6)]
    got = ga.linear_transform([ctx.plaintext_ext(d) for d in diag], 2, 1, 0)
    assert same(got.store(), E.linear_transform(a, diag, keys, 2, 1, 0, False)), "giant steps"
    ctx.close()
