"""Rotations that leave the key switch in P*Q against the oracle's extended
basis (needs a GPU), bit-exact: each ring size that rotates inside the key
switch and the ones past its line, one key and several over one source, and
transforms whose giant steps hand their special limbs on."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.gpu_util import log, make_env

pytestmark = pytest.mark.gpu

# (logN, L, dnum, K), as in the key switch's tests
SHAPES = [(11, 3, 2, 2), (12, 3, 4, 1), (12, 4, 5, 1), (12, 9, 1, 10), (13, 5, 3, 2), (14, 4, 2, 3), (15, 4, 2, 3),
          (16, 3, 2, 2), (17, 2, 3, 1)]


def same(got, want):
    return all(np.array_equal(x, y) for x, y in zip(got, want))


@pytest.mark.parametrize("logN,L,dnum,K", SHAPES)
def test_hoisted(logN, L, dnum, K):
    P = O.make_params(logN, 60, 50, L, 60, dnum, K=K)
    N2 = P.N // 2
    rots = (1, 3, N2 - 5)
    o, ctx, keys = make_env(P, relin=False, rotations=rots)
    E = O.ExtBasis(o)
    for level in (1, L):
        a = (o.random_poly(level + 1, 21), o.random_poly(level + 1, 22))
        ga = ctx.load(*a, noise=2.0 ** 50)
        want = [E.rotate(a[0], a[1], O.rot_index(logN, r), keys[r]) for r in rots]
        for idx in ((0,), (1,), (2, 0, 1)):
            log(f"hoisted P*Q rotations logN={logN} L={L} dnum={dnum} K={K} level={level} set {idx}")
            outs = ga.rotate_hoisted([rots[i] for i in idx], ext=True)
            assert all(same(x.store_ext(), want[i]) for i, x in zip(idx, outs)), idx
    ctx.close()


@pytest.mark.parametrize("logN,L,dnum,K", [s for s in SHAPES if 12 <= s[0] <= 16])
def test_transform(logN, L, dnum, K):
    P = O.make_params(logN, 60, 50, L, 60, dnum, K=K)
    o, ctx, keys = make_env(P, relin=False, rotations=(1, 2, 4, 6, 3))
    E = O.ExtBasis(o)
    pq = E.ids(L)
    # 4 giant steps of 2 (the last ragged), then 2 of 2
    for n, offset, batched, level in ((7, 3, False, L), (7, 0, False, 1), (7, 3, True, L), (4, 3, False, L),
                                      (4, 0, True, 1)):
        log(f"transform logN={logN} L={L} dnum={dnum} K={K} diagonals {n} offset {offset} batched {batched}")
        a = (o.random_poly(level + 1, 31), o.random_poly(level + 1, 32))
        full = [o.random_poly(len(pq), 40 + i, primeids=pq) for i in range(n)]
        cut = [np.ascontiguousarray(np.concatenate([d[:level + 1], d[L + 1:]])) for d in full]
        want = E.linear_transform(a, cut, keys, 2, 1, offset, batched)
        got = ctx.load(*a, noise=2.0 ** 50).linear_transform([ctx.plaintext_ext(d) for d in full], 2, 1, offset,
                                                             batched_giant=batched)
        assert same(got.store(), want), (n, offset, batched)
    ctx.close()
