"""Rescaling and products with a plaintext that are rescaled against the
oracle (needs a GPU), bit-exact: each ring size of the three-launch form and the
ones past its line, every level, dropped and staying primes of either kind, an
output that is the input and one that is not."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.gpu_util import log, make_env

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("first,bits", [(60, 50), (60, 59), (50, 25), (51, 50)])
@pytest.mark.parametrize("logN,L", [(11, 3), (12, 9), (13, 4), (14, 3), (15, 3), (16, 5), (17, 2)])
def test_rescale(logN, L, first, bits):
    P = O.make_params(logN, first, bits, L, 60, 1, K=1)
    o, ctx, _ = make_env(P, relin=False)
    for level in range(1, L + 1):
        log(f"rescale logN={logN} {first}/{bits} level={level}")
        top = np.stack([np.full(P.N, int(P.moduli[i]) - 1, dtype=np.uint64) for i in range(level + 1)])
        for a in ((top, top), (o.random_poly(level + 1, 3), o.random_poly(level + 1, 4))):
            w = o.random_poly(L + 1, 5)
            g = ctx.load(*a, noise=2.0 ** bits)
            pt = ctx.plaintext(w, noise=2.0 ** bits)
            want = o.rescale(o.mult_plain(a, w[: level + 1]))
            got = g.mult_plain(pt, rescale=True)
            assert all(np.array_equal(x, y) for x, y in zip(got.store(), want)), "product"
            assert got.level == level - 1
            g.mult_plain(pt, rescale=True, out=g)
            assert all(np.array_equal(x, y) for x, y in zip(g.store(), want)), "product in place"
            h = ctx.load(*a, noise=2.0 ** bits).mult_plain(pt, rescale=False)
            h.rescale()
            assert all(np.array_equal(x, y) for x, y in zip(h.store(), want)), "rescale"
    ctx.close()
