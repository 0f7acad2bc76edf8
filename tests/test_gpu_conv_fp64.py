"""Conversions into primes on the FP64 units against the oracle (needs a GPU),
bit-exact: the most source limbs with the widest and the narrowest primes on
either side, and rescaling from a dropped prime of either kind."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.gpu_util import log, make_env

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("first,bits,special", [(60, 50, 60), (60, 25, 60), (50, 50, 50), (50, 25, 25), (60, 59, 50)])
@pytest.mark.parametrize("logN,L,dnum,K", [(12, 9, 1, 10), (16, 1, 1, 1), (16, 8, 1, 9), (12, 12, 1, 13), (13, 11, 1, 12),
                                           (14, 10, 1, 11), (15, 11, 1, 12), (16, 10, 1, 11)])
def test_products_and_rotations(logN, L, dnum, K, first, bits, special):
    P = O.make_params(logN, first, bits, L, special, dnum, K=K)
    o, ctx, keys = make_env(P, rotations=(1,))
    for level in {1, L}:
        log(f"conversions logN={logN} L={L} K={K} {first}/{bits}/{special} level={level}")
        top = [np.stack([np.full(P.N, int(P.moduli[i]) - 1, dtype=np.uint64) for i in range(level + 1)])] * 2
        for a in (top, (o.random_poly(level + 1, 3), o.random_poly(level + 1, 4))):
            b = (o.random_poly(level + 1, 5), o.random_poly(level + 1, 6))
            ga, gb = ctx.load(*a, noise=2.0 ** bits), ctx.load(*b, noise=2.0 ** bits)
            want = o.mult(a, b, keys["relin"])
            for rescale, ref in ((False, want), (True, o.rescale(want))):
                got = ga.mult(gb, rescale=rescale).store()
                assert all(np.array_equal(x, y) for x, y in zip(got, ref)), ("product", rescale)
            got = ga.rotate(1).store()
            assert all(np.array_equal(x, y) for x, y in zip(got, o.rotate(a, 1, keys[1]))), "rotation"
    ctx.close()
