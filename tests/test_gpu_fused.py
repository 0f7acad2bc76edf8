"""The fused key switch against the oracle (needs a GPU), bit-exact: every
digit size and special-prime count it is built for and the first ones past
its line (which take the separate kernels), every ring size, and levels whose
last digit is ragged, whole or alone."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.gpu_util import log, make_env

pytestmark = pytest.mark.gpu

# (logN, L, dnum, K): digit size alpha = ceil((L + 1) / dnum)
SHAPES = [(12, 3, 4, 1), (12, 3, 2, 2), (12, 5, 2, 3), (12, 7, 2, 4), (12, 9, 2, 5), (12, 5, 1, 6), (12, 6, 1, 7),
          (12, 7, 1, 8), (12, 8, 1, 9), (12, 9, 1, 10), (13, 8, 3, 3), (14, 6, 4, 2), (15, 5, 3, 2), (16, 4, 2, 3),
          (12, 10, 1, 11), (12, 4, 5, 1), (11, 3, 2, 2), (17, 2, 3, 1)]


@pytest.mark.parametrize("logN,L,dnum,K", SHAPES)
def test_shapes(logN, L, dnum, K):
    P = O.make_params(logN, 60, 50, L, 60, dnum, K=K)
    o, ctx, keys = make_env(P, rotations=(3,))
    alpha = -(-(L + 1) // dnum)
    for level in sorted({1, alpha - 1, min(L, alpha), L - 1, L} - {0}):
        log(f"fused key switch logN={logN} L={L} dnum={dnum} K={K} level={level}")
        a = (o.random_poly(level + 1, 11), o.random_poly(level + 1, 12))
        b = (o.random_poly(level + 1, 13), o.random_poly(level + 1, 14))
        ga, gb = ctx.load(*a, noise=2.0 ** 50), ctx.load(*b, noise=2.0 ** 50)
        want = o.mult(a, b, keys["relin"])
        for rescale, ref in ((False, want), (True, o.rescale(want))):
            got = ga.mult(gb, rescale=rescale).store()
            assert all(np.array_equal(x, y) for x, y in zip(got, ref)), ("product", rescale)
        got = ga.rotate(3).store()
        assert all(np.array_equal(x, y) for x, y in zip(got, o.rotate(a, 3, keys[3]))), "rotation"
    ctx.close()
