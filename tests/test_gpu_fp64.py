"""The FP64 transforms of primes below 2^50 against the oracle's integer ones
(needs a GPU), bit-exact: prime sizes on both sides of the rule's line (50 and
51 bits), the smallest and largest rings, values at the ends of the range
(all 0, all p - 1, alternating), and products whose special primes are on
either side too."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.gpu_util import log, make_env, to_dev

pytestmark = pytest.mark.gpu


def _extremes(p, N, rng):
    top = np.full(N, p - 1, dtype=np.uint64)
    alt = np.where(np.arange(N) % 2 == 0, np.uint64(0), np.uint64(p - 1)).astype(np.uint64)
    one = np.zeros(N, dtype=np.uint64)
    one[0] = 1
    return [np.zeros(N, dtype=np.uint64), top, alt, one, rng.integers(0, p, N, dtype=np.uint64)]


@pytest.mark.parametrize("bits", [25, 40, 50, 51, 59])
@pytest.mark.parametrize("logN", [10, 11, 15, 16, 17])
def test_transforms_at_the_ends_of_the_range(logN, bits):
    L = 2 if logN < 17 else 1
    P = O.make_params(logN, 60, bits, L, 60, 1, K=1)
    o, ctx, _ = make_env(P, relin=False)
    rng = np.random.default_rng(logN * 64 + bits)
    log(f"transforms logN={logN} bits={bits}")
    cases = [_extremes(int(P.moduli[i]), P.N, rng) for i in range(L + 1)]
    for k in range(5):
        x = np.ascontiguousarray(np.stack([cases[i][k] for i in range(L + 1)]))
        ids = list(range(L + 1))
        for inverse in (False, True):
            d = to_dev(ctx, x)
            ctx.ntt(d, L + 1, 0, inverse)
            ctx.synchronize()
            assert np.array_equal(d.numpy(), o.ntt(x.copy(), ids, inverse=inverse)), (k, inverse)
    ctx.close()


@pytest.mark.parametrize("first,bits,special", [(50, 50, 50), (50, 40, 60), (60, 51, 50), (51, 50, 51), (60, 25, 45)])
@pytest.mark.parametrize("logN", [12, 15])
def test_products_of_mixed_prime_sizes(logN, first, bits, special):
    """Product, rescale and rotation at every level: primes of both kinds meet
    in the conversions, the centered lift of rescaling and the inner products."""
    L = 4
    P = O.make_params(logN, first, bits, L, special, 2)
    o, ctx, keys = make_env(P, rotations=(1,))
    for level in (L, 2, 1):
        log(f"mixed sizes logN={logN} {first}/{bits}/{special} level={level}")
        a = (o.random_poly(level + 1, 3), o.random_poly(level + 1, 4))
        b = (o.random_poly(level + 1, 5), o.random_poly(level + 1, 6))
        ga, gb = ctx.load(*a, noise=2.0 ** bits), ctx.load(*b, noise=2.0 ** bits)
        want = o.mult(a, b, keys["relin"])
        got = ga.mult(gb).store()
        assert all(np.array_equal(x, y) for x, y in zip(got, want)), "product"
        got = ga.mult(gb, rescale=True).store()
        assert all(np.array_equal(x, y) for x, y in zip(got, o.rescale(want))), "product and rescale"
        got = ga.mult(gb).rescale().store()
        assert all(np.array_equal(x, y) for x, y in zip(got, o.rescale(want))), "product, then rescale"
        got = ga.rotate(1).store()
        assert all(np.array_equal(x, y) for x, y in zip(got, o.rotate(a, 1, keys[1]))), "rotation"
    ctx.close()
