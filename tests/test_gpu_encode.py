"""The encoder (needs a GPU): rings whose special FFT runs on one thread and on
eight (from 2^13 on), real and complex slots, the ends of the coefficient range.

Every limb must hold the residues of one integer vector exactly, and that
vector must lie within 1 of scale * [Re w, Im w] computed in extended
precision: with |z| <= 1 and scale 2^40 the FFT's rounding, at most log2(n) 2^-52
of values up to 2^40, is below 2^-8, so only the rounding to integers counts."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.gpu_util import log, make_env

pytestmark = pytest.mark.gpu


def _coefficients(z):
    """[Re w, Im w] with w = U0^-1 z, slot j = w(zeta^(5^j)), in extended precision."""
    v = z.astype(np.clongdouble)
    n, h = len(v), len(v) // 2
    while h >= 1:
        e = np.array([pow(5, j, 8 * h) for j in range(h)], dtype=np.longdouble)
        a = 2 * np.longdouble("3.14159265358979323846264338327950288") * e / (8 * h)
        tw = np.cos(a) + 1j * np.sin(a)
        v = v.reshape(-1, 2, h)
        v = np.stack([(v[:, 0] + v[:, 1]) / 2, (v[:, 0] - v[:, 1]) / 2 / tw], axis=1).reshape(n)
        h //= 2
    bits = n.bit_length() - 1
    rev = np.array([int(format(i, f"0{bits}b")[::-1], 2) for i in range(n)])
    return np.concatenate([v[rev].real, v[rev].imag])


@pytest.mark.parametrize("logN,level", [(10, 0), (12, 2), (13, 1), (14, 3), (16, 2)])
@pytest.mark.parametrize("cplx", [False, True])
def test_residues_are_the_rounded_coefficients(logN, level, cplx):
    P = O.make_params(logN, 60, 45, 3, 60, 2)
    o, ctx, _ = make_env(P, relin=False)
    rng = np.random.default_rng(logN)
    z = rng.uniform(-1, 1, P.N // 2) + (1j * rng.uniform(-1, 1, P.N // 2) if cplx else 0)
    log(f"encode logN={logN} level={level} complex={cplx}")
    pt = ctx.encode(z, level, 2.0 ** 40)
    zero = np.zeros((level + 1, P.N), dtype=np.uint64)
    limbs = o.ntt(ctx.load(zero, zero, noise=2.0 ** 40).add_plain(pt).store()[0], list(range(level + 1)), inverse=True)
    q0 = int(P.moduli[0])
    v = limbs[0].astype(object)
    v = np.where(v > q0 // 2, v - q0, v)
    for i in range(level + 1):
        assert np.array_equal(limbs[i].astype(object), v % int(P.moduli[i])), i
    want = _coefficients(z) * np.longdouble(2.0 ** 40)
    assert np.abs(v.astype(np.longdouble) - want).max() <= 1
    ctx.close()


def test_out_of_range_values_are_refused():
    import pyfideslib_amd as F

    for logN in (12, 13):
        P = O.make_params(logN, 60, 45, 1, 60, 1)
        _, ctx, _ = make_env(P, relin=False)
        for bad in (np.full(P.N // 2, 2.0 ** 30), np.full(P.N // 2, np.nan), np.full(P.N // 2, np.inf)):
            with pytest.raises(F.FidesError):
                ctx.encode(bad, 1, 2.0 ** 40)
        ctx.close()
