"""Chebyshev series whose baby-step sums are taken together (needs a GPU):
from the fewest sums to the most and past them, weights for both kinds of
primes, sums that use some of the terms, one or none, and rings that rescale in
either form; the values against the FP64 series."""
import numpy as np
import pytest
from numpy.polynomial import chebyshev as npc

from oracle import oracle as O
from tests.gpu_util import log, make_env

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("logN,bits", [(11, 50), (12, 50), (12, 55), (12, 40)])
def test_series(logN, bits):
    P = O.make_params(logN, 60, bits, 12, 60, 3)
    o, ctx, keys = make_env(P, seed=5)
    rng = np.random.default_rng(bits)
    z = rng.uniform(-1, 1, P.N // 2)
    g = ctx.load(*o.encrypt_slots(z, P.L, 77), noise=2.0 ** P.scale_bits)
    for deg, keep in ((3, "all"), (6, "all"), (15, "odd"), (24, "all"), (47, "few"), (119, "all"), (119, "odd"),
                      (255, "all"), (287, "all")):
        c = rng.normal(0, 1, deg + 1) / (np.arange(deg + 1) + 1.0) ** 1.5
        if keep == "odd":
            c[0::2] = 0
        elif keep == "few":
            c[np.arange(deg + 1) % 8 != 7] = 0
        c[-1] = 0.01
        log(f"series logN={logN} bits={bits} degree {deg} {keep}")
        out = g.chebyshev_series([float(v) for v in c])
        dec = o.decrypt_slots(*out.store(), out.info()["noise"])
        err = np.abs(dec - npc.chebval(z, c)).max()
        assert err < 1e-5, (deg, keep, err)  # as the series' own tests
    ctx.close()
