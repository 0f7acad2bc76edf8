"""Large batches of Chebyshev series (needs a GPU): the baby-step sums are held
in groups of a bounded size, or formed one by one, and every member's words are
those of its own bootstrap, whose sums are all formed together: the grouped and
the single form agree exactly.  The memory is that of the sums one by one."""
import numpy as np
import pytest

from pyfideslib_amd import bootstrap as B
from pyfideslib_amd import params as PP
from tests.gpu_util import log

pytestmark = pytest.mark.gpu


# scaling primes on the FP64 units and past them
@pytest.mark.parametrize("bits", [50, 55])
def test_bootstraps_together(bits):
    import pyfideslib_amd as F

    raw = PP.ckks_params(10, 60, bits, 20, 60, 3)
    ctx = F.Context(raw)
    rng = np.random.default_rng(3)
    mods = list(raw.moduli) + list(raw.special_moduli)
    # exact arithmetic on uniform keys and inputs: the words are all that counts
    uniform = lambda qs: np.stack([rng.integers(0, q, raw.N, dtype=np.uint64) for q in qs])  # noqa: E731
    key = tuple(np.stack([uniform(mods) for _ in range(raw.dnum)]) for _ in range(2))
    ctx.load_eval_key(key)
    bs = B.Bootstrapper(ctx, 2.0 ** bits, level_budget=(3, 3), K=28, double_angle=3, degree=119)
    for r in bs.rotations:
        ctx.load_rotation_key(r, key)
    ctx.load_automorph_key(2 * raw.N - 1, key)
    n = 130  # two series each: 40 take three sums at a time, 130 one
    gs = [ctx.load(uniform(mods[:1]), uniform(mods[:1]), noise=2.0 ** bits) for _ in range(n)]
    outs = [ctx.ciphertext() for _ in range(n)]
    ctx.synchronize()
    before = ctx.pool_bytes()
    log("40 bootstraps")
    bs.bootstrap_batch(gs[:40], outs=outs[:40])
    ctx.synchronize()
    taken = (ctx.pool_bytes() - before) / (16 * (raw.L + 1) * raw.N)
    # sums one by one: 5638 ciphertexts; 8 sums of 80 series held at once: 5798
    assert taken < 5660, taken
    check = {0, 17, 39}
    got = {i: outs[i].store() for i in check}
    log("130 bootstraps")
    bs.bootstrap_batch(gs, outs=outs)
    for i in sorted(check | {77, 129}):
        want = bs.bootstrap(gs[i]).store()
        for words in [outs[i].store()] + ([got[i]] if i in got else []):
            assert all(np.array_equal(x, y) for x, y in zip(words, want)), i
    bs.close()
    ctx.close()
