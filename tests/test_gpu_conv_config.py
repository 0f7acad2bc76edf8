"""Configurations of the conversions reach the key switches that calls make
(needs a GPU): target groups in the fused conversions, a table's entry as a
forced one, and the matrix-core ModUp in place of them; products, rotations,
hoisted sets, batches and transforms give the same words under each."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.gpu_util import log, make_env

pytestmark = pytest.mark.gpu


def calls(ctx, a, b, diag, level):
    """Every kind of key-switched call; the words of all results."""
    out = [a.mult(b, rescale=True), a.mult(b, rescale=False), a.rotate(3)]
    out += a.rotate_hoisted([1, 2])
    outs = [ctx.ciphertext() for _ in range(2)]
    ctx.mult_batch([a, b], [b, a], outs, rescale=True)
    outs += [ctx.ciphertext() for _ in range(2)]
    ctx.rotate_batch([a, b], [1, 3], outs[2:])
    out += outs + [a.linear_transform(diag, 2, 1, 0, batched_giant=False)]
    return [w for x in out for w in x.store()] + [w for x in a.rotate_hoisted([1, 2], ext=True) for w in x.store_ext()]


@pytest.mark.parametrize("logN,L,dnum,K", [(12, 5, 3, 2), (15, 4, 2, 3), (16, 6, 2, 4), (11, 5, 3, 2)])
def test_results_under_each(logN, L, dnum, K, tmp_path):
    import pyfideslib_amd as F

    P = O.make_params(logN, 60, 50, L, 60, dnum, K=K)
    o, ctx, keys = make_env(P, rotations=(1, 2, 3, 4))
    pq = list(range(P.L + 1 + P.K))
    diag = [ctx.plaintext_ext(o.random_poly(len(pq), 60 + i, primeids=pq)) for i in range(6)]
    fused = 12 <= logN <= 16
    try:
        for level in (L, 1):
            a = ctx.load(o.random_poly(level + 1, 1), o.random_poly(level + 1, 2), noise=2.0 ** 50)
            b = ctx.load(o.random_poly(level + 1, 3), o.random_poly(level + 1, 4), noise=2.0 ** 50)
            assert ctx.fused == fused
            want = calls(ctx, a, b, diag, level)
            got = o.mult((a.store()[0], a.store()[1]), (b.store()[0], b.store()[1]), keys["relin"])
            assert all(np.array_equal(x, y) for x, y in zip(want[2:4], got))
            for kind, cfg in [(k, [tg]) for k in (F.TUNE_MODUP, F.TUNE_MODDOWN) for tg in (1, 2, 5, 64)] + [(F.TUNE_MODUP, [1, 1])]:
                log(f"conversions logN={logN} level={level} kind {kind} {cfg}")
                F.tune_force(kind, cfg)
                if len(cfg) == 1:
                    assert ctx.tune_config(kind, 2) == (cfg + [0, 0, 0], True)
                    assert ctx.fused == fused
                else:
                    assert not ctx.fused
                for _ in range(3):  # planned, captured, replayed
                    got = calls(ctx, a, b, diag, level)
                    assert all(np.array_equal(x, y) for x, y in zip(got, want)), (kind, cfg)
                F.tune_force(-1)
        table = tmp_path / "table.txt"
        table.write_text(f"modup {logN} 1 64 1 1 0 0\nmoddown {logN} 1 64 3 0 0 0\n")
        assert F.tune_load(str(table)) == 2
        assert not ctx.fused and ctx.tune_config(F.TUNE_MODDOWN, 2)[0][0] == 3
        got = calls(ctx, a, b, diag, level)
        assert all(np.array_equal(x, y) for x, y in zip(got, want))
    finally:
        F.tune_force(-1)
        F.tune_load()
    assert ctx.fused == fused
    ctx.close()


def test_rule_reported_for_a_key_switch():
    """What tune_config reports without a configuration is the fused conversions' rule where they run."""
    import pyfideslib_amd as F

    P = O.params_production()
    raw = F.RawParams.from_lists(P.logN, P.L, P.K, P.dnum, P.moduli, P.roots)
    ctx = F.Context(raw)
    try:
        # 64 tiles of 4 columns, targets two at a time, at most 1024 blocks in even rounds
        assert ctx.tune_config(F.TUNE_MODUP, 3) == ([4, 0, 0, 0], False)
        assert ctx.tune_config(F.TUNE_MODDOWN, 2) == ([7, 0, 0, 0], False)
        F.tune_force(F.TUNE_MODUP, [1, 1])
        assert not ctx.fused
    finally:
        F.tune_force(-1)
        ctx.close()


# special primes: tiles of 10 + 1 sources leave room for two blocks a CU, of 12 + 1 for one
@pytest.mark.parametrize("K,hoisted,product", [(10, 3, 5), (11, 1, 5)])
def test_groups_that_repeat_their_sources(K, hoisted, product):
    """Rings whose conversions run their sources' column pass: no more groups than one round of blocks."""
    import pyfideslib_amd as F

    P = O.make_params(13, 60, 59, 17, 59, 2, K=K)
    raw = F.RawParams.from_lists(P.logN, P.L, P.K, P.dnum, P.moduli, P.roots)
    ctx = F.Context(raw)
    # 16 tiles a conversion, 18 targets in rounds of 4
    assert ctx.fused
    assert ctx.tune_config(F.TUNE_MODDOWN, 10)[0][0] == hoisted  # 5 rotations
    assert ctx.tune_config(F.TUNE_MODDOWN, 2)[0][0] == product
    ctx.close()
