"""A server admits jobs for the scratch that their batch takes (needs a GPU):
the arena that a step allocates is the block of the jobs' admitted bytes, at a
job count where two limbs a job more would need a larger one."""
import pytest

from oracle import oracle as O
from tests.gpu_util import log, make_env

pytestmark = pytest.mark.gpu


def block(b):
    """The pool's size classes: eight to a power of two."""
    step = 1 << (b.bit_length() - 4)
    return -(-b // step) * step


def arena(b):
    return block(b // 8 * 9 // 8 * 8)  # whole words, an eighth of headroom


# rings of the fused kernels and of the separate ones
@pytest.mark.parametrize("logN,kind", [(12, "mult"), (12, "rotate"), (11, "mult"), (11, "rotate")])
def test_step_takes_what_was_admitted(logN, kind):
    import pyfideslib_amd as F

    P = O.make_params(logN, 60, 50, 5, 60, 2)
    o, ctx, keys = make_env(P, rotations=(1,))
    a = ctx.load(o.random_poly(P.L + 1, 1), o.random_poly(P.L + 1, 2), noise=2.0 ** 50)
    b = ctx.load(o.random_poly(P.L + 1, 3), o.random_poly(P.L + 1, 4), noise=2.0 ** 50)

    def submit(srv, out):
        srv.submit_mult(a, b, out) if kind == "mult" else srv.submit_rotate(a, 1, out)

    srv = F.Server(ctx, max_slots=256)
    one = ctx.ciphertext()
    submit(srv, one)
    srv.drain()
    # admitted bytes of one job: the smallest budget that takes it
    lo, used = 0, 1 << 30
    while used - lo > 1:
        mid = (lo + used) // 2
        tight = F.Server(ctx, max_slots=1, budget_bytes=mid)
        try:
            submit(tight, one)
            used = mid
        except F.FidesError:
            lo = mid
        tight.close()
    limb = 8 * P.N
    n = next(n for n in range(20, 200) if arena(n * used) < arena(n * (used + 2 * limb)) and n * used > 8 << 20)
    log(f"{kind} logN={logN}: {used} bytes a job, {n} jobs")
    outs = [ctx.ciphertext() for _ in range(n)]
    for x in outs:
        submit(srv, x)
    before = ctx.pool_bytes()
    srv.step()
    ctx.synchronize()
    taken = ctx.pool_bytes() - before
    assert arena(n * used) <= taken <= arena(n * used) + (512 << 10), (taken, arena(n * used))  # the job table beside it
    srv.drain()
    srv.close()
    ctx.close()
