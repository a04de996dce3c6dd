"""Learned solves over the multigrid V-cycle, whose network runs beside the
V-cycle on a stream of its own: the same solve repeated in one context, and in
a second context that was never used before, gives the same bits (the two
pieces share no buffer either writes), and a solve that follows a change of
the densities sees the new ones."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(64, 32), (96, 48), (320, 160), (16, 8, 8)])
def test_learned_over_multigrid_repeats_bit_for_bit(dims):
    import pansfem2_amd as pa
    make = pa.cantilever2d if len(dims) == 2 else pa.cantilever3d
    rng = np.random.default_rng(sum(dims))

    def setup():
        ctx = make(*dims)
        ctx.set_density(first)
        ctx.mg_setup(1)
        ctx.precond_init(seed=5)
        ctx.precond_collect_random(4, seed=9)
        ctx.precond_train(4, lr=1e-3, seed=3)
        return ctx

    ne = int(np.prod(dims))
    first, second = rng.uniform(1e-1, 1.0, ne), rng.uniform(1e-1, 1.0, ne)
    ctx = setup()
    b = ctx.load()
    out = []
    for rho in (first, second, first):
        ctx.set_density(rho)
        for _ in range(2):
            x, st = ctx.pcg(b, op=pa.PF_OP_LEARNED, eps=1e-8)
            assert st["status"] == 1 and st["true_residual"] <= 1.0000001e-8
            out.append((x, st["iterations"]))
    ctx.close()
    other = setup()
    x, st = other.pcg(b, op=pa.PF_OP_LEARNED, eps=1e-8)
    other.close()
    for y, it in (out[1], out[4], out[5], (x, st["iterations"])):
        assert it == out[0][1] and np.array_equal(y, out[0][0])
    assert np.array_equal(out[2][0], out[3][0]) and not np.array_equal(out[2][0], out[0][0])
