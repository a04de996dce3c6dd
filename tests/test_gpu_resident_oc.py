"""GPU parity of the resident OC bisection (k_oc_resident, the filtered volume as
the product of x+ with the filter's column sums) against the bisection restated
in numpy with the filter applied in every step: the same decisions, lambda and
steps (the volumes differ by rounding, about 1e-15, and none of these decisions
is that close), and x+ to the last bits of its formula.

Sizes: one workgroup with idle lanes, several, the borders between one, two,
four, eight and sixteen elements per thread (131072 times those on 256 compute
units) and beyond the last, which is launched, both element types, a radius that
reaches past one ring.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


SHAPES = [(1, 1), (7, 3), (120, 40), (37, 41), (363, 361), (512, 257), (5, 3, 4), (33, 17, 16)]
LARGE = [(1024, 512), (1025, 512), (1024, 1025), (2048, 1024), (2049, 1024), (128, 90, 90)]


@pytest.mark.parametrize("shape,R", [(s, R) for R in (1.5, 0.5, 2.3) for s in SHAPES] + [(s, 1.5) for s in LARGE])
def test_bisection_against_numpy(shape, R):
    import pansfem2_amd as pa
    print(f"resident OC {shape} R {R}", flush=True)
    n = int(np.prod(shape))
    rng = np.random.default_rng(n)
    make = pa.cantilever2d if len(shape) == 2 else pa.cantilever3d
    ctx = make(*shape, R=R)
    for _ in range(2):  # the second call finds the column sums
        x = rng.uniform(0.2, 0.8, n)
        df, dg = -rng.uniform(0.05, 2.0, n), rng.uniform(0.5, 1.5, n) / n
        l0, l1, steps = 0.0, 1e9, 0
        while (l1 - l0) / (l1 + l0) > 1e-3:
            lam = 0.5 * (l0 + l1)
            ref = np.clip(np.sqrt(-df / (dg * lam)) * x, np.maximum(0, 0.8 * x), np.minimum(1, 1.2 * x))
            if ctx.filter(ref).sum() / (0.5 * n) - 1.0 > 0:
                l0 = lam
            else:
                l1 = lam
            steps += 1
        new, lam_dev, steps_dev = ctx.oc_update(x, df, dg)
        assert lam_dev == lam and steps_dev == steps
        assert np.max(np.abs(new - ref)) < 1e-15
    assert ctx.resident_runs() == (2 if n <= 16 * 131072 else 0, 0)
    # another radius: the column sums follow
    ctx.filter_setup(1.1)
    new, lam_dev, _ = ctx.oc_update(x, df, dg, lambdaeps=1e-2)
    ctx2 = make(*shape, R=1.1)
    assert np.array_equal(new, ctx2.oc_update(x, df, dg, lambdaeps=1e-2)[0])
    ctx.close()
    ctx2.close()


@pytest.mark.parametrize("kw", [dict(vf=0.0), dict(vf=-0.0), dict(vf=float("nan")), dict(scale1=float("inf")),
                                dict(vf=float("inf")), dict(scale1=0.0), dict(vf=-1.0), dict(lambdamin=0.0, lambdamax=0.0)])
def test_unusual_volumes_as_launched(kw):
    """Constraints that divide by zero, are infinite or say nothing, on a design
    with single zero densities: decisions, lambda and x+ as launched."""
    import pansfem2_amd as pa
    ctx = pa.cantilever2d(40, 13)
    rng = np.random.default_rng(1)
    x, df, dg = rng.uniform(0.2, 0.8, ctx.ne), -rng.uniform(0.05, 2.0, ctx.ne), np.full(ctx.ne, 1.0 / ctx.ne)
    x[::17] = 0.0
    out = []
    for mode in (pa.PF_RESIDENT_OFF, pa.PF_RESIDENT_AUTO):
        ctx.set_resident(mode)
        out.append(ctx.oc_update(x, df, dg, **kw) + (ctx.last_status,))
    assert out[0][1:] == out[1][1:], (out[0][1:], out[1][1:])
    assert np.array_equal(out[0][0], out[1][0])
    ctx.close()
