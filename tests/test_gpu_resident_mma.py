"""GPU parity of the resident MMA / CONLIN update (k_mma_resident: one launch per
update) against the launched kernels, which the loops compare with the
reference's, at sizes around the borders of its variants: one workgroup with
idle lanes, several, and one, two and four variables per thread (the borders
are 131072 and 262144 variables on 256 compute units, the end 524288), and,
independently of both, against the solution of the subproblem.

The sums over n variables are added in another order: about sqrt(n) 1e-16 of
their magnitude, which the interior point (ended at 1e-7) passes on to x; 1e-9
holds with head room, as for the loops.  The asymptotes are formed variable by
variable from x's history, with the same operations in both, so that they
differ by what x differs.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["mma", "conlin"])
@pytest.mark.parametrize("nx,ny", [(3, 1), (32, 16), (40, 13), (120, 40), (363, 361), (512, 257), (521, 511),
                                   (1024, 512), (1025, 512)])
def test_updates_against_launched_and_solution(nx, ny, kind):
    import pansfem2_amd as pa
    print(f"resident {kind} {nx}x{ny}", flush=True)
    n = nx * ny
    rng = np.random.default_rng(n)
    ctx, launched = pa.cantilever2d(nx, ny), pa.cantilever2d(nx, ny)
    launched.set_resident(pa.PF_RESIDENT_OFF)
    update, update2 = ((c.mma_update if kind == "mma" else c.conlin_update) for c in (ctx, launched))
    for c in (ctx, launched):
        (c.mma_init if kind == "mma" else c.conlin_init)()
    xs = rng.uniform(0.2, 0.8, n)
    prev = []
    for it in range(4):
        df = -rng.uniform(0.1, 2.0, n)
        dg = np.full(n, 1.0 / (0.5 * n))
        g = float(xs.sum() / (0.5 * n) - 1.0)
        new, steps = update(xs, 1.0 + it, df, g, dg)
        assert 5 < steps < 200
        # both contexts are given the same x, so that each update is compared by itself
        new2, steps2 = update2(xs, 1.0 + it, df, g, dg)
        assert steps == steps2
        assert np.max(np.abs(new - new2)) < 1e-9, np.max(np.abs(new - new2))
        st = ctx.mma_get_state()
        assert st["k"] == it + 1 and np.array_equal(st["xkm1"], xs)
        assert it == 0 or np.array_equal(st["xkm2"], prev[-1])
        if kind == "mma":
            st2 = launched.mma_get_state()
            assert np.array_equal(st["L"], st2["L"]) and np.array_equal(st["U"], st2["U"])
        ref = subproblem(kind, xs, prev, df, g, dg, st)
        # the interior point ends at eps = 1e-7: x is within its barrier's bias
        # of the subproblem's solution, the same at every size
        assert np.max(np.abs(new - ref)) < 2e-3, np.max(np.abs(new - ref))
        assert np.all(new >= 0.01 - 1e-12) and np.all(new <= 1.0 + 1e-12)
        prev.append(xs)
        xs = new
    assert ctx.resident_runs() == (4 if n <= 524288 else 0, 0) and launched.resident_runs() == (0, 0)
    launched.close()
    # the same inputs give the same bits
    ctx2 = pa.cantilever2d(nx, ny)
    (ctx2.mma_init if kind == "mma" else ctx2.conlin_init)()
    (ctx.mma_init if kind == "mma" else ctx.conlin_init)()
    df = -rng.uniform(0.1, 2.0, n)
    u2 = ctx2.mma_update if kind == "mma" else ctx2.conlin_update
    assert np.array_equal(update(xs, 1.0, df, 0.1, dg)[0], u2(xs, 1.0, df, 0.1, dg)[0])
    ctx.close()
    ctx2.close()


def subproblem(kind, x, prev, df, g, dg, st):
    """The separable subproblem solved by bisection on its dual variable."""
    xmin, xmax, move, raa0, albefa = 0.01, 1.0, 0.2, 1e-5, 0.1
    wd = xmax - xmin
    if kind == "mma":
        L, U = st["L"], st["U"]
        al = np.maximum(np.maximum(L + albefa * (x - L), x - move * wd), xmin)
        be = np.minimum(np.minimum(U - albefa * (U - x), x + move * wd), xmax)

        def split(d):
            a, b = np.maximum(d, 0), np.maximum(-d, 0)
            return (U - x) ** 2 * (1.001 * a + 0.001 * b + raa0 / wd), (x - L) ** 2 * (0.001 * a + 1.001 * b + raa0 / wd)
        value = lambda p, q, v: np.sum(p / (U - v) + q / (v - L))  # noqa: E731
        best = lambda p, q: (np.sqrt(p) * L + np.sqrt(q) * U) / (np.sqrt(p) + np.sqrt(q))  # noqa: E731
    else:
        al, be = np.maximum(x - move * wd, xmin), np.minimum(x + move * wd, xmax)
        split = lambda d: (np.maximum(d, 0), np.maximum(-d, 0) * x * x)  # noqa: E731
        value = lambda p, q, v: np.sum(p * v + q / v)  # noqa: E731
        best = lambda p, q: np.sqrt(q / np.maximum(p, 1e-300))  # noqa: E731
    p0, q0 = split(df)
    p, q = split(dg)
    bound = value(p, q, x) - g
    lo, hi = 0.0, 1e4
    for _ in range(200):
        lam = 0.5 * (lo + hi)
        v = np.clip(best(p0 + lam * p, q0 + lam * q), al, be)
        if value(p, q, v) > bound:
            lo = lam
        else:
            hi = lam
    return v


def test_step_cap_leaves_the_state():
    import pansfem2_amd as pa
    ctx = pa.cantilever2d(30, 10)
    ctx.mma_init(max_newton=3)
    x = np.full(300, 0.5)
    new, steps = ctx.mma_update(x, 1.0, -np.ones(300), 0.1, np.full(300, 1 / 150.0))
    assert ctx.last_status == pa.PF_NOT_CONVERGED and steps == 3
    assert np.array_equal(new, x) and ctx.mma_get_state()["k"] == 0
    ctx.close()
