"""What follows when a resident kernel gives up: the launched kernels start the
call over and give the bits that they give with the resident ones switched off,
whether the resident kernel had written nothing (its first launch) or a partial
x (a later one).  PF_RESIDENT_STALL marks a launch as stalled from the host, so
that every kernel ends normally."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pa():
    import pansfem2_amd
    return pansfem2_amd


def problem(pa, dims, ctx=None):
    ctx = (pa.cantilever2d if len(dims) == 2 else pa.cantilever3d)(*dims, ctx=ctx)
    rng = np.random.default_rng(sum(dims))
    ctx.set_density(rng.uniform(0.2, 1.0, ctx.ne))
    return ctx, ctx.load() + rng.uniform(-1e-3, 1e-3, ctx.N)


# (after, eps, itrmax): the first launch, or the second one of a solve that takes 2200 iterations
FIRST, SECOND = (0, 1e-10, 100000), (1, 0.0, 2200)


@pytest.mark.parametrize("dims,form,op,when", [
    ((120, 40), 0, "EBE64", FIRST), ((120, 40), 2, "EBE64", FIRST), ((301, 149), 0, "EBE64", FIRST),
    ((9, 5, 3), 0, "EBE64", FIRST), ((33, 16, 16), 0, "EBE64", FIRST),
    ((120, 40), 0, "EBE64", SECOND), ((301, 149), 2, "EBE64", SECOND), ((60, 6, 5), 0, "EBE64", SECOND),
    ((120, 40), 0, "EBE32", FIRST), ((33, 16, 16), 0, "EBE32", FIRST)])
def test_stalled_solve(pa, dims, form, op, when):
    after, eps, itrmax = when
    print(f"stalled solve {dims} form {form} {op} after {after}", flush=True)
    ctx, b = problem(pa, dims)
    ctx.set_pcg_form(form)
    op = getattr(pa, "PF_OP_" + op)
    ctx.set_resident(pa.PF_RESIDENT_OFF)
    ref, sref = ctx.pcg(b, op=op, eps=eps, itrmax=itrmax)
    assert ctx.resident_runs() == (0, 0)
    ctx.set_resident(pa.PF_RESIDENT_STALL, after)
    x, st = ctx.pcg(b, op=op, eps=eps, itrmax=itrmax)
    assert ctx.resident_runs() == (0, 1)
    assert st["status"] == sref["status"]
    if op == pa.PF_OP_EBE64:  # a mixed hex8 solve aims further when it starts resident
        assert st["iterations"] == sref["iterations"] and np.array_equal(x, ref)
    else:
        assert st["true_residual"] <= 1.0000001 * eps
    ctx.close()


def test_calls_after_stalls_are_launched_and_then_tried_again(pa):
    """One call after the first stall, two after the second in a row, four after
    the third; a solve that ends resident, or a new grid, ends the count."""
    ctx, b = problem(pa, (40, 13))
    solve = lambda: ctx.pcg(b, eps=1e-8)[1]["status"] == 1  # noqa: E731
    runs = []
    ctx.set_resident(pa.PF_RESIDENT_STALL)
    for _ in range(10):
        assert solve()
        runs.append(ctx.resident_runs())
    assert runs == [(0, k) for k in (1, 1, 2, 2, 2, 3, 3, 3, 3, 3)]
    ctx.set_resident(pa.PF_RESIDENT_AUTO)
    assert solve() and solve() and ctx.resident_runs() == (2, 3)
    ctx.set_resident(pa.PF_RESIDENT_STALL)
    assert solve() and solve() and ctx.resident_runs() == (2, 4)
    ctx.set_resident(pa.PF_RESIDENT_AUTO)
    assert solve() and ctx.resident_runs() == (3, 4)
    # updates and bisections count as calls, solves that cannot run resident do not
    ctx.set_resident(pa.PF_RESIDENT_STALL)
    assert solve() and ctx.resident_runs() == (3, 5)
    ctx.set_resident(pa.PF_RESIDENT_AUTO)
    ctx.assemble_csr()
    ctx.pcg(b, op=pa.PF_OP_CSR64, eps=1e-8)
    x, g = np.full(ctx.ne, 0.5), np.full(ctx.ne, 1.0 / ctx.ne)
    ctx.oc_update(x, -g, g)
    assert ctx.resident_runs() == (3, 5)
    ctx.oc_update(x, -g, g)
    assert ctx.resident_runs() == (4, 5)
    ctx.set_resident(pa.PF_RESIDENT_STALL)
    assert solve() and ctx.resident_runs() == (4, 6)
    ctx.set_resident(pa.PF_RESIDENT_AUTO)
    ctx, b = problem(pa, (33, 13), ctx)
    assert solve() and ctx.resident_runs() == (5, 6)
    ctx.close()


@pytest.mark.parametrize("dims", [(1, 1), (40, 13), (363, 361), (5, 3, 4)])
def test_stalled_oc_update(pa, dims):
    ctx, _ = problem(pa, dims)
    rng = np.random.default_rng(3)
    x, df, dg = rng.uniform(0.2, 0.8, ctx.ne), -rng.uniform(0.05, 2.0, ctx.ne), rng.uniform(0.5, 1.5, ctx.ne) / ctx.ne
    ctx.set_resident(pa.PF_RESIDENT_OFF)
    ref = ctx.oc_update(x, df, dg)
    capped = ctx.oc_update(x, df, dg, max_steps=7)
    ctx.set_resident(pa.PF_RESIDENT_STALL)
    got = ctx.oc_update(x, df, dg)
    assert ctx.resident_runs() == (0, 1)
    assert np.array_equal(got[0], ref[0]) and got[1:] == ref[1:]
    # and the resident bisection itself, two calls later: the same decisions
    ctx.set_resident(pa.PF_RESIDENT_AUTO)
    ctx.oc_update(x, df, dg)
    for want, kw in ((ref, {}), (capped, dict(max_steps=7))):
        got = ctx.oc_update(x, df, dg, **kw)
        assert got[1:] == want[1:] and np.max(np.abs(got[0] - want[0])) < 1e-15
    assert ctx.resident_runs() == (2, 1)
    ctx.close()


@pytest.mark.parametrize("kind", ["mma", "conlin"])
@pytest.mark.parametrize("n", [(3, 1), (120, 40)])
def test_stalled_mma_update(pa, n, kind):
    rng = np.random.default_rng(5)
    ne = n[0] * n[1]
    calls = [(-rng.uniform(0.1, 2.0, ne), np.full(ne, 2.0 / ne)) for _ in range(3)]
    out = {}
    for mode in (pa.PF_RESIDENT_OFF, pa.PF_RESIDENT_STALL):
        ctx = pa.cantilever2d(*n)
        (ctx.mma_init if kind == "mma" else ctx.conlin_init)()
        update = ctx.mma_update if kind == "mma" else ctx.conlin_update
        x, steps = np.full(ne, 0.5), []
        for k, (df, dg) in enumerate(calls):
            ctx.set_resident(mode)
            x, s = update(x, 1.0, df, float(2.0 * x.mean() - 1.0), dg)
            steps.append(s)
        st = ctx.mma_get_state()
        assert ctx.resident_runs() == (0, 0 if mode == pa.PF_RESIDENT_OFF else 2)  # the second call is launched
        out[mode] = (x, steps, st["k"], st["xkm1"], st["xkm2"], st["L"], st["U"])
        ctx.close()
    a, b = out.values()
    assert a[1] == b[1] and a[2] == b[2] == len(calls)
    for i in (0, 3, 4) + ((5, 6) if kind == "mma" else ()):
        assert np.array_equal(a[i], b[i])


@pytest.mark.parametrize("dims,op,after", [((120, 40), "EBE64", 0), ((120, 40), "EBE32", 0),
                                           ((33, 16, 16), "EBE64", 0), ((33, 16, 16), "EBE64", 1),
                                           ((33, 16, 16), "EBE32", 0), ((33, 16, 16), "EBE32", 1)])
def test_solve_without_memory_for_the_exchange(pa, dims, op, after):
    """Resident solves allocate an exchange buffer, on hex8 another for x: where
    one of them cannot be had the launched kernels solve, which need neither."""
    ctx, b = problem(pa, dims)
    op = getattr(pa, "PF_OP_" + op)
    ctx.set_resident(pa.PF_RESIDENT_OFF)
    ref, sref = ctx.pcg(b, op=op, eps=1e-9)
    for _ in range(2):
        ctx.set_resident(pa.PF_RESIDENT_NOMEM, after)
        x, st = ctx.pcg(b, op=op, eps=1e-9)
        assert st["status"] == sref["status"] == 1 and st["true_residual"] < 1e-8
        if op == pa.PF_OP_EBE64:
            assert np.array_equal(x, ref)
        assert ctx.resident_runs() == (0, 0)
        after = 0  # the exchange buffer is there by now, if it could be had
    ctx.set_resident(pa.PF_RESIDENT_AUTO)
    ctx.pcg(b, op=op, eps=1e-9)
    assert ctx.resident_runs()[0] >= 1
    ctx.close()


def test_oc_update_without_memory_for_the_column_sums(pa):
    ctx, _ = problem(pa, (40, 13))
    rng = np.random.default_rng(3)
    x, df, dg = rng.uniform(0.2, 0.8, ctx.ne), -rng.uniform(0.05, 2.0, ctx.ne), np.full(ctx.ne, 1.0 / ctx.ne)
    ctx.set_resident(pa.PF_RESIDENT_OFF)
    ref = ctx.oc_update(x, df, dg)
    ctx.set_resident(pa.PF_RESIDENT_NOMEM)
    got = ctx.oc_update(x, df, dg)
    assert ctx.resident_runs() == (0, 0) and np.array_equal(got[0], ref[0]) and got[1:] == ref[1:]
    ctx.set_resident(pa.PF_RESIDENT_AUTO)
    ctx.oc_update(x, df, dg)
    assert ctx.resident_runs() == (1, 0)
    ctx.close()


def test_refused_launches(pa):
    """A refusal costs the runtime 40 ms, more than a small solve: it is asked
    again after 1024 launched calls, also on a new grid, and every kind of call
    gives the bits of the launched kernels meanwhile."""
    ctx, b = problem(pa, (40, 13))
    rng = np.random.default_rng(3)
    x, df, dg = rng.uniform(0.2, 0.8, ctx.ne), -rng.uniform(0.05, 2.0, ctx.ne), np.full(ctx.ne, 1.0 / ctx.ne)

    def calls():
        ctx.mma_init()
        return (ctx.pcg(b, eps=1e-8)[0], ctx.oc_update(x, df, dg)[0], ctx.mma_update(x, 1.0, df, 0.1, dg)[0],
                ctx.pcg(b, op=pa.PF_OP_EBE32, eps=1e-8)[0])
    ctx.set_resident(pa.PF_RESIDENT_OFF)
    ref = calls()
    for turn in range(4):  # each kind of call is the one refused
        ctx.close()
        ctx, b = problem(pa, (40, 13))
        ctx.set_resident(pa.PF_RESIDENT_OFF)
        ctx.mma_init()
        first = (lambda: ctx.pcg(b, eps=1e-8), lambda: ctx.oc_update(x, df, dg),
                 lambda: ctx.mma_update(x, 1.0, df, 0.1, dg), lambda: ctx.pcg(b, op=pa.PF_OP_EBE32, eps=1e-8))[turn]
        want = first()
        ctx.mma_init()
        ctx.set_resident(pa.PF_RESIDENT_REFUSED)
        got = first()
        assert np.array_equal(got[0], want[0]) and ctx.resident_runs() == (0, 1)
        for got, want in zip(calls(), ref):
            assert np.array_equal(got, want)
        assert ctx.resident_runs() == (0, 1)
    ctx, b = problem(pa, (8, 4), ctx)
    for _ in range(1025 - 4 - 1):
        ctx.pcg(b, eps=1e-2)
    assert ctx.resident_runs() == (0, 1)
    ctx.set_resident(pa.PF_RESIDENT_AUTO)
    ctx.pcg(b, eps=1e-2)
    assert ctx.resident_runs() == (1, 1)
    ctx.close()


def test_mode_argument_checked(pa):
    ctx = pa.cantilever2d(8, 4)
    for mode, after in ((5, 0), (-1, 0), (2, -1)):
        with pytest.raises(pa.PfError):
            ctx.set_resident(mode, after)
    ctx.close()
