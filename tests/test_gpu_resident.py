"""GPU parity of the resident Jacobi-PCG (k_pcg_q4_resident: one workgroup per
tile for the whole solve, edge values and sums exchanged through tagged words)
against the assembled-matrix solve, which launches every iteration.

Grid shapes: one workgroup (with idle rows and lanes), a single row or column of
elements, several workgroups with uneven tiles, every rows-per-thread variant,
the largest grids of some shapes that fit the chip and the next that do not; the
context counts its resident solves, so that each test knows which kernel ran.
The first iterates
differ from the assembled solve's by the order of sums only: a few hundred
roundings of 1e-16 per entry, 1e-12 with the head room of the recurrences.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1), (2, 1), (1, 9), (16, 8), (31, 15), (63, 1), (7, 130), (120, 40), (97, 53), (301, 149), (255, 255)]


@pytest.fixture(scope="module")
def pa():
    import pansfem2_amd
    return pansfem2_amd


def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def problem(pa, nx, ny, seed=11):
    ctx = pa.cantilever2d(nx, ny)
    rng = np.random.default_rng(seed)
    ctx.set_density(rng.uniform(0.2, 1.0, nx * ny))
    return ctx, ctx.load() + rng.uniform(-1e-3, 1e-3, ctx.N)


@pytest.mark.parametrize("form", [0, 2])
@pytest.mark.parametrize("nx,ny", SHAPES)
def test_iterates_against_assembled(pa, nx, ny, form):
    print(f"resident {nx}x{ny} form {form}", flush=True)
    ctx, b = problem(pa, nx, ny)
    ctx.assemble_csr()
    ctx.set_pcg_form(form)
    for k in (1, 2, 6):
        xr, sr = ctx.pcg(b, op=pa.PF_OP_CSR64, eps=1e-12, itrmax=k)
        x, st = ctx.pcg(b, op=pa.PF_OP_EBE64, eps=1e-12, itrmax=k)
        assert st["iterations"] == sr["iterations"] and st["status"] == sr["status"], (k, st, sr)
        assert rel(x, xr) < 1e-12, (k, rel(x, xr))
    # to the end (301x149: more iterations than one launch runs)
    xr, sr = ctx.pcg(b, op=pa.PF_OP_CSR64, eps=1e-10)
    x, st = ctx.pcg(b, op=pa.PF_OP_EBE64, eps=1e-10)
    assert st["status"] == 1 and st["rel_residual"] < 1e-10
    # CG in exact arithmetic ends within N steps: where a slender beam's takes
    # more (63x1: condition 12 * 63^4 = 2e8, 1400 steps for 252 unknowns),
    # rounding alone decides the count, and the solution is known to the
    # residual times that condition number, so only the residual is bounded
    if sr["iterations"] < ctx.N:
        assert abs(st["iterations"] - sr["iterations"]) <= max(3, 0.005 * sr["iterations"])
        # the operators differ by rounding of K, amplified by the condition
        # number (1e5 at these sizes, so 1e-10 with head room)
        assert rel(x, xr) < 1e-8
    assert st["true_residual"] < 1e-7
    x2, _ = ctx.pcg(b, op=pa.PF_OP_EBE64, eps=1e-10)
    assert np.array_equal(x, x2)
    assert ctx.resident_runs() == (5, 0)
    ctx.close()


# square, 2:1, 3:2, 8:3 and 4:1 grids of 584,000 to 614,000 nodes that fit 256
# workgroups of 150 KB LDS (12 x 8 bytes a node, its rows padded to five), the
# next of some of these shapes, and larger ones
@pytest.mark.parametrize("nx,ny,fits", [(1024, 512, True), (769, 769, True), (1086, 543, True), (958, 639, True),
                                        (1279, 479, True), (1536, 384, True), (770, 770, False), (1088, 544, False),
                                        (815, 791, False), (1023, 703, False)])
def test_large_grids_against_recomputed_form(pa, nx, ny, fits):
    """Near the largest grid a chip holds, and beyond it: the resident (or then
    the launched) forms against the launched recomputing form."""
    print(f"resident large {nx}x{ny}", flush=True)
    ctx, b = problem(pa, nx, ny)
    xs = {}
    for form in (0, 2, 3):
        ctx.set_pcg_form(form)
        xs[form], st = ctx.pcg(b, op=pa.PF_OP_EBE64, eps=1e-12, itrmax=40)
        assert st["iterations"] == 40 and st["status"] == 2
    for form in (0, 2):
        assert rel(xs[form], xs[3]) < 1e-11, rel(xs[form], xs[3])
    assert ctx.resident_runs() == (2 if fits else 0, 0)
    ctx.close()


def test_zero_load_zero_steps_and_grid_change(pa):
    ctx, b = problem(pa, 64, 32)
    for form in (0, 2):
        ctx.set_pcg_form(form)
        x, st = ctx.pcg(np.zeros_like(b), eps=1e-10)
        assert st["status"] == 1 and st["iterations"] == 0 and not np.any(x)
        x, st = ctx.pcg(b, eps=1e-10, itrmax=0)
        assert st["iterations"] == 0 and not np.any(x)
        assert pa.cantilever2d(40, 24, ctx=ctx) is ctx  # another grid in the same context
        ctx.set_density(np.full(40 * 24, 0.5))
        x, st = ctx.pcg(ctx.load(), eps=1e-10)
        assert st["status"] == 1 and st["true_residual"] < 1e-9
        pa.cantilever2d(64, 32, ctx=ctx)
        ctx.set_density(np.random.default_rng(11).uniform(0.2, 1.0, 64 * 32))
    ctx.close()


@pytest.mark.parametrize("form", [0, 2])
def test_no_iterations_allowed(pa, form):
    """itrmax = 0 gives x = 0, and so do the solves of a loop whose cg_itrmax is
    negative (which the loop takes); the solves that follow do not see their
    exchanges as their own (the tags go up all the same)."""
    ctx, b = problem(pa, 97, 53)
    ctx.set_pcg_form(form)
    rho = np.full(ctx.ne, 0.5)
    ctx.set_density(rho)
    x, st = ctx.pcg(b, eps=1e-10)
    x0, s0 = ctx.pcg(b, eps=1e-10, itrmax=0)
    assert s0["status"] == 2 and s0["iterations"] == 0 and not np.any(x0)
    for itrmax in (-1, -7, -1000, -2**31):
        r = ctx.simp_run(1, pa.simp_default_params(cg_itrmax=itrmax))
        assert r["status"] == pa.PF_NOT_CONVERGED and r["cg_iters"][0] == 0 and r["f"][0] == 0.0
        ctx.set_density(rho)
        x1, s1 = ctx.pcg(b, eps=1e-10)
        assert s1["iterations"] == st["iterations"] and np.array_equal(x1, x)
    assert ctx.resident_runs()[0] >= 10 and ctx.resident_runs()[1] == 0
    ctx.close()


@pytest.mark.parametrize("form,last", [(0, 2048), (2, 2047)])
def test_solve_that_ends_with_a_launch(pa, form, last):
    """A solve whose last iterate is the last that its first launch finishes: the
    second launch finds it converged before its first exchange, so that every
    workgroup leaves it by itself, with x complete.  eps is set a billionth above
    the residual of that iterate; right-hand sides whose earlier residuals
    already lie below it are passed over."""
    ctx, _ = problem(pa, 120, 40)
    ctx.set_pcg_form(form)
    ctx.assemble_csr()
    ended = 0
    for seed in range(60):
        b = ctx.load() + np.random.default_rng(seed).uniform(-1e-3, 1e-3, ctx.N)
        _, st = ctx.pcg(b, op=pa.PF_OP_EBE64, eps=0.0, itrmax=last)
        x, st = ctx.pcg(b, op=pa.PF_OP_EBE64, eps=st["rel_residual"] * (1.0 + 1e-9))
        assert st["status"] == 1 and st["iterations"] <= last
        if st["iterations"] == last:
            xr, _ = ctx.pcg(b, op=pa.PF_OP_CSR64, eps=1e-12)
            assert rel(x, xr) < 1e-7, rel(x, xr)
            ended += 1
        if ended == 3:
            break
    assert ended == 3, ended
    ctx.close()


def test_fp32_inner_solves(pa):
    """The FP32 variant inside FP64 refinement."""
    ctx, b = problem(pa, 75, 31)
    x64, _ = ctx.pcg(b, eps=1e-11)
    x32, st = ctx.pcg(b, op=pa.PF_OP_EBE32, eps=1e-10)
    assert st["status"] == 1 and st["true_residual"] <= 1.0000001e-10
    assert rel(x32, x64) < 1e-7
    ctx.close()
