"""GPU parity of the resident hex8 Jacobi-PCG (k_pcg_h8_resident: the element
matrix in its parity basis, shared nodes' sums completed axis by axis) against
the assembled-matrix solve, and the rule that decides on the parity basis.

Shapes: one box, one layer per half box and none, 16 elements along a box's edge,
boxes split along one, two and all three axes (nodes with two, four and eight
holders) in equal and unequal parts, both sizes of the kernel (4 and 16 values
per thread).  The first iterates differ from the
assembled solve's by the order of sums and the transforms' roundings: some
hundreds of 1e-16 per entry, 1e-12 with the head room of the recurrences.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (2, 1, 3), (1, 5, 2), (4, 2, 2), (8, 4, 4), (17, 9, 5), (3, 18, 16), (5, 3, 37), (33, 16, 16),
          (30, 15, 17)]


@pytest.fixture(scope="module")
def pa():
    import pansfem2_amd
    return pansfem2_amd


def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def problem(pa, nx, ny, nz):
    ctx = pa.cantilever3d(nx, ny, nz)
    rng = np.random.default_rng(nx * 10000 + ny * 100 + nz)
    ctx.set_density(rng.uniform(0.2, 1.0, nx * ny * nz))
    return ctx, ctx.load() + rng.uniform(-1e-3, 1e-3, ctx.N)


@pytest.mark.parametrize("nx,ny,nz", SHAPES)
def test_iterates_against_assembled(pa, nx, ny, nz):
    print(f"hex8 resident {nx}x{ny}x{nz}", flush=True)
    ctx, b = problem(pa, nx, ny, nz)
    ctx.assemble_csr()
    for k in (1, 2, 6):
        xr, sr = ctx.pcg(b, op=pa.PF_OP_CSR64, eps=1e-14, itrmax=k)
        x, st = ctx.pcg(b, op=pa.PF_OP_EBE64, eps=1e-14, itrmax=k)
        assert st["iterations"] == sr["iterations"]
        assert rel(x, xr) < 1e-12, (k, rel(x, xr))
    xr, sr = ctx.pcg(b, op=pa.PF_OP_CSR64, eps=1e-10)
    x, st = ctx.pcg(b, op=pa.PF_OP_EBE64, eps=1e-10)
    assert st["status"] == 1 and st["true_residual"] < 1e-9
    assert abs(st["iterations"] - sr["iterations"]) <= max(3, 0.005 * sr["iterations"])
    assert rel(x, xr) < 1e-8
    assert np.array_equal(x, ctx.pcg(b, op=pa.PF_OP_EBE64, eps=1e-10)[0])
    x32, s32 = ctx.pcg(b, op=pa.PF_OP_EBE32, eps=1e-9)
    assert s32["status"] == 1 and s32["true_residual"] <= 1.0000001e-9
    assert rel(x32, xr) < 1e-6
    assert ctx.resident_runs() == (5 + s32["outer"], 0)
    ctx.close()


# 256 workgroups: 30x4x2 boxes, 24x5x2 and 14x6x3 uneven ones (4 values per
# thread); 15x5x3 uneven along j and k and 10x6x4 uneven along all axes (16)
@pytest.mark.parametrize("nx,ny,nz", [(60, 30, 30), (47, 26, 23), (41, 33, 35), (75, 37, 39), (97, 47, 51)])
def test_boxes_split_along_three_axes(pa, nx, ny, nz):
    print(f"hex8 resident {nx}x{ny}x{nz}", flush=True)
    ctx, b = problem(pa, nx, ny, nz)
    ctx.assemble_csr()
    for k in (1, 2, 6, 25):
        xr, sr = ctx.pcg(b, op=pa.PF_OP_CSR64, eps=1e-30, itrmax=k)
        x, st = ctx.pcg(b, op=pa.PF_OP_EBE64, eps=1e-30, itrmax=k)
        assert st["iterations"] == sr["iterations"] == k
        assert rel(x, xr) < 1e-12, (k, rel(x, xr))
    assert ctx.resident_runs() == (4, 0)
    ctx.close()


@pytest.mark.parametrize("nx,ny,nz,fits", [(128, 64, 64, True), (132, 66, 66, False)])
def test_largest_boxes_against_launched(pa, nx, ny, nz, fits):
    """16x4x4 boxes of 8x16x16 elements, the largest that the kernel takes, with
    random densities, and a grid beyond it."""
    ctx, b = problem(pa, nx, ny, nz)
    for k in (6, 25):
        x, st = ctx.pcg(b, op=pa.PF_OP_EBE64, eps=1e-30, itrmax=k)
        ctx.set_resident(pa.PF_RESIDENT_OFF)
        xr, sr = ctx.pcg(b, op=pa.PF_OP_EBE64, eps=1e-30, itrmax=k)
        ctx.set_resident(pa.PF_RESIDENT_AUTO)
        assert st["iterations"] == sr["iterations"] == k and rel(x, xr) < 1e-12, (k, rel(x, xr))
    assert ctx.resident_runs() == (2 if fits else 0, 0)
    ctx.close()


@pytest.mark.parametrize("nx,ny,nz", [(17, 9, 5), (47, 26, 23), (75, 37, 39)])
def test_fp32_operator_by_the_work_it_takes(pa, nx, ny, nz):
    """The refinement hides a wrong FP32 operator in the solution, not in the
    steps and inner iterations it takes.  The resident solve aims at an eighth of
    inner_eps and eps, and its operator's roundings are smaller: its steps are as
    many or one fewer, its iterations fewer (602 and 833 in 3 and 3 steps, 1705
    and 2021 in 3 and 3, 2721 and 4177 in 3 and 4); a quarter more than the
    launched solve's is a wrong operator."""
    ctx, b = problem(pa, nx, ny, nz)
    x, st = ctx.pcg(b, op=pa.PF_OP_EBE32, eps=1e-9)
    assert ctx.resident_runs()[0] == st["outer"]
    ctx.set_resident(pa.PF_RESIDENT_OFF)
    xl, sl = ctx.pcg(b, op=pa.PF_OP_EBE32, eps=1e-9)
    print(st, sl, flush=True)
    assert st["status"] == sl["status"] == 1 and st["fallbacks"] == sl["fallbacks"] == 0
    assert abs(st["outer"] - sl["outer"]) <= 1 and st["iterations"] <= 1.25 * sl["iterations"]
    assert rel(x, xl) < 1e-6
    ctx.close()


def test_more_iterations_than_one_launch(pa):
    ctx, _ = problem(pa, 60, 6, 5)
    rng = np.random.default_rng(3)
    ctx.set_density(rng.uniform(0.05, 1.0, 60 * 6 * 5))
    b = ctx.load()
    ctx.assemble_csr()
    for k in (2047, 2048, 2049):
        x, st = ctx.pcg(b, op=pa.PF_OP_EBE64, eps=0.0, itrmax=k)
        assert st["iterations"] == k and st["status"] == 2
    xr, _ = ctx.pcg(b, op=pa.PF_OP_CSR64, eps=1e-11)
    assert rel(x, xr) < 1e-7
    ctx.close()


def test_no_iterations_allowed(pa):
    """itrmax = 0 gives x = 0, and so do the solves of a loop whose cg_itrmax is
    negative (which the loop takes); the solves that follow do not see their
    exchanges as their own (the tags go up all the same)."""
    ctx, b = problem(pa, 17, 9, 5)
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


def test_solve_that_ends_with_a_launch(pa):
    """A solve whose last iterate is the last of its first launch (2048): the
    second launch finds it converged before its first exchange, so that every
    workgroup leaves it by itself, and each has to write its part of x.  eps is
    set a billionth above the residual of iterate 2048; right-hand sides whose
    earlier residuals already lie below that are passed over."""
    ctx, _ = problem(pa, 60, 6, 5)
    ctx.set_density(np.random.default_rng(3).uniform(0.05, 1.0, 60 * 6 * 5))
    ctx.assemble_csr()
    ended = 0
    for seed in range(60):
        b = ctx.load() + np.random.default_rng(seed).uniform(-1e-3, 1e-3, ctx.N)
        _, st = ctx.pcg(b, op=pa.PF_OP_EBE64, eps=0.0, itrmax=2048)
        x, st = ctx.pcg(b, op=pa.PF_OP_EBE64, eps=st["rel_residual"] * (1.0 + 1e-9))
        assert st["status"] == 1 and st["iterations"] <= 2048
        if st["iterations"] == 2048:
            xr, _ = ctx.pcg(b, op=pa.PF_OP_CSR64, eps=1e-12)
            assert rel(x, xr) < 1e-7, rel(x, xr)
            ended += 1
        if ended == 3:
            break
    assert ended == 3, ended
    ctx.close()


def test_element_matrix_without_parity_blocks(pa):
    """A matrix that the mirrors do not leave as it is (a sheared material), one
    that is not symmetric and one that resists translations take the general
    operator: the same iterates as the MFMA operator, which applies any
    matrix.  The scaled original still takes the resident solve."""
    rng = np.random.default_rng(7)
    ctx, b = problem(pa, 6, 4, 5)
    K = ctx.element_stiffness(0, 1.0, 0.3)
    S = rng.uniform(-1, 1, (24, 24))
    other, _ = problem(pa, 6, 4, 5)
    other.set_h8_operator(pa.PF_H8_OP_MFMA)
    for k0 in (K + 1e-3 * (S @ S.T) / 24, K + 1e-6 * rng.uniform(-1, 1, (24, 24)), K + 1e-3 * np.eye(24), 2.0 * K):
        ctx.set_element_matrix(k0)
        other.set_element_matrix(k0)
        x = ctx.pcg(b, op=pa.PF_OP_EBE64, eps=1e-30, itrmax=5)[0]
        xm = other.pcg(b, op=pa.PF_OP_EBE64, eps=1e-30, itrmax=5)[0]
        assert rel(x, xm) < 1e-12
    ctx.close()
    other.close()


def test_mixed_solve_with_nothing_to_do(pa):
    """x = 0 meets eps >= 1: no step is taken, resident or launched."""
    ctx, b = problem(pa, 9, 5, 3)
    for mode in (pa.PF_RESIDENT_AUTO, pa.PF_RESIDENT_OFF):
        ctx.set_resident(mode)
        for eps in (1.0, 3.0):
            x, st = ctx.pcg(b, op=pa.PF_OP_EBE32, eps=eps)
            assert (st["status"], st["iterations"], st["outer"]) == (1, 0, 0) and not np.any(x)
    ctx.close()


def test_default_operator_after_another(pa):
    """PF_H8_OP_AUTO brings a context back to the resident kernel, with the bits
    that it gave before."""
    ctx, b = problem(pa, 9, 5, 3)
    x, _ = ctx.pcg(b, eps=1e-10)
    for kind in (pa.PF_H8_OP_VALU, pa.PF_H8_OP_MFMA):
        ctx.set_h8_operator(kind)
        ran = ctx.resident_runs()[0]
        assert rel(ctx.pcg(b, eps=1e-10)[0], x) < 1e-8 and ctx.resident_runs()[0] == ran
        ctx.set_h8_operator(pa.PF_H8_OP_AUTO)
        assert np.array_equal(ctx.pcg(b, eps=1e-10)[0], x) and ctx.resident_runs()[0] == ran + 1
    for kind in (-2, 2):
        with pytest.raises(pa.PfError):
            ctx.set_h8_operator(kind)
    ctx.close()
