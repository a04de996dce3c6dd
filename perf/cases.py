"""The work whose time matters to users of pansfem2_amd, as measurable cases.

Each case is a dict of plain values.  Kinds:

  loop   simp_run: the SIMP loop (filter, volume, moduli, solve, compliance and
         sensitivities, OC / MMA / CONLIN update) for a few iterations from a
         given design;
  solve  one solve K u = b at a given design, with Jacobi-PCG (ScalingCG's
         order or the single-reduction form), mixed precision, multigrid, the
         learned preconditioner over the V-cycle, or the assembled CSR matrix
         (assembly included, as the C++ facade's CSR + ScalingCG do it);
  train  Adam steps of the preconditioner's network (forward and backward).

Grids are the cantilevers of the repository's tests and benchmark (left edge
or face clamped, SIMP moduli with E0 = 1e-9 and p = 3).  Designs are smooth
multi-scale random fields pushed towards solid and void, as they look part of
the way through an optimisation; every random value comes from the seed.
"""
import itertools
import math

import numpy as np
import torch
import torch.nn.functional as F

import pansfem2_amd as pa

OPS = {"jacobi": pa.PF_OP_EBE64, "mixed": pa.PF_OP_EBE32, "mg": pa.PF_OP_MG, "learned": pa.PF_OP_LEARNED,
       "csr": pa.PF_OP_CSR64}
OPTIMISERS = {"oc": 0, "mma": 1, "conlin": 2}
E0, PENAL, NU, VF, RADIUS = 1e-9, 3.0, 0.3, 0.5, 1.5


def listed():
    return [
        # the small sample run: latency and launches count
        dict(name="loop_oc_q4_120x40", kind="loop", nx=120, ny=40, nz=0, op="jacobi", form=0, opt="oc", iters=5,
             heaviside=False),
        # a mid-size run with the projection filter, odd sizes, single-reduction solves
        dict(name="loop_oc_heaviside_q4_301x149", kind="loop", nx=301, ny=149, nz=0, op="jacobi", form=1, opt="oc",
             iters=2, heaviside=True),
        # the benchmark's solve: FP64 Jacobi-PCG at 1024x512, single-reduction form
        dict(name="solve_q4_1024x512", kind="solve", nx=1024, ny=512, nz=0, op="jacobi", form=1),
        # the benchmark's largest plane problem (beyond the last-level cache), to its 1e-8
        dict(name="solve_q4_2048x1024", kind="solve", nx=2048, ny=1024, nz=0, op="jacobi", form=1, eps=1e-8),
        # the default solver (ScalingCG's order) on a ragged grid
        dict(name="solve_default_q4_601x333", kind="solve", nx=601, ny=333, nz=0, op="jacobi", form=0),
        # FP32 operator inside FP64 refinement, solid elements
        dict(name="solve_mixed_h8_60x30x30", kind="solve", nx=60, ny=30, nz=30, op="mixed", form=0, eps=1e-8),
        # assembled matrix: what the reference's drivers do through the facade
        dict(name="solve_csr_q4_256x128", kind="solve", nx=256, ny=128, nz=0, op="csr", form=0),
        # solid elements: the benchmark's grid with plain Jacobi-PCG
        dict(name="solve_h8_128x64x64", kind="solve", nx=128, ny=64, nz=64, op="jacobi", form=0),
        # multigrid-preconditioned runs, plane and solid
        dict(name="loop_mma_mg_q4_1024x512", kind="loop", nx=1024, ny=512, nz=0, op="mg", form=0, opt="mma", iters=3,
             heaviside=False),
        dict(name="loop_oc_mg_h8_128x64x64", kind="loop", nx=128, ny=64, nz=64, op="mg", form=0, opt="oc", iters=2,
             heaviside=False),
        # the learned preconditioner over the V-cycle: a solve, and training steps
        dict(name="solve_learned_q4_1024x512", kind="solve", nx=1024, ny=512, nz=0, op="learned", form=0,
             eps=1e-8),
        dict(name="train_q4_1024x512", kind="train", nx=1024, ny=512, nz=0, steps=8),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mg_size(rng, dim):
    """Element counts that coarsen by halves to a small level."""
    if dim == 2:
        k = rng.randint(3, 7)
        return rng.randint(5, 7) << k, rng.randint(2, 5) << k, 0
    k = rng.randint(2, 4)
    return rng.randint(3, 7) << k, rng.randint(2, 3) << k, rng.randint(2, 3) << k


def draw(rng):
    kind = rng.choice(["loop", "loop", "loop_mg", "loop_mg_h8", "solve", "solve", "solve_big", "solve_h8", "solve_h8",
                       "mixed", "csr", "solve_mg", "learned", "train"])
    opt = rng.choice(["oc", "oc", "mma", "conlin"])
    heaviside = rng.random() < 0.3
    form = rng.randint(0, 1)
    nx = _log_int(rng, 30, 420)
    ny = max(8, int(nx * rng.uniform(0.3, 1.0)))
    if kind == "loop":
        return dict(kind="loop", nx=nx, ny=ny, nz=0, op="jacobi", form=form, opt=opt, iters=rng.randint(1, 3),
                    heaviside=heaviside)
    if kind in ("loop_mg", "loop_mg_h8"):
        nx, ny, nz = _mg_size(rng, 2 if kind == "loop_mg" else 3)
        return dict(kind="loop", nx=nx, ny=ny, nz=nz, op="mg", form=0, opt=opt, iters=rng.randint(1, 3),
                    heaviside=heaviside)
    if kind in ("solve", "csr"):
        return dict(kind="solve", nx=nx, ny=ny, nz=0, op="jacobi" if kind == "solve" else kind, form=form)
    if kind == "solve_big":
        nx = _log_int(rng, 420, 1400)
        return dict(kind="solve", nx=nx, ny=int(nx * rng.uniform(0.3, 0.8)), nz=0, op="jacobi", form=form, eps=1e-8)
    if kind in ("solve_h8", "mixed"):
        nx = _log_int(rng, 10, 120 if kind == "solve_h8" else 72)
        ny, nz = (max(6, int(nx * rng.uniform(0.25, 0.7))) for _ in range(2))
        return dict(kind="solve", nx=nx, ny=ny, nz=nz, op="jacobi" if kind == "solve_h8" else kind, form=0,
                    eps=1e-10 if kind == "solve_h8" else 1e-8)
    nx, ny, nz = _mg_size(rng, 2)
    if kind == "train":
        return dict(kind="train", nx=nx, ny=ny, nz=0, steps=rng.randint(2, 8))
    return dict(kind="solve", nx=nx, ny=ny, nz=nz, op="mg" if kind == "solve_mg" else "learned", form=0,
                eps=1e-8)


# ------------------------------------------------------------------ inputs --
def _shape(case):
    return (case["nx"], case["ny"]) + ((case["nz"],) if case["nz"] else ())


def _field(shape, gen, cells):
    """Smooth random field: a coarse lattice of normal values interpolated to
    the element grid."""
    lat = torch.randn((1, 1) + tuple(max(2, c) for c in cells), generator=gen, dtype=torch.float64)
    return F.interpolate(lat, size=shape, mode="bilinear" if len(shape) == 2 else "trilinear",
                         align_corners=True)[0, 0]


def _noise(shape, gen):
    longest = max(shape)
    f = torch.zeros(shape, dtype=torch.float64)
    for cells, amp in ((6, 1.0), (20, 0.6), (60, 0.3)):
        f += amp * _field(shape, gen, [max(2, cells * n // longest) for n in shape])
    return (f - f.mean()) / f.std()


def _density(case, seed):
    """Densities in (0.1, 1): members, thin material and grey transitions.  Jacobi-PCG
    takes as many iterations on them as on the benchmark's designs (about 13
    per element of the longer side)."""
    gen = torch.Generator().manual_seed(int(seed))
    return (0.1 + 0.9 * torch.sigmoid(2.0 * _noise(_shape(case), gen))).numpy().reshape(-1)


def _design(case, seed):
    """Design variables of an early optimisation step: 0.5 with variations."""
    gen = torch.Generator().manual_seed(int(seed))
    return (VF + 0.1 * torch.tanh(_noise(_shape(case), gen))).numpy().reshape(-1)


def _loads(case, seed):
    """(node, dof, value): one to three point loads on the free end."""
    rng = np.random.default_rng(int(seed))
    dim = len(_shape(case))
    face = (case["ny"] + 1) * (case["nz"] + 1 if dim == 3 else 1)
    k = int(rng.integers(1, 4))
    node = face * case["nx"] + rng.integers(0, face, k)
    return node.astype(np.int32), rng.integers(0, dim, k).astype(np.int32), -rng.uniform(0.2, 1.0, k)


def _weights(count, dim, seed):
    """Network parameters of the size of a trained network's (12 layers)."""
    spec = [(16, 16), (16, 16), (16, 32), (32, 32), (32, 32), (32, 32), (32, 64), (64, 32), (32, 32), (32, 16),
            (16, 16), (16, 16)]
    rng = np.random.default_rng(int(seed))
    out = []
    for cin, cout in spec:
        a = math.sqrt(6.0 / (3 ** dim * cin))
        out.append(rng.uniform(-a, a, 3 ** dim * cin * cout).astype(np.float32))
    w = np.concatenate(out)
    assert w.size == count
    return w


def prepare(case, seed):
    nz = case["nz"]
    ctx = pa.cantilever3d(*_shape(case)) if nz else pa.cantilever2d(*_shape(case))
    st = dict(case=case, ctx=ctx)
    if case["kind"] == "loop":
        ctx.set_pcg_form(case["form"])
        if case["op"] == "mg":
            ctx.mg_setup(1)
        st["s0"] = _design(case, seed)
        st["params"] = pa.simp_default_params(solver=OPS[case["op"]], use_mma=OPTIMISERS[case["opt"]], vf=VF,
                                              heaviside=int(case["heaviside"]))
        return st
    ctx.set_density(_density(case, seed))
    if case["kind"] == "train":
        ctx.precond_init(seed=1)
        ctx.precond_collect_random(8, seed=int(seed) + 1)
        st["w0"] = _weights(ctx.precond_num_params(), 2, seed)
        st["seed"] = int(seed) + 2
        return st
    ctx.set_pcg_form(case["form"])
    if case["op"] in ("mg", "learned"):
        ctx.mg_setup(1)
    if case["op"] == "learned":
        ctx.precond_init(seed=1)
        ctx.precond_load(_weights(ctx.precond_num_params(), 2, seed))
    ctx.set_point_loads(*_loads(case, seed))
    st["b"] = torch.from_numpy(ctx.load()).cuda()
    st["x"] = torch.empty_like(st["b"])
    return st


def run(state):
    case, ctx = state["case"], state["ctx"]
    if case["kind"] == "loop":
        r = ctx.simp_run(case["iters"], state["params"], state["s0"])
        return {k: r[k] for k in ("s", "rho", "f", "g")}
    if case["kind"] == "train":
        ctx.precond_load(state["w0"])
        first, last = ctx.precond_train(case["steps"], lr=1e-3, seed=state["seed"])
        return {"loss": [first, last], "params": ctx.precond_save()}
    if case["op"] == "csr":
        ctx.assemble_csr()
    ctx.pcg_dev(state["b"].data_ptr(), state["x"].data_ptr(), op=OPS[case["op"]], eps=case.get("eps", 1e-10))
    return state["x"]


# ------------------------------------------------------------------- sizes --
def _counts(case):
    sh = _shape(case)
    dim = len(sh)
    ne = math.prod(sh)
    n = dim * math.prod(s + 1 for s in sh)
    return sh, dim, ne, n


def _solve_flops(case):
    """Iterations such systems take (Jacobi-PCG: in proportion to the longest
    side; V-cycle: about constant) times the operator and the vector updates."""
    sh, dim, ne, n = _counts(case)
    nd = dim * 2 ** dim
    per = ne * (2 * nd * nd + nd) + 12 * n
    if case["op"] in ("mg", "learned"):
        cycle = 3 * (4 if dim == 2 else 8) / (3 if dim == 2 else 7) * ne * 2 * nd * nd
        net = 0.0
        if case["op"] == "learned":
            net = 2 * 9 * n / dim * (4 * 256 + (512 + 1024 + 512) / 4 + 3 * 1024 / 16 + 4096 / 64)
        return 40 * (per + cycle + net)
    its = (14 if dim == 2 else 27) * max(sh)
    return its * per


def work(case):
    sh, dim, ne, n = _counts(case)
    if case["kind"] == "train":
        net = 2 * 9 * n / dim * (4 * 256 + (512 + 1024 + 512) / 4 + 3 * 1024 / 16 + 4096 / 64)
        # forward, input gradients, weight gradients; three operator products
        return dict(bytes=case["steps"] * 4.0 * (ne + 2 * n), flops=case["steps"] * (3 * net + 3 * ne * 136))
    if case["kind"] == "loop":
        # design in and out, per iteration the solve and about 30 trial updates
        return dict(bytes=case["iters"] * (16.0 * ne + 8.0 * n) + 16.0 * ne,
                    flops=case["iters"] * (_solve_flops(case) + 30 * 30 * ne))
    return dict(bytes=8.0 * (ne + 2 * n), flops=_solve_flops(case))


def tolerance(case):
    """About four times what reordered sums change (the other form of the
    recurrences, the other operator kernel, the other prolongation), rounded up
    over the sizes that are drawn."""
    if case["kind"] == "train":
        # weights perturbed by 1e-5, well below their bf16 rounding
        return {"rel": 0.02, "max": 0.3}
    if case["kind"] == "loop":
        # the volume constraint passes near zero: 7e-9 of it against 64 bits
        return {"rel": 3e-8, "max": 3e-7}
    return {"rel": 2e-7 if case.get("eps", 1e-10) > 1e-9 else 2e-8}


# ----------------------------------------------------- the same in 64 bits --
def _element_matrix(dim):
    """Stiffness of the unit element at E = 1 (plane strain, or solid), two
    Gauss points a side; corners in lexicographic order."""
    corners = list(itertools.product((0, 1), repeat=dim))
    pairs = [(0, 1)] if dim == 2 else [(0, 1), (1, 2), (0, 2)]
    nv = dim + len(pairs)
    D = np.zeros((nv, nv))
    D[:dim, :dim] = NU
    D[range(dim), range(dim)] = 1 - NU
    D[range(dim, nv), range(dim, nv)] = (1 - 2 * NU) / 2
    D /= (1 + NU) * (1 - 2 * NU)
    g = (0.5 - 0.5 / math.sqrt(3.0), 0.5 + 0.5 / math.sqrt(3.0))
    K = np.zeros((dim * len(corners),) * 2)
    for pt in itertools.product(g, repeat=dim):
        B = np.zeros((nv, dim * len(corners)))
        for c, cor in enumerate(corners):
            f = [x if s else 1 - x for x, s in zip(pt, cor)]
            grad = [(1 if cor[k] else -1) * math.prod(f[:k] + f[k + 1:]) for k in range(dim)]
            for k in range(dim):
                B[k, dim * c + k] = grad[k]
            for q, (a, b) in enumerate(pairs):
                B[dim + q, dim * c + a] = grad[b]
                B[dim + q, dim * c + b] = grad[a]
        K += B.T @ D @ B / 2 ** dim
    return torch.from_numpy(K).cuda(), corners


class _Grid:
    """The cantilever in plain torch, FP64."""

    def __init__(self, case):
        self.sh = _shape(case)
        self.dim = len(self.sh)
        self.K, self.corners = _element_matrix(self.dim)
        self.nodes = tuple(s + 1 for s in self.sh)
        self.win = [tuple(slice(c, c + s) for c, s in zip(cor, self.sh)) for cor in self.corners]
        self.fixed = self.dim * math.prod(self.nodes[1:])

    def gather(self, u):
        return torch.cat([u[w] for w in self.win], dim=-1)

    def scatter(self, fe):
        y = torch.zeros(self.nodes + (self.dim,), dtype=torch.float64, device="cuda")
        for c, w in enumerate(self.win):
            y[w] += fe[..., self.dim * c:self.dim * (c + 1)]
        y[0] = 0
        return y

    def solve(self, E, b, most=60000):
        """Jacobi-PCG to a residual of 1e-13; None if it takes too many steps."""
        Ee = E.reshape(self.sh + (1,))
        D = self.scatter(Ee * self.K.diagonal())
        D[0] = 1
        x = torch.zeros_like(b)
        r = b.clone()
        z = r / D
        p = z.clone()
        rz = (r * z).sum()
        stop = 1e-13 * float(b.norm())
        for k in range(most):
            q = self.scatter(Ee * (self.gather(p) @ self.K))
            a = rz / (p * q).sum()
            x += a * p
            r -= a * q
            z = r / D
            new = (r * z).sum()
            p = z + (new / rz) * p
            rz = new
            if k % 64 == 63 and float(r.norm()) < stop:
                return x
        return None

    def filter(self, v):
        num, den = torch.zeros_like(v), torch.zeros_like(v)
        for off in itertools.product((-1, 0, 1), repeat=self.dim):
            d = math.sqrt(sum(o * o for o in off))
            if d > RADIUS:
                continue
            w = (RADIUS - d) / RADIUS
            to = tuple(slice(max(0, -o), s - max(0, o)) for o, s in zip(off, self.sh))
            frm = tuple(slice(max(0, o), s - max(0, -o)) for o, s in zip(off, self.sh))
            num[to] += w * v[frm]
            den[to] += w
        return num / den


def _exact_loop(case, seed):
    g = _Grid(case)
    s = torch.from_numpy(_design(case, seed)).cuda().reshape(g.sh)
    ne = s.numel()
    b = torch.zeros(g.nodes + (g.dim,), dtype=torch.float64, device="cuda")
    if g.dim == 2:
        b[-1, 0, 1] = -1.0
    else:
        nz = case["nz"]
        b[-1, 0, :, 1] = -1.0 / nz
        b[-1, 0, 0, 1] = b[-1, 0, -1, 1] = -0.5 / nz
    dg = torch.full_like(s, 1.0 / (VF * ne))
    beta = 0.0

    def project(v):
        t = math.tanh(0.5 * beta)
        return 0.5 * (t + torch.tanh(beta * (v - 0.5))) / t if beta > 0 else v

    def slope(v):
        return 0.5 * beta * (1 - torch.tanh(beta * (v - 0.5)) ** 2) / math.tanh(0.5 * beta) if beta > 0 else 1.0

    old = []
    fs, gs = [], []
    low = up = None
    for it in range(case["iters"]):
        if case["heaviside"]:
            beta = 0.5 * 2.0 ** (it // 40 + 1)
        st = g.filter(s)
        rho = project(st)
        E = rho ** PENAL + E0 * (1 - rho ** PENAL)
        u = g.solve(E, b)
        if u is None:
            return None
        ue = g.gather(u)
        ce = ((ue @ g.K) * ue).sum(-1)
        f = float((E * ce).sum())
        vol = float(rho.sum()) / (VF * ne) - 1.0
        fs.append(f)
        gs.append(vol)
        df = g.filter(-PENAL * (1 - E0) * rho ** (PENAL - 1) * ce * slope(st))
        dgs = g.filter(dg * slope(st))
        if case["opt"] == "oc":
            l0, l1 = 0.0, 1e9
            while (l1 - l0) / (l1 + l0) > 1e-3:
                lam = 0.5 * (l0 + l1)
                x = s * torch.sqrt(-df / (dgs * lam))
                x = torch.minimum(torch.maximum(x, (0.8 * s).clamp(min=0)), (1.2 * s).clamp(max=1))
                if float(project(g.filter(x)).sum()) / (VF * ne) > 1.0:
                    l0 = lam
                else:
                    l1 = lam
            s = x
            continue
        # MMA / CONLIN: the separable subproblem solved by bisection on its dual
        prm = pa.simp_default_params().mma
        xmin, xmax, mv = prm.xmin, prm.xmax, prm.move
        dx = xmax - xmin
        if case["opt"] == "mma":
            if it < 2:
                low, up = s - prm.asyinit * dx, s + prm.asyinit * dx
            else:
                t = (s - old[-1]) * (old[-1] - old[-2])
                k = torch.where(t < 0, prm.asydecr, torch.where(t > 0, prm.asyincr, 1.0))
                low, up = s - k * (old[-1] - low), s + k * (up - old[-1])
            low = torch.minimum(torch.maximum(low, s - 10 * dx), s - 0.01 * dx)
            up = torch.maximum(torch.minimum(up, s + 10 * dx), s + 0.01 * dx)
            al = torch.maximum(torch.maximum(low + prm.albefa * (s - low), s - mv * dx), torch.full_like(s, xmin))
            be = torch.minimum(torch.minimum(up - prm.albefa * (up - s), s + mv * dx), torch.full_like(s, xmax))

            def split(d):
                a, c = d.clamp(min=0), (-d).clamp(min=0)
                return ((up - s) ** 2 * (1.001 * a + 0.001 * c + prm.raa0 / dx),
                        (s - low) ** 2 * (0.001 * a + 1.001 * c + prm.raa0 / dx))

            def value(p, q, x):
                return float((p / (up - x) + q / (x - low)).sum())

            def best(p, q):
                return (p.sqrt() * low + q.sqrt() * up) / (p.sqrt() + q.sqrt())
        else:
            al, be = (s - mv * dx).clamp(min=xmin), (s + mv * dx).clamp(max=xmax)

            def split(d):
                return d.clamp(min=0), (-d).clamp(min=0) * s * s

            def value(p, q, x):
                return float((p * x + q / x).sum())

            def best(p, q):
                return (q / p).sqrt()
        p0, q0 = split(df)
        p, q = split(dgs)
        bound = value(p, q, s) - vol
        l0, l1 = 0.0, prm.c
        for _ in range(100):
            lam = 0.5 * (l0 + l1)
            x = torch.minimum(torch.maximum(best(p0 + lam * p, q0 + lam * q), al), be)
            if value(p, q, x) > bound:
                l0 = lam
            else:
                l1 = lam
        old.append(s)
        s = x
    return dict(s=s.reshape(-1).cpu().numpy(), rho=project(g.filter(s)).reshape(-1).cpu().numpy(), f=np.array(fs),
                g=np.array(gs))


def exact(case, seed):
    if case["kind"] == "train":
        # the training pairs are made inside the library, and Adam turns
        # gradients that differ in their last bf16 digits into whole steps
        return None
    sh, dim, ne, n = _counts(case)
    its = (14 if dim == 2 else 27) * max(sh)
    if its * max(2.5e-4, (n if dim == 2 else 4 * n) * 2.5e-10) * case.get("iters", 1) > 18:
        return None  # the plain solve takes too long
    if case["kind"] == "loop":
        return _exact_loop(case, seed)
    g = _Grid(case)
    rho = torch.from_numpy(_density(case, seed)).cuda().reshape(g.sh)
    b = torch.zeros(math.prod(g.nodes) * dim, dtype=torch.float64, device="cuda")
    for nd, d, v in zip(*_loads(case, seed)):
        b[dim * int(nd) + int(d)] += float(v)
    u = g.solve(rho ** PENAL + E0 * (1 - rho ** PENAL), b.reshape(g.nodes + (dim,)))
    return None if u is None else u.reshape(-1)[g.fixed:].contiguous()
