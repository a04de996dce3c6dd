"""Python host mirror of the pansfem2_amd C ABI (include/pansfem2_amd.h).

Loads the in-tree libpansfem2_amd.so (built by __graft_entry__.build() /
`make -C pansfem2_amd/csrc`) and exposes the entry points under the names of
the reference routines they replace.  There is no fallback: if the library
is missing, or a call fails, an exception is raised.
"""
import ctypes
import os

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(HERE, "libpansfem2_amd.so")

PF_OK, PF_NOT_CONVERGED = 0, 1
PF_OP_CSR64, PF_OP_EBE64, PF_OP_EBE32, PF_OP_LEARNED, PF_OP_MG, PF_OP_MG32 = 0, 1, 2, 3, 4, 5
PF_FILTER_VARIABLES, PF_FILTER_SENSITIVITIES = 0, 1
PF_PCG_SCALINGCG, PF_PCG_SINGLE_REDUCTION = 0, 1
PF_PCG_SINGLE_REDUCTION_CARRIED, PF_PCG_SINGLE_REDUCTION_RECOMPUTED = 2, 3
PF_MG_PROLONG_BILINEAR, PF_MG_PROLONG_STIFFNESS = 0, 1
PF_MG_RESIDUAL_AUTO, PF_MG_RESIDUAL_NODE, PF_MG_RESIDUAL_ELEMENT = 0, 1, 2
PF_H8_OP_AUTO, PF_H8_OP_VALU, PF_H8_OP_MFMA = -1, 0, 1
PF_RESIDENT_AUTO, PF_RESIDENT_OFF, PF_RESIDENT_STALL, PF_RESIDENT_NOMEM, PF_RESIDENT_REFUSED = 0, 1, 2, 3, 4

_i32p = np.ctypeslib.ndpointer(np.int32, flags="C_CONTIGUOUS")
_f64p = np.ctypeslib.ndpointer(np.float64, flags="C_CONTIGUOUS")
_f32p = np.ctypeslib.ndpointer(np.float32, flags="C_CONTIGUOUS")


class PfError(RuntimeError):
    def __init__(self, code, msg):
        super().__init__(f"pansfem2_amd error {code}: {msg}")
        self.code = code


class SolveStats(ctypes.Structure):
    _fields_ = [("iterations", ctypes.c_int), ("status", ctypes.c_int), ("rel_residual", ctypes.c_double),
                ("true_residual", ctypes.c_double), ("seconds", ctypes.c_double), ("outer", ctypes.c_int),
                ("fallbacks", ctypes.c_int)]

    def as_dict(self):
        return {k: getattr(self, k) for k, _ in self._fields_}


class OcParams(ctypes.Structure):
    _fields_ = [(n, ctypes.c_double) for n in ("iota", "lambdamin", "lambdamax", "lambdaeps", "movelimit", "vf",
                                               "scale1")] + [("max_steps", ctypes.c_int), ("beta", ctypes.c_double)]


class MmaParams(ctypes.Structure):
    _fields_ = [("m", ctypes.c_int)] + [(n, ctypes.c_double) for n in (
        "a0", "a", "c", "d", "xmin", "xmax", "raa0", "albefa", "move", "asyinit", "asydecr", "asyincr",
        "epsvalue")] + [("max_newton", ctypes.c_int)]


class SimpParams(ctypes.Structure):
    _fields_ = [(n, ctypes.c_double) for n in ("E1", "E0", "nu", "t", "p", "vf", "R", "scale0", "scale1",
                                               "cg_eps")] + \
               [("cg_itrmax", ctypes.c_int), ("use_mma", ctypes.c_int), ("solver", ctypes.c_int),
                ("mixed", ctypes.c_int), ("inner_eps", ctypes.c_double), ("learned", ctypes.c_int),
                ("stop_on_convergence", ctypes.c_int), ("oc", OcParams), ("mma", MmaParams),
                ("collect", ctypes.c_int), ("collect_max", ctypes.c_int), ("heaviside", ctypes.c_int),
                ("beta0", ctypes.c_double), ("beta_factor", ctypes.c_double), ("beta_every", ctypes.c_int),
                ("iter_offset", ctypes.c_int), ("resume_optimizer", ctypes.c_int)]


class SimpHistory(ctypes.Structure):
    _fields_ = [("f", ctypes.c_void_p), ("g", ctypes.c_void_p), ("lambda_", ctypes.c_void_p),
                ("cg_iters", ctypes.c_void_p), ("bisect", ctypes.c_void_p), ("seconds", ctypes.c_void_p),
                ("iterations", ctypes.c_int), ("residual", ctypes.c_void_p), ("fallbacks", ctypes.c_void_p)]


_lib = None


def lib():
    """The loaded C library (raises if it has not been built)."""
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise ImportError(f"{LIB_PATH} is missing: build it with __graft_entry__.build() "
                              "or make -C pansfem2_amd/csrc")
        L = ctypes.CDLL(LIB_PATH)
        c_int, c_double, c_void_p, c_int64 = ctypes.c_int, ctypes.c_double, ctypes.c_void_p, ctypes.c_int64
        P = ctypes.POINTER
        sig = {
            "pf_create": ([P(c_void_p), c_int], c_int),
            "pf_destroy": ([c_void_p], c_int),
            "pf_last_error": ([c_void_p], ctypes.c_char_p),
            "pf_build_info": ([], ctypes.c_char_p),
            "pf_grid2d": ([c_void_p, c_int, c_int, c_double, c_double], c_int),
            "pf_grid3d": ([c_void_p, c_int, c_int, c_int, c_double, c_double, c_double], c_int),
            "pf_set_dirichlet": ([c_void_p, _i32p, _i32p, c_int, P(ctypes.c_int32)], c_int),
            "pf_get_dofmap": ([c_void_p, _i32p], c_int),
            "pf_set_point_loads": ([c_void_p, _i32p, _i32p, _f64p, c_int], c_int),
            "pf_get_load": ([c_void_p, _f64p], c_int),
            "pf_set_element_matrix": ([c_void_p, _f64p, c_int], c_int),
            "pf_element_stiffness": ([c_void_p, c_int, c_double, c_double, c_double, _f64p], c_int),
            "pf_set_material": ([c_void_p, c_double, c_double, c_double, c_double, c_double], c_int),
            "pf_set_density": ([c_void_p, _f64p], c_int),
            "pf_set_moduli": ([c_void_p, _f64p], c_int),
            "pf_assemble_csr": ([c_void_p, P(c_int64)], c_int),
            "pf_assemble_csr_elements": ([c_void_p, _f64p, P(c_int64)], c_int),
            "pf_get_csr": ([c_void_p, _i32p, _i32p, _f64p], c_int),
            "pf_apply_K": ([c_void_p, c_int, _f64p, _f64p], c_int),
            "pf_pcg": ([c_void_p, c_int, _f64p, _f64p, c_double, c_int, P(SolveStats)], c_int),
            "pf_pcg_dev": ([c_void_p, c_int, c_void_p, c_void_p, c_double, c_int, P(SolveStats)], c_int),
            "pf_set_pcg_form": ([c_void_p, c_int], c_int),
            "pf_set_resident": ([c_void_p, c_int, c_int], c_int),
            "pf_resident_runs": ([c_void_p, P(c_int64), P(c_int64)], c_int),
            "pf_set_h8_operator": ([c_void_p, c_int], c_int),
            "pf_mg_setup": ([c_void_p, c_int, c_double], c_int),
            "pf_mg_set_prolongation": ([c_void_p, c_int], c_int),
            "pf_mg_set_residual_form": ([c_void_p, c_int], c_int),
            "pf_mg_build": ([c_void_p], c_int),
            "pf_mg_apply": ([c_void_p, _f64p, _f64p], c_int),
            "pf_mg_level": ([c_void_p, c_int, P(c_int), P(c_int), P(c_int), P(c_int), c_void_p, c_void_p, c_void_p],
                            c_int),
            "pf_compliance_sens": ([c_void_p, _f64p, c_double, P(c_double), _f64p], c_int),
            "pf_compliance_sens_dev_noalloc": ([c_void_p, c_void_p, c_double, c_void_p, c_void_p], c_int),
            "pf_filter_setup": ([c_void_p, c_double], c_int),
            "pf_filter": ([c_void_p, c_int, _f64p, _f64p], c_int),
            "pf_filter_set_lists": ([c_void_p, _i32p, _i32p, _f64p], c_int),
            "pf_heaviside": ([c_void_p, c_double, c_int, _f64p, c_void_p, _f64p], c_int),
            "pf_sensitivity_filter": ([c_void_p, c_int, _f64p, _f64p, _f64p], c_int),
            "pf_oc_candidate": ([c_void_p, _f64p, _f64p, _f64p, c_double, c_double, c_double, _f64p], c_int),
            "pf_oc_update": ([c_void_p, _f64p, _f64p, _f64p, P(OcParams), P(c_double), P(c_int)], c_int),
            "pf_mma_init": ([c_void_p, P(MmaParams)], c_int),
            "pf_mma_update": ([c_void_p, _f64p, c_double, _f64p, c_double, _f64p, P(c_int)], c_int),
            "pf_mma_get_state": ([c_void_p, P(c_int), P(c_double), c_void_p, c_void_p, c_void_p, c_void_p], c_int),
            "pf_mma_set_state": ([c_void_p, c_int, c_double, _f64p, _f64p, _f64p, _f64p], c_int),
            "pf_conlin_init": ([c_void_p, P(MmaParams)], c_int),
            "pf_conlin_update": ([c_void_p, _f64p, c_double, _f64p, c_double, _f64p, P(c_int)], c_int),
            "pf_simp_run": ([c_void_p, P(SimpParams), c_int, _f64p, c_void_p, P(SimpHistory)], c_int),
            "pf_simp_default_params": ([P(SimpParams)], None),
            "pf_profile_kernels": ([c_void_p, c_int, c_int, _f64p], c_int),
            "pf_precond_init": ([c_void_p, c_int, ctypes.c_uint64], c_int),
            "pf_precond_num_params": ([c_void_p, P(c_int64)], c_int),
            "pf_precond_save": ([c_void_p, c_void_p, P(c_int64)], c_int),
            "pf_precond_load": ([c_void_p, _f32p, c_int64], c_int),
            "pf_precond_collect": ([c_void_p, c_int, c_int, P(c_int)], c_int),
            "pf_precond_collect_random": ([c_void_p, c_int, ctypes.c_uint64, P(c_int)], c_int),
            "pf_precond_train": ([c_void_p, c_int, c_double, ctypes.c_uint64, P(c_double), P(c_double)], c_int),
            "pf_precond_apply": ([c_void_p, _f64p, _f64p], c_int),
            "pf_precond_forward_raw": ([c_void_p, _f32p, _f32p], c_int),
            "pf_precond_forward_nodal": ([c_void_p, _f32p, _f64p], c_int),
            "pf_precond_backward_raw": ([c_void_p, _f32p, _f32p], c_int),
            "pf_conv_raw": ([c_void_p, c_int, c_int, c_int, c_int, c_int, c_int, _f32p, _f32p, _f32p], c_int),
        }
        for name, (args, res) in sig.items():
            fn = getattr(L, name)
            fn.argtypes = args
            fn.restype = res
        _lib = L
    return _lib


def simp_default_params(**kw):
    p = SimpParams()
    lib().pf_simp_default_params(ctypes.byref(p))
    for k, v in kw.items():
        if k.startswith("oc_"):
            setattr(p.oc, k[3:], v)
        elif k.startswith("mma_"):
            setattr(p.mma, k[4:], v)
        else:
            setattr(p, k, v)
    return p


def _f64(a):
    return np.ascontiguousarray(a, dtype=np.float64)


def _i32(a):
    return np.ascontiguousarray(a, dtype=np.int32)


class Context:
    """One pf_ctx: a device, a stream and the buffers of one grid."""

    def __init__(self, device=0):
        self._h = ctypes.c_void_p()
        rc = lib().pf_create(ctypes.byref(self._h), device)
        if rc != PF_OK:
            raise PfError(rc, "pf_create failed (no HIP device?)")
        self.N = 0
        self.nx = self.ny = self.nz = 0
        # status and message of the last call that returned PF_NOT_CONVERGED
        # (a warning with a valid result) through an allow_nc wrapper
        self.last_status = PF_OK
        self.last_message = ""

    def close(self):
        if self._h:
            lib().pf_destroy(self._h)
            self._h = ctypes.c_void_p()

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    def __enter__(self):
        return self

    def __exit__(self, *a):
        self.close()

    def _ck(self, rc, allow_nc=False):
        if rc == PF_OK or (allow_nc and rc == PF_NOT_CONVERGED):
            self.last_status = rc
            self.last_message = lib().pf_last_error(self._h).decode() if rc != PF_OK else ""
            return rc
        raise PfError(rc, lib().pf_last_error(self._h).decode())

    # ---- mesh / DOFs -----------------------------------------------------
    def grid2d(self, nx, ny, lx=None, ly=None):
        """SquareMesh(lx, ly, nx, ny) (SquareMesh.h:48-106)."""
        self._ck(lib().pf_grid2d(self._h, nx, ny, float(nx if lx is None else lx), float(ny if ly is None else ly)))
        self.nx, self.ny, self.dim, self.ndpn = nx, ny, 2, 2
        self.nn, self.ne = (nx + 1) * (ny + 1), nx * ny
        self.nd = 8
        return self

    def grid3d(self, nx, ny, nz, lx=None, ly=None, lz=None):
        self._ck(lib().pf_grid3d(self._h, nx, ny, nz, float(nx if lx is None else lx),
                                 float(ny if ly is None else ly), float(nz if lz is None else lz)))
        self.nx, self.ny, self.nz, self.dim, self.ndpn = nx, ny, nz, 3, 3
        self.nn, self.ne = (nx + 1) * (ny + 1) * (nz + 1), nx * ny * nz
        self.nd = 24
        return self

    def set_dirichlet(self, nodes, dofs):
        """SetDirichlet + Renumbering (BoundaryCondition.h:19-25, Assembling.h:175-186)."""
        nodes, dofs = _i32(nodes), _i32(dofs)
        n = ctypes.c_int32(0)
        self._ck(lib().pf_set_dirichlet(self._h, nodes, dofs, len(nodes), ctypes.byref(n)))
        self.N = n.value
        return self.N

    def dofmap(self):
        out = np.zeros(self.nn * self.ndpn, np.int32)
        self._ck(lib().pf_get_dofmap(self._h, out))
        return out

    def set_point_loads(self, nodes, dofs, values):
        """Assembling(F, qfixed, nodetoglobal) (Assembling.h:151-158)."""
        self._ck(lib().pf_set_point_loads(self._h, _i32(nodes), _i32(dofs), _f64(values), len(nodes)))

    def load(self):
        out = np.zeros(self.N)
        self._ck(lib().pf_get_load(self._h, out))
        return out

    # ---- element matrices / material ---------------------------------------
    def set_element_matrix(self, K0):
        K0 = _f64(K0)
        self._ck(lib().pf_set_element_matrix(self._h, K0.reshape(-1), K0.shape[0]))

    def element_stiffness(self, e, E=1.0, nu=0.3, t=1.0):
        """PlaneStrainStiffness for element e evaluated on the device in reference order."""
        nd = 8 if self.dim == 2 else 24
        out = np.zeros(nd * nd)
        self._ck(lib().pf_element_stiffness(self._h, e, E, nu, t, out))
        return out.reshape(nd, nd)

    def set_material(self, E1=1.0, E0=1e-9, p=3.0, nu=0.3, t=1.0):
        self._ck(lib().pf_set_material(self._h, E1, E0, p, nu, t))

    def set_density(self, rho):
        self._ck(lib().pf_set_density(self._h, _f64(rho)))

    def set_moduli(self, E):
        self._ck(lib().pf_set_moduli(self._h, _f64(E)))

    # ---- CSR check path ----------------------------------------------------
    def assemble_csr(self):
        nnz = ctypes.c_int64(0)
        self._ck(lib().pf_assemble_csr(self._h, ctypes.byref(nnz)))
        self.nnz = nnz.value
        return self.nnz

    def assemble_csr_elements(self, ke_all):
        """CSR from caller-given element matrices (ne x nd x nd)."""
        ke = np.ascontiguousarray(ke_all, dtype=np.float64).reshape(-1)
        assert ke.size == self.ne * self.nd * self.nd, "ke_all must hold ne x nd x nd values"
        nnz = ctypes.c_int64(0)
        self._ck(lib().pf_assemble_csr_elements(self._h, ke, ctypes.byref(nnz)))
        self.nnz = nnz.value
        return self.nnz

    def csr(self):
        ip = np.zeros(self.N + 1, np.int32)
        ix = np.zeros(max(self.nnz, 1), np.int32)
        dv = np.zeros(max(self.nnz, 1))
        self._ck(lib().pf_get_csr(self._h, ip, ix, dv))
        return ip, ix[:self.nnz], dv[:self.nnz]

    # ---- operators / solvers ----------------------------------------------
    def apply_K(self, x, op=PF_OP_EBE64):
        y = np.zeros(self.N)
        self._ck(lib().pf_apply_K(self._h, op, _f64(x), y))
        return y

    def mg_setup(self, nu=1, omega=0.0):
        """Geometric multigrid V-cycle as the flexible CG's base step
        (PF_OP_MG, and PF_OP_LEARNED's base); nu = 0 switches it off;
        omega <= 0: the element's default Jacobi weight (0.6 quad4, 0.4 hex8)."""
        self._ck(lib().pf_mg_setup(self._h, nu, omega))

    def mg_set_residual_form(self, form):
        """PF_MG_RESIDUAL_AUTO (the default), PF_MG_RESIDUAL_NODE or
        PF_MG_RESIDUAL_ELEMENT for the hex8 hierarchy's coarse levels."""
        self._ck(lib().pf_mg_set_residual_form(self._h, form))

    def mg_set_prolongation(self, mode):
        """PF_MG_PROLONG_BILINEAR or PF_MG_PROLONG_STIFFNESS (the default) for
        the quad4 hierarchy of this context."""
        self._ck(lib().pf_mg_set_prolongation(self._h, mode))

    def mg_build(self):
        self._ck(lib().pf_mg_build(self._h))

    def mg_apply(self, r):
        z = np.zeros(self.N)
        self._ck(lib().pf_mg_apply(self._h, _f64(r), z))
        return z

    def mg_level(self, level, want_ke=True):
        """(nx, ny, nz, Ke (ne x 8 x 8, or ne x 24 x 24 for hex8) or None, D, fix) of a built level."""
        nl, nx, ny, nz = ctypes.c_int(0), ctypes.c_int(0), ctypes.c_int(0), ctypes.c_int(0)
        refs = (ctypes.byref(nl), ctypes.byref(nx), ctypes.byref(ny), ctypes.byref(nz))
        self._ck(lib().pf_mg_level(self._h, level, *refs, None, None, None))
        h8 = nz.value > 0
        nn = (nx.value + 1) * (ny.value + 1) * (nz.value + 1 if h8 else 1)
        ne = nx.value * ny.value * (nz.value if h8 else 1)
        nd = 24 if h8 else 8
        ke = np.zeros((ne, nd, nd)) if (want_ke and level > 0) else None
        D = np.zeros((3 if h8 else 2) * nn, np.float32)
        fix = np.zeros(nn, np.uint8)
        self._ck(lib().pf_mg_level(self._h, level, *refs, ke.ctypes.data if ke is not None else None,
                                   D.ctypes.data, fix.ctypes.data))
        return dict(levels=nl.value, nx=nx.value, ny=ny.value, nz=nz.value, Ke=ke, D=D, fix=fix)

    def set_pcg_form(self, form):
        """PF_PCG_SCALINGCG (ScalingCG's order, the default) or a
        single-reduction form (one reduction per iteration) for the FP64 quad4
        matrix-free solves of this context: PF_PCG_SINGLE_REDUCTION_CARRIED
        (s = K p carried), PF_PCG_SINGLE_REDUCTION_RECOMPUTED (s = K p
        recomputed on a two-node halo) or PF_PCG_SINGLE_REDUCTION (the
        carried kernel while its working set stays below 150 MB)."""
        self._ck(lib().pf_set_pcg_form(self._h, form))

    def set_resident(self, mode, after=0):
        """PF_RESIDENT_AUTO (the default: one resident kernel per solve, MMA /
        CONLIN update and OC bisection where the grid fits the chip),
        PF_RESIDENT_OFF (always the launched kernels); for tests of the
        fallback PF_RESIDENT_STALL (resident launches after the first `after`
        of a solve end as stalled), PF_RESIDENT_NOMEM (the buffers they
        allocate after the first `after` cannot be had) and
        PF_RESIDENT_REFUSED (no cooperative launch is made)."""
        self._ck(lib().pf_set_resident(self._h, mode, after))

    def resident_runs(self):
        """(ended, gave way): resident solves, updates and bisections so far
        that ran to their end, and that stalled or were refused."""
        d, s = ctypes.c_int64(0), ctypes.c_int64(0)
        self._ck(lib().pf_resident_runs(self._h, ctypes.byref(d), ctypes.byref(s)))
        return d.value, s.value

    def set_h8_operator(self, kind):
        """PF_H8_OP_AUTO (the default: the resident kernel where the grid
        fits the chip, else PF_H8_OP_VALU), PF_H8_OP_VALU (one node per thread
        on the vector units) or PF_H8_OP_MFMA (the element matrix as a batched
        product on the matrix cores) for the hex8 Jacobi-PCG of this context."""
        self._ck(lib().pf_set_h8_operator(self._h, kind))

    def pcg(self, b, op=PF_OP_EBE64, eps=1e-10, itrmax=100000):
        """ScalingCG(K, b, itrmax, eps) (CG.h:419-453) on the device."""
        x = np.zeros(self.N)
        st = SolveStats()
        self._ck(lib().pf_pcg(self._h, op, _f64(b), x, eps, itrmax, ctypes.byref(st)), allow_nc=True)
        return x, st.as_dict()

    def pcg_dev(self, b_ptr, x_ptr, op=PF_OP_EBE64, eps=1e-10, itrmax=100000):
        st = SolveStats()
        self._ck(lib().pf_pcg_dev(self._h, op, ctypes.c_void_p(b_ptr), ctypes.c_void_p(x_ptr), eps, itrmax,
                                  ctypes.byref(st)), allow_nc=True)
        return st.as_dict()

    def compliance_sens(self, u, scale0=1.0):
        f = ctypes.c_double(0.0)
        d = np.zeros(self.ne)
        self._ck(lib().pf_compliance_sens(self._h, _f64(u), scale0, ctypes.byref(f), d))
        return f.value, d

    def compliance_sens_dev_noalloc(self, u_ptr, f_ptr, dfdrho_ptr, scale0=1.0):
        """pf_compliance_sens on device pointers (u: N, f: 1, dfdrho: ne) with
        no device allocation (the library's static scratch)."""
        self._ck(lib().pf_compliance_sens_dev_noalloc(self._h, ctypes.c_void_p(u_ptr), scale0,
                                                      ctypes.c_void_p(f_ptr), ctypes.c_void_p(dfdrho_ptr)))

    def filter_setup(self, R=1.5):
        self._ck(lib().pf_filter_setup(self._h, R))

    def filter_set_lists(self, ptr, idx, w):
        """DensityFilter(n, neighbors, w) with explicit lists (CSR-like)."""
        self._ck(lib().pf_filter_set_lists(self._h, np.ascontiguousarray(ptr, np.int32),
                                           np.ascontiguousarray(idx, np.int32), _f64(w)))

    def oc_candidate(self, x, dfdx, dgdx, lam, iota=0.5, movelimit=0.2):
        out = np.zeros(self.ne)
        self._ck(lib().pf_oc_candidate(self._h, _f64(x), _f64(dfdx), _f64(dgdx), lam, iota, movelimit, out))
        return out

    def filter(self, x, mode=PF_FILTER_VARIABLES):
        out = np.zeros(self.ne)
        self._ck(lib().pf_filter(self._h, mode, _f64(x), out))
        return out

    def sensitivity_filter(self, s, dfds, scheme=1):
        """SensitivityFilter (scheme 1) / SensitivityFilter2 (scheme 2)."""
        out = np.zeros(self.ne)
        self._ck(lib().pf_sensitivity_filter(self._h, scheme, _f64(s), _f64(dfds), out))
        return out

    def heaviside(self, beta, s, dfdrho=None):
        """HeavisideFilter at beta over the current filter: the projected
        filtered variables, or (with dfdrho) the filtered sensitivities."""
        out = np.zeros(self.ne)
        d = None if dfdrho is None else _f64(dfdrho)
        self._ck(lib().pf_heaviside(self._h, beta, 0 if d is None else 1, _f64(s),
                                    None if d is None else d.ctypes.data, out))
        return out

    def oc_update(self, x, dfdx, dgdx, iota=0.5, lambdamin=0.0, lambdamax=1e9, lambdaeps=1e-3, movelimit=0.2,
                  vf=0.5, scale1=1.0, max_steps=200, beta=0.0):
        """OC<T>::UpdateVariables (OC.h:76-107) with the filtered-volume closure
        (HeavisideFilter at beta when beta > 0)."""
        prm = OcParams(iota, lambdamin, lambdamax, lambdaeps, movelimit, vf, scale1, max_steps, beta)
        x = np.array(x, dtype=np.float64)
        lam = ctypes.c_double(0.0)
        steps = ctypes.c_int(0)
        self._ck(lib().pf_oc_update(self._h, x, _f64(dfdx), _f64(dgdx), ctypes.byref(prm), ctypes.byref(lam),
                                    ctypes.byref(steps)), allow_nc=True)
        return x, lam.value, steps.value

    def mma_init(self, **kw):
        p = simp_default_params().mma
        for k, v in kw.items():
            setattr(p, k, v)
        self._ck(lib().pf_mma_init(self._h, ctypes.byref(p)))

    def mma_update(self, x, f, dfdx, g, dgdx):
        x = np.array(x, dtype=np.float64)
        steps = ctypes.c_int(0)
        self._ck(lib().pf_mma_update(self._h, x, f, _f64(dfdx), g, _f64(dgdx), ctypes.byref(steps)), allow_nc=True)
        return x, steps.value

    def mma_get_state(self):
        """MMA<T>'s carried state (MMA.h:31-54): k, previousvalue, xkm1, xkm2, L, U."""
        k, pv = ctypes.c_int(0), ctypes.c_double(0.0)
        arrs = [np.zeros(self.ne) for _ in range(4)]
        self._ck(lib().pf_mma_get_state(self._h, ctypes.byref(k), ctypes.byref(pv), *[a.ctypes.data for a in arrs]))
        return dict(k=k.value, previousvalue=pv.value, xkm1=arrs[0], xkm2=arrs[1], L=arrs[2], U=arrs[3])

    def mma_set_state(self, st):
        self._ck(lib().pf_mma_set_state(self._h, int(st["k"]), float(st["previousvalue"]), _f64(st["xkm1"]),
                                        _f64(st["xkm2"]), _f64(st["L"]), _f64(st["U"])))

    def conlin_init(self, **kw):
        """CONLIN<T>(n, 1, a0, a, c, d, xmin, xmax) + SetParameters(move, epsvalue)."""
        p = simp_default_params().mma
        for k, v in kw.items():
            setattr(p, k, v)
        self._ck(lib().pf_conlin_init(self._h, ctypes.byref(p)))

    def conlin_update(self, x, f, dfdx, g, dgdx):
        x = np.array(x, dtype=np.float64)
        steps = ctypes.c_int(0)
        self._ck(lib().pf_conlin_update(self._h, x, f, _f64(dfdx), g, _f64(dgdx), ctypes.byref(steps)))
        return x, steps.value

    def profile_kernels(self, op=PF_OP_EBE64, reps=50):
        """Average device ms of the PCG operator kernel, the PCG vector kernel,
        the filter, one OC bisection step and the single-reduction PCG kernel
        (HIP events on the library stream)."""
        ms = np.zeros(5)
        self._ck(lib().pf_profile_kernels(self._h, op, reps, ms))
        return dict(k1_ms=ms[0], k2_ms=ms[1], filter_ms=ms[2], oc_step_ms=ms[3], cg1_ms=ms[4])

    # ---- learned preconditioner ----------------------------------------------
    def precond_init(self, seed=20261204):
        self._ck(lib().pf_precond_init(self._h, 16, seed))

    def precond_num_params(self):
        n = ctypes.c_int64(0)
        self._ck(lib().pf_precond_num_params(self._h, ctypes.byref(n)))
        return n.value

    def precond_save(self):
        out = np.zeros(self.precond_num_params(), np.float32)
        n = ctypes.c_int64(0)
        self._ck(lib().pf_precond_save(self._h, out.ctypes.data, ctypes.byref(n)))
        return out

    def precond_load(self, params):
        params = np.ascontiguousarray(params, np.float32)
        self._ck(lib().pf_precond_load(self._h, params, len(params)))

    def precond_collect(self, every=8, max_pairs=32):
        n = ctypes.c_int(0)
        self._ck(lib().pf_precond_collect(self._h, every, max_pairs, ctypes.byref(n)))
        return n.value

    def precond_collect_random(self, count, seed=1):
        n = ctypes.c_int(0)
        self._ck(lib().pf_precond_collect_random(self._h, count, seed, ctypes.byref(n)))
        return n.value

    def precond_train(self, steps, lr=1e-3, seed=1):
        a, b = ctypes.c_double(0), ctypes.c_double(0)
        self._ck(lib().pf_precond_train(self._h, steps, lr, seed, ctypes.byref(a), ctypes.byref(b)))
        return a.value, b.value

    def precond_apply(self, r):
        d = np.zeros(self.N)
        self._ck(lib().pf_precond_apply(self._h, _f64(r), d))
        return d

    def precond_forward_raw(self, x0):
        x0 = np.ascontiguousarray(x0, np.float32).reshape(-1)
        y = np.zeros_like(x0)
        self._ck(lib().pf_precond_forward_raw(self._h, x0, y))
        return y

    def precond_forward_nodal(self, x0):
        """The network's output channels 0 .. ndpn-1 as a nodal FP64 vector,
        zero at fixed DOFs (the form the solver consumes)."""
        x0 = np.ascontiguousarray(x0, np.float32).reshape(-1)
        y = np.zeros(self.nn * self.ndpn)
        self._ck(lib().pf_precond_forward_nodal(self._h, x0, y))
        return y

    def precond_backward_raw(self, dy):
        dy = np.ascontiguousarray(dy, np.float32).reshape(-1)
        g = np.zeros(self.precond_num_params(), np.float32)
        self._ck(lib().pf_precond_backward_raw(self._h, dy, g))
        return g

    def conv_raw(self, x, w, cout=None):
        """One network convolution on the device: x (H, W[, D], cin), w
        (taps, cout, cin) -> y (H, W[, D], cout), FP32."""
        x = np.ascontiguousarray(x, np.float32)
        w = np.ascontiguousarray(w, np.float32)
        sp = x.shape[:-1]
        cin, cout = x.shape[-1], w.shape[1]
        y = np.zeros(sp + (cout,), np.float32)
        Dp = sp[2] if len(sp) == 3 else 0
        self._ck(lib().pf_conv_raw(self._h, 0, cin, cout, sp[0], sp[1], Dp, x.reshape(-1), w.reshape(-1),
                                   y.reshape(-1)))
        return y

    def conv_wgrad_raw(self, x, dz):
        """Weight gradient of one network convolution on the device:
        [tap][cout][cin] = sum_p dz[p][cout] x[p + tap][cin]."""
        x = np.ascontiguousarray(x, np.float32)
        dz = np.ascontiguousarray(dz, np.float32)
        sp = x.shape[:-1]
        cin, cout = x.shape[-1], dz.shape[-1]
        ntap = 3 ** len(sp)
        g = np.zeros((ntap, cout, cin), np.float32)
        Dp = sp[2] if len(sp) == 3 else 0
        self._ck(lib().pf_conv_raw(self._h, 1, cin, cout, sp[0], sp[1], Dp, x.reshape(-1), dz.reshape(-1),
                                   g.reshape(-1)))
        return g

    def simp_run(self, iters, params=None, s0=0.5):
        """The device-resident SIMP loop (sample_optimize_density_oc.cpp:83-208)."""
        params = params or simp_default_params()
        s = np.full(self.ne, s0) if np.isscalar(s0) else np.array(s0, dtype=np.float64)
        rho = np.zeros(self.ne)
        h = {k: np.zeros(iters) for k in ("f", "g", "lambda", "seconds", "residual")}
        h["cg_iters"] = np.zeros(iters, np.int32)
        h["bisect"] = np.zeros(iters, np.int32)
        h["fallbacks"] = np.zeros(iters, np.int32)
        H = SimpHistory(h["f"].ctypes.data, h["g"].ctypes.data, h["lambda"].ctypes.data, h["cg_iters"].ctypes.data,
                        h["bisect"].ctypes.data, h["seconds"].ctypes.data, 0, h["residual"].ctypes.data,
                        h["fallbacks"].ctypes.data)
        rc = self._ck(lib().pf_simp_run(self._h, ctypes.byref(params), iters, s, rho.ctypes.data, ctypes.byref(H)),
                      allow_nc=True)
        n = H.iterations
        return dict(s=s, rho=rho, status=rc, message=self.last_message, **{k: v[:n] for k, v in h.items()})


def cantilever2d(nx, ny, device=0, ctx=None, E1=1.0, E0=1e-9, p=3.0, nu=0.3, t=1.0, R=1.5):
    """The SIMP workload's grid: SquareMesh(nx, ny, nx, ny), left edge clamped,
    unit downward load at the bottom-right node, K0 = element 0 at E = 1."""
    ctx = ctx or Context(device)
    ctx.grid2d(nx, ny, float(nx), float(ny))
    nodes = np.repeat(np.arange(ny + 1, dtype=np.int32), 2)
    dofs = np.tile(np.array([0, 1], np.int32), ny + 1)
    ctx.set_dirichlet(nodes, dofs)
    ctx.set_point_loads([(ny + 1) * nx], [1], [-1.0])
    ctx.set_material(E1, E0, p, nu, t)
    ctx.set_element_matrix(ctx.element_stiffness(0, 1.0, nu, t))
    ctx.filter_setup(R)
    return ctx


def line_load_nodes3d(nx, ny, nz, total=-1.0):
    """Unit line load along the bottom edge (y = 0) of the x = max face,
    split consistently over the edge's nz + 1 nodes (end nodes half)."""
    nodes = np.array([(ny + 1) * (nz + 1) * nx + k for k in range(nz + 1)], np.int32)
    vals = np.full(nz + 1, total / nz)
    vals[0] *= 0.5
    vals[-1] *= 0.5
    return nodes, np.ones(nz + 1, np.int32), vals


def cantilever3d(nx, ny, nz, device=0, ctx=None, E1=1.0, E0=1e-9, p=3.0, nu=0.3, R=1.5):
    """Hex8 SIMP grid: x = 0 face clamped, unit line load on the bottom edge
    of the x = max face (-y), K0 = element 0 at E = 1."""
    ctx = ctx or Context(device)
    ctx.grid3d(nx, ny, nz, float(nx), float(ny), float(nz))
    face = np.arange((ny + 1) * (nz + 1), dtype=np.int32)
    ctx.set_dirichlet(np.repeat(face, 3), np.tile(np.arange(3, dtype=np.int32), len(face)))
    ctx.set_point_loads(*line_load_nodes3d(nx, ny, nz))
    ctx.set_material(E1, E0, p, nu, 1.0)
    ctx.set_element_matrix(ctx.element_stiffness(0, 1.0, nu))
    ctx.filter_setup(R)
    return ctx
