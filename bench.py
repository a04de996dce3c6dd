"""Benchmark of the SIMP topology-optimisation loop on one MI355X.

Workload: plane-strain SIMP compliance minimisation on a 1024 x 512 grid of
unit quad4 elements (524,288 elements, 1,050,624 free DOFs): left edge
clamped, unit downward load at the bottom-right node, E1 = 1, E0 = 1e-9,
nu = 0.3, p = 3, volume fraction 0.5, density filter R = 1.5, FP64
matrix-free Jacobi-PCG to a 1e-10 recursive residual, OC update (move 0.2,
damping 0.5).  A step is one OC iteration (filter, volume, moduli, PCG solve,
compliance and sensitivities, filtered sensitivities, OC bisection).  The
PCG runs in its single-reduction form (one reduction per iteration, the same
iterates as ScalingCG's order in exact arithmetic), resident on the chip; the
loop is timed again with ScalingCG's own order beside it.

Prints one JSON line: OC iterations/sec over the timed steps, the roofline
of the dominant kernel measured live with HIP events, the PCG
time-to-1e-8-residual of the solvers on the final design, and the reference
(compiled from its own sources, g++ -O3 -fopenmp) timed on a bounded sample
of the same iteration on this host's cores.
"""
import argparse
import json
import os
import subprocess
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK_GBS = 8000.0
FP64_PEAK_TFLOPS = 78.6


def cpu_baseline(nx, ny, n_cg, n_bis, cg_sample=2000, oc_sample=30):
    """Reference build (oracle/_ref/ref_harness) on one OC iteration, bounded:
    ScalingCG capped at `cg_sample` iterations, OC bisection at `oc_sample`
    steps; per-iteration/per-step times are scaled to the GPU run's mean CG
    iterations and bisection steps."""
    exe = os.path.join(ROOT, "oracle", "_ref", "ref_harness")
    if not os.path.exists(exe):
        return None
    cores = int(os.environ.get("OMP_NUM_THREADS", os.cpu_count() or 1))
    env = dict(os.environ, OMP_NUM_THREADS=str(cores), OMP_PROC_BIND="close")
    t0 = time.time()
    out = subprocess.run([exe, "time", str(nx), str(ny), str(cg_sample), str(oc_sample)], capture_output=True,
                         text=True, env=env, timeout=600)
    wall = time.time() - t0
    line = [l for l in out.stdout.splitlines() if l.startswith("{")]
    if out.returncode != 0 or not line:
        return None
    t = json.loads(line[-1])
    per_cg = t["cg_s"] / t["cg_itrmax"]
    per_step = t["oc_s"] / max(1, t["oc_steps"])
    it_s = (t["filter_s"] + t["assemble_s"] + t["csr_s"] + per_cg * n_cg + t["sens_s"] + t["sens_filter_s"]
            + per_step * n_bis)
    return {
        "value": 1.0 / it_s, "unit": "OC iters/sec", "cores": cores, "kind": "reference",
        "sample": (f"reference (g++ -O3 -fopenmp, {cores} OpenMP threads) on OC iteration 0 at {nx}x{ny}: "
                   f"assembly+CSR+reactions/sensitivities+filters timed in full, ScalingCG {cg_sample} iterations "
                   f"({per_cg * 1e3:.2f} ms each) and OC {oc_sample} bisection steps ({per_step * 1e3:.2f} ms each) "
                   f"scaled to the GPU run's mean {n_cg:.0f} CG iterations and {n_bis:.1f} steps; sample wall "
                   f"{wall:.1f} s"),
        "phases_s": {k: t[k] for k in ("filter_s", "assemble_s", "csr_s", "sens_s", "sens_filter_s")},
        "cg_iter_ms": per_cg * 1e3, "oc_step_ms": per_step * 1e3,
    }


def ref_harness_time(args, timeout=1800):
    """One run of the reference build's timing mode (oracle/_ref/ref_harness
    time ...) on this host's cores; its JSON line, or None."""
    exe = os.path.join(ROOT, "oracle", "_ref", "ref_harness")
    if not os.path.exists(exe):
        return None
    cores = int(os.environ.get("OMP_NUM_THREADS", os.cpu_count() or 1))
    env = dict(os.environ, OMP_NUM_THREADS=str(cores), OMP_PROC_BIND="close")
    t0 = time.time()
    out = subprocess.run([exe, "time"] + [str(a) for a in args], capture_output=True, text=True, env=env,
                         timeout=timeout)
    line = [l for l in out.stdout.splitlines() if l.startswith("{")]
    if out.returncode != 0 or not line:
        return None
    t = json.loads(line[-1])
    t["wall_s"] = time.time() - t0
    t["cores"] = cores
    return t


def cpu_reference_runs():
    """The reference's own timings that the bounded baseline scales from,
    measured in full once: the 120 x 40 loop's 50 OC iterations per phase,
    the 1024 x 512 iteration-0 system's ScalingCG to 1e-8 and to 1e-10 (one
    whole solve each), and one MMA update on that iteration's sensitivities."""
    out = {"cpu_model": None, "nproc": os.cpu_count()}
    try:
        for l in open("/proc/cpuinfo"):
            if l.startswith("model name"):
                out["cpu_model"] = l.split(":", 1)[1].strip()
                break
    except OSError:
        pass
    print("cpu reference: 120x40, 50 OC iterations", file=sys.stderr, flush=True)
    out["c1_loop_50"] = ref_harness_time([120, 40, 100000, 10 ** 9, 50, 1e-10])
    for eps in (1e-8, 1e-10):
        print(f"cpu reference: 1024x512 iteration 0, ScalingCG to {eps:g}", file=sys.stderr, flush=True)
        out[f"c2_iteration0_scalingcg_{eps:g}"] = ref_harness_time([1024, 512, 100000, 1, 1, eps])
    print("cpu reference: 1024x512 iteration 0 with the MMA update", file=sys.stderr, flush=True)
    out["c2_iteration0_mma"] = ref_harness_time([1024, 512, 100000, 1, 1, 1e-10, "mma"])
    return out


def c2_loops(pa, torch, nx=1024, ny=512, iters=100):
    """The whole 1024 x 512 workload once: 100 OC iterations and the MMA
    variant's 100 iterations, both with FP64 matrix-free Jacobi-PCG to 1e-10
    (single-reduction form), timed whole from the uniform design."""
    out = {}
    for label, kw in (("oc_jacobi", {}), ("mma_jacobi", {"use_mma": 1})):
        ctx = pa.cantilever2d(nx, ny)
        ctx.set_pcg_form(pa.PF_PCG_SINGLE_REDUCTION)
        print(f"c2 loop: {label}, {iters} iterations", file=sys.stderr, flush=True)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        r = ctx.simp_run(iters, pa.simp_default_params(**kw))
        torch.cuda.synchronize()
        wall = time.perf_counter() - t0
        out[label] = {"iterations": int(len(r["f"])), "seconds": wall, "oc_iters_per_s": len(r["f"]) / wall,
                      "cg_iterations": int(np.sum(r["cg_iters"])), "mean_cg_iters": float(np.mean(r["cg_iters"])),
                      "compliance_first_last": [float(r["f"][0]), float(r["f"][-1])],
                      "volume_last": float(np.mean(r["rho"])), "status": int(r["status"])}
        ctx.close()
    return out


def kernels_only(ctx, pa, torch, nx, ny, reps=20, copy_mib=256):
    """The PCG operator and vector kernels, the filter and the OC step on a
    density field drawn i.i.d. uniform in [1e-3, 1] (seed 20261202), then one
    device-to-device copy of `copy_mib` MiB: the copy's counter readings
    calibrate the byte counters (it reads and writes exactly copy_mib MiB)."""
    rng = np.random.default_rng(20261202)
    ctx.set_density(rng.uniform(1e-3, 1.0, ctx.ne))
    prof = ctx.profile_kernels(pa.PF_OP_EBE64, reps=reps)
    src = torch.ones(copy_mib * 2**20 // 4, dtype=torch.float32, device="cuda")
    dst = torch.empty_like(src)
    torch.cuda.synchronize()
    dst.copy_(src)
    torch.cuda.synchronize()
    print(json.dumps({"kernels_only": True, "nx": nx, "ny": ny, "reps": reps, "copy_bytes": copy_mib * 2**20,
                      "N": ctx.N, "ne": ctx.ne, "kernels_ms": prof}))


def form_sweep(pa, sizes=((1024, 512), (1280, 640), (1536, 768), (1792, 896), (2048, 1024)), iters=2000):
    """Device time per FP64 Jacobi-PCG iteration of ScalingCG's order and of
    the two single-reduction kernels, on quad4 cantilevers of several sizes
    (density i.i.d. uniform in [1e-3, 1], seed 20261202; best of three solves
    of `iters` iterations each): where the carried kernel's working set
    leaves the last-level cache, the recomputing kernel takes over."""
    forms = (("scalingcg", pa.PF_PCG_SCALINGCG), ("carried", pa.PF_PCG_SINGLE_REDUCTION_CARRIED),
             ("recomputed", pa.PF_PCG_SINGLE_REDUCTION_RECOMPUTED))
    for nx, ny in sizes:
        ctx = pa.cantilever2d(nx, ny)
        ctx.set_density(np.random.default_rng(20261202).uniform(1e-3, 1.0, ctx.ne))
        b = ctx.load()
        nv = 2 * (nx + 1) * (ny + 1)
        row = {"nx": nx, "ny": ny, "carried_working_set_MB": round(8 * (9 * nv + ctx.ne) / 1e6, 1)}
        for name, form in forms:
            ctx.set_pcg_form(form)
            best = min(ctx.pcg(b, op=pa.PF_OP_EBE64, eps=1e-30, itrmax=iters)[1]["seconds"] for _ in range(3))
            row[name + "_us_per_iteration"] = round(best / iters * 1e6, 2)
        print(json.dumps(row), flush=True)
        ctx.close()


def h8_operators(pa, nx=128, ny=64, nz=64, iters=500):
    """The hex8 fused PCG kernel with each operator kernel (vector units,
    matrix cores) at C5's 128x64x64 (density i.i.d. uniform in [1e-2, 1],
    seed 20261203): FP64 Jacobi-PCG for `iters` iterations (best of three
    solves, device time per iteration) and the mixed solve (FP32 inner PCG,
    FP64 refinement) to a 1e-8 true residual.  The kernels' own durations come
    from a kernel trace of this program."""
    ctx = pa.cantilever3d(nx, ny, nz)
    ctx.set_density(np.random.default_rng(20261203).uniform(1e-2, 1.0, ctx.ne))
    b = ctx.load()
    out = {"nx": nx, "ny": ny, "nz": nz}
    xs = {}
    for name, kind in (("valu", pa.PF_H8_OP_VALU), ("mfma", pa.PF_H8_OP_MFMA)):
        ctx.set_h8_operator(kind)
        best = min(ctx.pcg(b, op=pa.PF_OP_EBE64, eps=1e-30, itrmax=iters)[1]["seconds"] for _ in range(3))
        x, st = ctx.pcg(b, op=pa.PF_OP_EBE64, eps=1e-8)
        x32, s32 = ctx.pcg(b, op=pa.PF_OP_EBE32, eps=1e-8)
        xs[name] = x
        out[name] = {"fp64_us_per_iteration": round(best / iters * 1e6, 2),
                     "fp64_to_1e-8": {"seconds": st["seconds"], "iterations": st["iterations"]},
                     "mixed_to_1e-8": {"seconds": s32["seconds"], "inner_iterations": s32["iterations"],
                                       "outer": s32["outer"], "true_residual": s32["true_residual"]}}
    out["fp64_solution_rel_diff"] = float(np.linalg.norm(xs["mfma"] - xs["valu"]) / np.linalg.norm(xs["valu"]))
    ctx.close()
    return out


def conv_kernels(pa, nx=1024, ny=512, pairs=32, steps=20, applies=20):
    """The learned preconditioner's kernels at 1024x512 on their own (for
    kernel traces and counter runs, whose full workload is too long to trace
    with counters): `pairs` synthetic training pairs, `steps` Adam steps, then
    `applies` network applications to a residual, on a density field i.i.d.
    uniform in [1e-3, 1] (seed 20261203)."""
    ctx = pa.cantilever2d(nx, ny)
    ctx.set_density(np.random.default_rng(20261203).uniform(1e-3, 1.0, ctx.ne))
    ctx.precond_init(seed=11)
    ctx.precond_collect_random(pairs)
    t0 = time.perf_counter()
    loss0, loss1 = ctx.precond_train(steps, lr=2e-3, seed=17)
    t_train = time.perf_counter() - t0
    r = ctx.load()
    t0 = time.perf_counter()
    for _ in range(applies):
        y = ctx.precond_apply(r)
    t_apply = time.perf_counter() - t0
    ctx.close()
    return {"nx": nx, "ny": ny, "pairs": pairs, "steps": steps, "train_seconds": t_train, "loss": [loss0, loss1],
            "applies": applies, "apply_seconds_each": t_apply / applies, "y_finite": bool(np.all(np.isfinite(y)))}


def other_configs(pa):
    """The other full-size workloads, timed once each on one GPU (their
    parity is in tests/test_gpu_fullsize.py): 2048x1024 quad4 on a density
    field i.i.d. uniform in [1e-3, 1] (seed 20261204) -- FP64 Jacobi-PCG to
    1e-8 (the single-reduction form, which at this size runs the recomputing
    kernel), the mixed-precision solve (FP32 inner PCG inside FP64 refinement)
    to a 1e-8 FP64 true residual, multigrid PCG to 1e-8 with FP64 vectors and
    with FP32 ones inside FP64 refinement (PF_OP_MG32); 128x64x64 hex8 on an
    i.i.d. field (seed 20261205) -- the same solves, then 10 OC
    iterations of the hex8 SIMP loop (volume fraction 0.3) with multigrid
    solves to 1e-10 from the uniform start."""
    def solve(ctx, b, op):
        x, st = ctx.pcg(b, op=op, eps=1e-8)
        return x, {"seconds": st["seconds"], "iterations": st["iterations"], "true_residual": st["true_residual"],
                   "status": st["status"], "outer": st["outer"], "fallbacks": st.get("fallbacks", 0)}

    def three(ctx, b):
        ctx.mg_setup(1)
        out = {}
        x64, out["jacobi_fp64"] = solve(ctx, b, pa.PF_OP_EBE64)
        x32, out["mixed_fp32_ir"] = solve(ctx, b, pa.PF_OP_EBE32)
        ctx.pcg(b, op=pa.PF_OP_MG, eps=1e-8)  # the hierarchy's allocations
        xmg, out["multigrid_pcg"] = solve(ctx, b, pa.PF_OP_MG)
        xmg32, out["multigrid_fp32_ir"] = solve(ctx, b, pa.PF_OP_MG32)
        c64 = float(x64 @ b)
        out["multigrid_fp32_ir_rel_diff_compliance"] = abs(float(xmg32 @ b) - c64) / abs(c64)
        out["speedup_multigrid_fp32_ir_vs_multigrid"] = (out["multigrid_pcg"]["seconds"] /
                                                         out["multigrid_fp32_ir"]["seconds"])
        out["mixed_rel_diff_u"] = float(np.linalg.norm(x32 - x64) / np.linalg.norm(x64))
        out["mixed_rel_diff_compliance"] = abs(float(x32 @ b) - c64) / abs(c64)
        out["multigrid_rel_diff_compliance"] = abs(float(xmg @ b) - c64) / abs(c64)
        out["speedup_multigrid_vs_jacobi"] = out["jacobi_fp64"]["seconds"] / out["multigrid_pcg"]["seconds"]
        out["speedup_mixed_vs_jacobi"] = out["jacobi_fp64"]["seconds"] / out["mixed_fp32_ir"]["seconds"]
        return out

    res = {}
    ctx = pa.cantilever2d(2048, 1024)
    ctx.set_pcg_form(pa.PF_PCG_SINGLE_REDUCTION)
    ctx.set_density(np.random.default_rng(20261204).uniform(1e-3, 1.0, 2048 * 1024))
    res["quad4_2048x1024_iid"] = three(ctx, ctx.load())
    ctx.close()
    nx, ny, nz = 128, 64, 64
    ctx = pa.cantilever3d(nx, ny, nz)
    ctx.set_density(np.random.default_rng(20261205).uniform(1e-3, 1.0, nx * ny * nz))
    res["hex8_128x64x64_iid"] = three(ctx, ctx.load())
    ctx.simp_run(2, pa.simp_default_params(vf=0.3, solver=pa.PF_OP_MG), s0=0.3)  # warm-up
    t0 = time.perf_counter()
    r = ctx.simp_run(10, pa.simp_default_params(vf=0.3, solver=pa.PF_OP_MG), s0=0.3)
    dt = time.perf_counter() - t0
    res["hex8_128x64x64_simp_multigrid"] = {
        "oc_iterations": 10, "seconds": dt, "oc_iters_per_s": 10 / dt,
        "mean_cg_iters": float(np.mean(r["cg_iters"])),
        "compliance_first_last": [float(r["f"][0]), float(r["f"][-1])]}
    ctx.close()
    return res


def stream_copy_gbs(torch, mib=256, reps=20):
    """STREAM-like device-to-device copy of `mib` MiB on torch's stream, timed
    with events: bytes read + written per second, the bandwidth a plain
    streaming kernel reaches on this GPU.  At 256 MiB the copy streams from
    and to HBM; at half the working set of a cache-resident kernel (source
    plus destination as large as that working set) it runs from the 256 MB
    last-level cache, as that kernel does."""
    src = torch.ones(int(mib * 2**20) // 4, dtype=torch.float32, device="cuda")
    dst = torch.empty_like(src)
    dst.copy_(src)
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record()
    for _ in range(reps):
        dst.copy_(src)
    e1.record()
    torch.cuda.synchronize()
    sec = e0.elapsed_time(e1) * 1e-3 / reps
    return 2 * (int(mib * 2**20) // 4) * 4 / sec / 1e9


def learned_vs_jacobi(pa, nx, ny, train_iters=30, collect_every=20, collect_max=16, steps=500, lr=2e-3):
    """Learned-preconditioner workload: the network is trained on (residual,
    error) pairs that the plain FP64 Jacobi-PCG produces during the first
    `train_iters` OC iterations (every `collect_every` chunks of 32 CG
    iterations, at most `collect_max` per solve), plus 120 synthetic (K v, v)
    pairs, as a correction over the multigrid V-cycle (FP32); then three
    solvers take the system of a later OC iteration to a 1e-8 FP64 true
    relative residual: plain FP64 Jacobi-PCG, PCG with the V-cycle alone
    (PF_OP_MG), and flexible CG with the network over the V-cycle.  Then the
    run's OC iterations 35-100 are repeated from the same state with each of
    the three solvers (to 1e-8) and timed whole."""
    ctx = pa.cantilever2d(nx, ny)
    ctx.set_pcg_form(pa.PF_PCG_SINGLE_REDUCTION)  # the Jacobi leg at its fastest
    ctx.precond_init(seed=11)
    ctx.mg_setup(1, 0.6)
    t0 = time.perf_counter()
    r = ctx.simp_run(train_iters, pa.simp_default_params(collect=collect_every, collect_max=collect_max))
    t_collect = time.perf_counter() - t0
    s = r["s"]
    for k in range(3):
        rr = ctx.simp_run(1, pa.simp_default_params(), s0=s)
        s = rr["s"]
        ctx.set_density(rr["rho"])
        pairs = ctx.precond_collect_random(40, seed=100 + k)
    t0 = time.perf_counter()
    loss0, loss1 = ctx.precond_train(steps, lr=lr, seed=17)
    t_train = time.perf_counter() - t0
    rr = ctx.simp_run(1, pa.simp_default_params(), s0=s)
    s34 = rr["s"]
    ctx.set_density(rr["rho"])
    b = ctx.load()
    out = {"design": f"OC iteration {train_iters + 4} of the {nx}x{ny} loop", "pairs": pairs,
           "train_steps": steps, "loss_first": loss0, "loss_last": loss1, "train_seconds": t_train,
           "collect_oc_seconds": t_collect}
    comp = {}
    for label, op in (("jacobi_fp64", pa.PF_OP_EBE64), ("multigrid_pcg", pa.PF_OP_MG),
                      ("learned_fcg", pa.PF_OP_LEARNED)):
        x, st = ctx.pcg(b, op=op, eps=1e-8)  # untimed first call: allocations
        x, st = ctx.pcg(b, op=op, eps=1e-8)
        comp[label] = float(x @ b)  # u^T K u = u^T f
        out[label] = {"seconds": st["seconds"], "iterations": st["iterations"], "true_residual": st["true_residual"],
                      "status": st["status"], "fallbacks": st["fallbacks"]}
    # the V-cycle with bilinear prolongation (the geometric hierarchy the
    # stiffness-weighted one replaces), on the same system
    ctx.mg_set_prolongation(pa.PF_MG_PROLONG_BILINEAR)
    x, st = ctx.pcg(b, op=pa.PF_OP_MG, eps=1e-8)
    x, st = ctx.pcg(b, op=pa.PF_OP_MG, eps=1e-8)
    out["multigrid_pcg_bilinear"] = {"seconds": st["seconds"], "iterations": st["iterations"],
                                     "true_residual": st["true_residual"], "status": st["status"]}
    ctx.mg_set_prolongation(pa.PF_MG_PROLONG_STIFFNESS)
    # multigrid PCG in FP32 inside FP64 iterative refinement (PF_OP_MG32)
    x, st = ctx.pcg(b, op=pa.PF_OP_MG32, eps=1e-8)
    x, st = ctx.pcg(b, op=pa.PF_OP_MG32, eps=1e-8)
    out["multigrid_fp32_ir"] = {"seconds": st["seconds"], "iterations": st["iterations"], "outer": st["outer"],
                                "fallbacks": st["fallbacks"], "true_residual": st["true_residual"],
                                "status": st["status"],
                                "compliance_rel_diff": abs(float(x @ b) - comp["jacobi_fp64"]) / abs(comp["jacobi_fp64"])}
    out["speedup_learned_vs_jacobi"] = out["jacobi_fp64"]["seconds"] / out["learned_fcg"]["seconds"]
    out["speedup_multigrid_vs_jacobi"] = out["jacobi_fp64"]["seconds"] / out["multigrid_pcg"]["seconds"]
    out["iteration_ratio"] = out["learned_fcg"]["iterations"] / out["jacobi_fp64"]["iterations"]
    out["network_gain_iterations"] = out["multigrid_pcg"]["iterations"] / out["learned_fcg"]["iterations"]
    out["compliance_rel_diff"] = abs(comp["learned_fcg"] - comp["jacobi_fp64"]) / abs(comp["jacobi_fp64"])
    out["compliance_rel_diff_multigrid"] = abs(comp["multigrid_pcg"] - comp["jacobi_fp64"]) / abs(comp["jacobi_fp64"])
    # the rest of the run, OC iterations 35-100, from the same state with each
    # solver to 1e-8: whole OC iterations timed (solve, filter, OC)
    loop = {}
    for label, kw in (("jacobi_fp64", {}), ("multigrid_pcg", {"solver": pa.PF_OP_MG}),
                      ("learned_fcg", {"learned": 1})):
        h = ctx.simp_run(66, pa.simp_default_params(cg_eps=1e-8, **kw), s0=s34)
        loop[label] = {"seconds": float(np.sum(h["seconds"])), "cg_iterations": int(np.sum(h["cg_iters"])),
                       "compliance_last": float(h["f"][-1])}
    for label in ("multigrid_pcg", "learned_fcg"):
        loop[label]["speedup_vs_jacobi"] = loop["jacobi_fp64"]["seconds"] / loop[label]["seconds"]
        loop[label]["compliance_rel_diff"] = (abs(loop[label]["compliance_last"] - loop["jacobi_fp64"]["compliance_last"])
                                              / loop["jacobi_fp64"]["compliance_last"])
    out["oc_iterations_35_100"] = loop
    ctx.close()
    return out


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=10)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--repeats", type=int, default=3,
                    help="timed windows of --steps OC iterations, each from the same warmed design; "
                         "value is the median")
    ap.add_argument("--nx", type=int, default=1024)
    ap.add_argument("--ny", type=int, default=512)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-extras", action="store_true")
    ap.add_argument("--no-learned", action="store_true", help="skip the learned-preconditioner comparison")
    ap.add_argument("--no-others", action="store_true",
                    help="skip the 2048x1024 and 128x64x64 solves and the hex8 loop (other_configs)")
    ap.add_argument("--save-design", metavar="NPY",
                    help="run --design-iters OC iterations of the Jacobi-PCG loop, save the densities, exit")
    ap.add_argument("--design-iters", type=int, default=34)
    ap.add_argument("--mg-solve", metavar="NPY",
                    help="multigrid-preconditioned solves to 1e-8 on the densities saved by --save-design "
                         "(the program the multigrid profile traces)")
    ap.add_argument("--kernels-only", action="store_true",
                    help="only the PCG/filter/OC kernels (pf_profile_kernels) on a seeded density field, then a "
                         "plain device copy of known size: the program the counter runs profile")
    ap.add_argument("--learned-only", action="store_true",
                    help="only the learned-preconditioner comparison (training and the three solves): the program "
                         "the learned profile traces")
    ap.add_argument("--form-sweep", action="store_true",
                    help="only the per-iteration time of the three FP64 Jacobi-PCG forms at five grid sizes")
    ap.add_argument("--cpu-reference", action="store_true",
                    help="only the reference's full CPU timings: the 120x40 loop per phase, ScalingCG to 1e-8 and "
                         "1e-10 on the 1024x512 iteration-0 system, one MMA update there")
    ap.add_argument("--h8-operators", action="store_true",
                    help="only the hex8 fused PCG kernel with each operator kernel (vector units, matrix cores) at "
                         "128x64x64")
    ap.add_argument("--conv-kernels", action="store_true",
                    help="only the learned preconditioner's kernels at 1024x512: a few training steps and network "
                         "applications (the program the counter runs of those kernels profile)")
    ap.add_argument("--c2-loops", action="store_true",
                    help="only the whole 1024x512 workload: 100 OC iterations and 100 MMA iterations with FP64 "
                         "Jacobi-PCG")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py runs on one GPU only (asked for --gpus {args.gpus}); a multi-GPU decomposition of "
              "this path is not built.", file=sys.stderr)
        sys.exit(2)

    if args.cpu_reference:
        print(json.dumps({"cpu_reference": cpu_reference_runs()}))
        return

    import torch
    import pansfem2_amd as pa

    if args.c2_loops:
        print(json.dumps({"c2_loops": c2_loops(pa, torch)}))
        return
    if args.h8_operators:
        print(json.dumps({"h8_operators": h8_operators(pa)}))
        return
    if args.conv_kernels:
        print(json.dumps({"conv_kernels": conv_kernels(pa)}))
        return
    if args.form_sweep:
        form_sweep(pa)
        return
    if args.learned_only:
        print(json.dumps({"learned": learned_vs_jacobi(pa, args.nx, args.ny)}))
        return
    nx, ny = args.nx, args.ny
    ctx = pa.cantilever2d(nx, ny)
    N, ne = ctx.N, ctx.ne
    if args.kernels_only:
        kernels_only(ctx, pa, torch, nx, ny)
        return
    if args.save_design:
        ctx.set_pcg_form(pa.PF_PCG_SINGLE_REDUCTION)
        r = ctx.simp_run(args.design_iters)
        np.save(args.save_design, r["rho"])
        print(json.dumps({"saved_design": args.save_design, "oc_iterations": args.design_iters}))
        return
    if args.mg_solve:
        ctx.set_density(np.load(args.mg_solve))
        b = ctx.load()
        out = {}
        for label, mode in (("stiffness", pa.PF_MG_PROLONG_STIFFNESS), ("bilinear", pa.PF_MG_PROLONG_BILINEAR)):
            ctx.mg_set_prolongation(mode)
            ctx.mg_setup(1, 0.6)
            out[label] = []
            for _ in range(2):
                x, st = ctx.pcg(b, op=pa.PF_OP_MG, eps=1e-8)
                out[label].append({"seconds": st["seconds"], "iterations": st["iterations"],
                                   "true_residual": st["true_residual"]})
        print(json.dumps({"multigrid_solves": out}))
        return
    # warmup OC iterations (untimed), then K timed iterations continuing the same trajectory,
    # repeated from the same warmed design; the median window is reported
    ctx.set_pcg_form(pa.PF_PCG_SINGLE_REDUCTION)
    w = ctx.simp_run(args.warmup) if args.warmup > 0 else {"s": np.full(ne, 0.5)}
    walls, runs = [], []
    for _ in range(max(1, args.repeats)):
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        rk = ctx.simp_run(args.steps, s0=w["s"])
        torch.cuda.synchronize()
        walls.append(time.perf_counter() - t0)
        runs.append(rk)
    r = runs[0]
    repeats_identical = all(np.array_equal(q["f"], r["f"]) and np.array_equal(q["rho"], r["rho"]) for q in runs)
    wall = float(np.median(walls))
    value = args.steps / wall
    n_cg = float(np.mean(r["cg_iters"]))
    n_bis = float(np.mean(r["bisect"]))
    # the same steps with ScalingCG's order
    ctx.set_pcg_form(pa.PF_PCG_SCALINGCG)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    r0 = ctx.simp_run(args.steps, s0=w["s"])
    torch.cuda.synchronize()
    wall0 = time.perf_counter() - t0
    ctx.set_pcg_form(pa.PF_PCG_SINGLE_REDUCTION)
    # and with multigrid-preconditioned CG to the same 1e-10 (true residual)
    ctx.mg_setup(1, 0.6)
    ctx.simp_run(1, pa.simp_default_params(solver=pa.PF_OP_MG), s0=w["s"])  # allocations
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    rm = ctx.simp_run(args.steps, pa.simp_default_params(solver=pa.PF_OP_MG), s0=w["s"])
    torch.cuda.synchronize()
    wallm = time.perf_counter() - t0
    # the MMA variant (one volume constraint; asymptotes 0.5, shrink 0.7, grow 1.2) with the same solves
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    rmma = ctx.simp_run(args.steps, pa.simp_default_params(solver=pa.PF_OP_MG, use_mma=1), s0=w["s"])
    torch.cuda.synchronize()
    wallmma = time.perf_counter() - t0
    ctx.mg_setup(0, 0.0)

    # dominant kernel: the resident solve, timed over 4000 iterations on the final
    # design (warm), and HIP-event timing of the launched PCG kernels beside it
    ctx.set_density(r["rho"])
    b_res = ctx.load()
    for _ in range(2):
        _, st_res = ctx.pcg(b_res, op=pa.PF_OP_EBE64, eps=0.0, itrmax=4000)
    ms_res = 1e3 * st_res["seconds"] / st_res["iterations"]
    # operator 136 per element, vector updates and sums 22 per DOF
    flops_res = 136.0 * ne + 22.0 * N
    prof = ctx.profile_kernels(pa.PF_OP_EBE64, reps=100)
    bytes_k1 = 8 * ne + 4 * 8 * N   # p_old, z read; p_new, q written; E read
    bytes_k2 = 8 * 8 * N            # x, r, p, q, D read; x, r, z written
    # r, w, s, D, p read; r, w, s, p written; E read; x read and written by every
    # other launch (the even ones): 8 ne + 80 N on average over a pair
    bytes_cg1 = 8 * ne + 10 * 8 * N
    name = "pcg_cg1_q4 (launched single-reduction iteration, grids beyond the resident solve's)"
    ms, byts = prof["cg1_ms"], bytes_cg1
    achieved = byts / (ms * 1e-3) / 1e9
    iter_ms = prof["k1_ms"] + prof["k2_ms"]
    copy_gbs = stream_copy_gbs(torch)
    # a copy whose source and destination together are the kernel's working
    # set stays in the last-level cache, as the kernel's own traffic does
    copy_resident_gbs = stream_copy_gbs(torch, mib=byts / 2 / 2**20, reps=100)
    # the scope table's unit for an FP64 matrix-free Jacobi-PCG iteration
    # (13 vector passes: 8 ne + 104 N bytes), against the same kernel time
    bytes_unit = 8 * ne + 13 * 8 * N
    traffic = None
    tfile = os.path.join(ROOT, "profiles", "traffic_pcg_q4_1024x512.json")
    if os.path.exists(tfile):
        try:
            traffic = json.load(open(tfile)).get(name.split()[0])
        except Exception:
            traffic = None

    extras = {}
    if not args.no_extras:
        b = ctx.load()
        for label, op, form in (("jacobi_fp64", pa.PF_OP_EBE64, pa.PF_PCG_SINGLE_REDUCTION),
                                ("jacobi_fp64_scalingcg_order", pa.PF_OP_EBE64, pa.PF_PCG_SCALINGCG),
                                ("mixed_fp32_ir", pa.PF_OP_EBE32, pa.PF_PCG_SINGLE_REDUCTION)):
            ctx.set_pcg_form(form)
            x, st = ctx.pcg(b, op=op, eps=1e-8)
            extras[label] = {"seconds": st["seconds"], "iterations": st["iterations"],
                             "true_residual": st["true_residual"], "status": st["status"], "outer": st["outer"]}
        ctx.set_pcg_form(pa.PF_PCG_SINGLE_REDUCTION)
        extras["speedup_mixed_vs_jacobi"] = extras["jacobi_fp64"]["seconds"] / extras["mixed_fp32_ir"]["seconds"]
        if not args.no_learned:
            extras["learned"] = learned_vs_jacobi(pa, nx, ny)
    others = None if (args.no_extras or args.no_others) else other_configs(pa)

    cpu = None if args.no_cpu else cpu_baseline(nx, ny, n_cg, n_bis)
    out = {
        "metric": "SIMP OC iters/sec @1024x512 quad4; PCG time to 1e-8 resid, learned vs Jacobi",
        "value": value, "unit": "OC iters/sec", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": 1000.0 * wall / args.steps, "higher_is_better": True, "scaling": "weak",
        "vs_baseline": None, "dtype": "f64", "data": "synthetic (uniform initial design 0.5, deterministic load case)",
        "timing": {"windows_s": walls, "median_s": wall, "windows_bit_identical": repeats_identical},
        "config": {"workload": f"SIMP OC loop, plane-strain quad4 {nx}x{ny} cantilever, FP64 matrix-free "
                               "Jacobi-PCG to 1e-10, density filter R=1.5, OC move 0.2",
                   "nx": nx, "ny": ny, "elements": ne, "free_dofs": N,
                   "solver": "EBE64 Jacobi-PCG, single-reduction form",
                   "mean_cg_iters": n_cg, "mean_bisection_steps": n_bis,
                   "scalingcg_order": {"value": args.steps / wall0, "ms_per_step": 1000.0 * wall0 / args.steps,
                                       "mean_cg_iters": float(np.mean(r0["cg_iters"])),
                                       "compliance_rel_diff": float(np.max(np.abs(r0["f"] - r["f"]) / r["f"]))},
                   "multigrid_pcg": {"value": args.steps / wallm, "ms_per_step": 1000.0 * wallm / args.steps,
                                     "mean_cg_iters": float(np.mean(rm["cg_iters"])),
                                     "compliance_rel_diff": float(np.max(np.abs(rm["f"] - r["f"]) / r["f"])),
                                     "density_max_abs_diff": float(np.max(np.abs(rm["rho"] - r["rho"])))},
                   "mma_multigrid_pcg": {"value": args.steps / wallmma, "ms_per_step": 1000.0 * wallmma / args.steps,
                                         "mean_cg_iters": float(np.mean(rmma["cg_iters"])),
                                         "compliance_first_last": [float(rmma["f"][0]), float(rmma["f"][-1])]}},
        # one iteration of the resident solve moves no vector through memory: its rate
        # against the FP64 peak, and on the scope table's bytes (above the HBM peak:
        # the vectors are on the chip)
        "roofline": {"bound": "fp64 issue, LDS and the exchange between workgroups",
                     "kernel": "k_pcg_q4_resident (single-reduction form)",
                     "achieved": flops_res / (ms_res * 1e-3) / 1e12, "peak": FP64_PEAK_TFLOPS, "unit": "TFLOP/s",
                     "frac": flops_res / (ms_res * 1e-3) / 1e12 / FP64_PEAK_TFLOPS, "traffic": None,
                     "avg_ms": ms_res, "algorithmic_flops": flops_res,
                     "scope_unit": {"bytes": bytes_unit, "formula": "8 ne + 104 N",
                                    "achieved": bytes_unit / (ms_res * 1e-3) / 1e9,
                                    "frac": bytes_unit / (ms_res * 1e-3) / 1e9 / HBM_PEAK_GBS,
                                    "on_chip": True}},
        "launched": {"bound": "hbm", "kernel": name, "achieved": achieved, "peak": HBM_PEAK_GBS, "unit": "GB/s",
                     "frac": achieved / HBM_PEAK_GBS, "traffic": traffic, "avg_ms": ms, "algorithmic_bytes": byts,
                     "scalingcg_order": {"k1_ms": prof["k1_ms"], "k2_ms": prof["k2_ms"], "iteration_ms": iter_ms,
                                         "bytes": bytes_k1 + bytes_k2,
                                         "achieved": (bytes_k1 + bytes_k2) / (iter_ms * 1e-3) / 1e9},
                     "stream_copy_GBs": copy_gbs, "frac_of_copy": achieved / copy_gbs,
                     "stream_copy_cache_resident_GBs": copy_resident_gbs,
                     "frac_of_cache_resident_copy": achieved / copy_resident_gbs,
                     "scope_unit": {"bytes": bytes_unit, "formula": "8 ne + 104 N",
                                    "achieved": bytes_unit / (ms * 1e-3) / 1e9,
                                    "frac": bytes_unit / (ms * 1e-3) / 1e9 / HBM_PEAK_GBS}},
        "kernels_ms": prof,
        "pcg_time_to_1e-8": extras,
        "other_configs": others,
        "cpu_baseline": cpu,
        "compliance_final": float(r["f"][-1]),
    }
    print(json.dumps(out))


if __name__ == "__main__":
    main()
