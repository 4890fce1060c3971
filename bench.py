"""Benchmark of miniFE's assemble-and-solve path on one MI355X.

Workload: the 300^3 hex8 box problem (27,270,901 rows, 731,432,701 non-zeros,
FP64 values, int32 indices), assembled on the GPU, then plain FP64 CG with 200
iterations (the reference's max_iters, driver.hpp:241).  A "step" is one
200-iteration CG solve from x = 0 on the resident matrix; `value` is CG
iterations per second over the timed steps.

Also reported (not part of `value`): the SpMV kernel's HBM rate and roofline
fraction (HIP events around back-to-back launches of the exact kernel the CG
runs), assembly rate (elements/s) and its roofline, time to ||r||/||b|| <= 1e-10
in FP64 and mixed precision, the batched, many-RHS and adjoint workloads, and a
CPU baseline: the reference's own CG compiled from its sources (openmp/src on
all host threads, ref/src serial) timed on this host over a bounded sample of
the same matrix, beside the oracle's restatement of it.

Usage: python bench.py [--gpus 1] [--steps K] [--warmup W] [--n 300]
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK_GBS = 8000.0  # MI355X HBM3E
# MI355X FP64 vector peak is 78.6 TFLOP/s counting an FMA as two flops; the
# assembly keeps the reference's separate multiply and add (no contraction),
# one flop per instruction, so its arithmetic peak is half that.
FP64_NOFMA_PEAK_TFLOPS = 78.6 / 2
# FP64 flops per element of the fused element computation (diffusion matrix
# 4,488 incl. 8 divides, source vector 400 more with the Jacobian shared).
FLOPS_PER_ELEMENT = 4888


def log(msg):
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def spmv_bytes(n: int, nnz: int, value_bytes: int = 8) -> int:
    """Algorithmic HBM bytes of one CSR SpMV: values + int32 columns, row
    offsets, x read once and y written once."""
    return (value_bytes + 4) * nnz + 4 * (n + 1) + 2 * value_bytes * n


def sell_bytes(n: int, plan: dict, value_bytes: int = 8) -> int:
    """HBM bytes of one SELL-64 SpMV: every stored entry (padding included)
    as value + int32 column, one length byte per row slot, the slice offsets,
    x read once and y written once."""
    slots, ns = plan["stored"], plan["slices"]
    return (value_bytes + 4) * slots + 64 * ns + 4 * (ns + 1) + 2 * value_bytes * n


def sellx_bytes(n: int, plan: dict, value_bytes: int = 8) -> int:
    """HBM bytes of one SELL-64 SpMV with staged x: every stored entry's value,
    a 16-bit local column for the entries of slices without bases, one flag
    byte per slice and 27 16-bit bases per slice with bases, one length byte
    per row slot, the slice offsets, the plan's runs (first column, list
    position) and per-tile run offsets and distinct counts, x read once and y
    written once."""
    slots, ns, runs = plan["stored"], plan["slices"], plan["runs"]
    tiles = -(-n // 256)
    return (value_bytes * slots + 2 * plan["explicit_entries"] + ns + 54 * plan["base_slices"]
            + 64 * ns + 4 * (ns + 1) + 8 * runs + 4 * (tiles + 1) + 4 * tiles
            + 2 * value_bytes * n)


def box_bytes(dims, plan: dict, value_bytes: int = 8) -> int:
    """HBM bytes of one SpMV on the box layout: 27 values per row (each row is
    padded to 27 slots; rows past the box's edge in a block are not loaded),
    the x window of every plane step (the block and its one-node ring, inside
    the box, for the chunk's planes and the one before and after it), y
    written once.  No column indices."""
    gx, gy, gz = dims
    n = gx * gy * gz
    zc, nzc = plan["planes_per_chunk"], plan["z_chunks"]
    cells = 0
    for bx in range(plan["blocks_x"]):
        wx = min(gx, bx * 16 + 17) - max(0, bx * 16 - 1)
        for by in range(plan["blocks_y"]):
            wy = min(gy, by * 16 + 17) - max(0, by * 16 - 1)
            cells += wx * wy
    planes = 0
    for c in range(nzc):
        z0, z1 = c * zc, min(c * zc + zc, gz)
        planes += min(gz, z1 + 1) - max(0, z0 - 1)
    return value_bytes * (27 * n + cells * planes + n)


def boxsym_bytes(dims, plan: dict, value_bytes: int = 8) -> int:
    """HBM bytes of one SpMV on the symmetric box layout: 14 upper values per
    row, 282 values per (block, plane) for the lower slots whose neighbour is
    outside the block, the previous plane's nine upper-plane values per row
    at the start of each z chunk but the first, the x window as for the box
    layout, y written once."""
    gx, gy, gz = dims
    n = gx * gy * gz
    full = box_bytes(dims, plan, value_bytes) - value_bytes * 27 * n
    nb = plan["blocks_x"] * plan["blocks_y"]
    return full + value_bytes * (14 * n + 282 * nb * gz + 9 * gx * gy * (plan["z_chunks"] - 1))


PACKED_BOUNDARY_ROWS = 1 << 23  # rows from which the CG's kernel reads it packed


def boxpack_bytes(dims, plan: dict, value_bytes: int = 8) -> int:
    """HBM bytes of one SpMV on the symmetric box layout with packed upper
    values: as boxsym_bytes, but a row's packed slots cost its 32-bit words
    of fields instead of value_bytes each, plus a record of 30 values per
    (block, plane): 14 bases, 14 powers of two and the codes flag as words, the
    rest padding; where the CG's kernel reads the FP64 boundary stream packed too
    (from 2^23 rows on), its words and 13 (base, power of two) pairs and a
    flag per (block, plane) instead of its 282 values."""
    import minife_amd as mfe
    gx, gy, gz = dims
    n = gx * gy * gz
    nb = plan["blocks_x"] * plan["blocks_y"]
    words, fulls = mfe.pack_row_layout(plan["pack"] if value_bytes == 8 else plan["pack_fp32"])
    wform = plan.get("wpack") if value_bytes == 8 and n >= PACKED_BOUNDARY_ROWS else None
    wbytes = (4 * mfe.pack_bnd_words(wform) + value_bytes * 27 - value_bytes * 282) if wform else 0
    return (boxsym_bytes(dims, plan, value_bytes) - value_bytes * (14 - fulls) * n
            + 4 * words * n + value_bytes * (2 * 14 + 2) * nb * gz + wbytes * nb * gz)


def plan_bytes(n: int, nnz: int, plan: dict, value_bytes: int = 8, dims=None) -> int:
    """Bytes of one SpMV in the format the plan chose (FP32: the FP32 layout's)."""
    if plan["kernel"] == "box-sym-packed":
        if value_bytes == 4 and not plan.get("pack_fp32"):
            return boxsym_bytes(dims, plan, 4)
        return boxpack_bytes(dims, plan, value_bytes)
    if plan["kernel"] == "box-sym":
        return boxsym_bytes(dims, plan, value_bytes)
    if plan["kernel"] == "box":
        return box_bytes(dims, plan, value_bytes)
    if plan["kernel"] == "sell64-staged-x":
        return sellx_bytes(n, plan, value_bytes)
    if plan["kernel"] == "sell64":
        return sell_bytes(n, plan, value_bytes)
    return spmv_bytes(n, nnz, value_bytes)


KERNEL_NAMES = {"box-sym-packed": "spmv_boxsym_kernel", "box-sym": "spmv_boxsym_kernel",
                "box": "spmv_box_kernel",
                "sell64-staged-x": "spmv_sellx_kernel",
                "sell64": "spmv_sell_kernel",
                "csr-stream": "spmv_stream_kernel", "csr-rowwise": "spmv_rowwise_kernel"}


# the CG's SpMV kernel of each format as rocprofv3 names it
CG_KERNEL_PROFILE_NAMES = {"box-sym-packed": "spmv_boxsym_kernel<double, false, 1, {form}, {wpk}>",
                           "box-sym": "spmv_boxsym_kernel<double, false, 1, 0>",
                           "box": "spmv_box_kernel<double, false, 1>",
                           "sell64-staged-x": "spmv_sellx_kernel<double, false, 1>"}


def measured_traffic(N: int, kernel: str):
    """HBM bytes per launch of the CG SpMV kernel from the committed rocprofv3
    FETCH_SIZE/WRITE_SIZE summary for this workload (calibrated against a
    kernel of known size; see the summary for the commands), else None --
    also when the summary was taken of another kernel."""
    path = os.path.join(ROOT, "profiles", f"spmv_cg_{N}_traffic.json")
    if not os.path.exists(path):
        return None
    with open(path) as f:
        d = json.load(f)
    if d.get("kernel", "") != kernel:
        return None
    return d.get("traffic_bytes_per_launch")


def cpu_model() -> str:
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def cpu_baseline(A_dev, b_dev, n, nnz, iters: int, omp_iters: int):
    """The reference CPU path on this host, on the same 300^3 matrix: the
    compiled reference's cg_solve (openmp/src on all the host threads = the
    reported baseline, kind "reference"; ref/src serial beside it), each next
    to the oracle's restatement of the same form (the "port") for
    calibration.  Rates come from each CG's own TOTAL timer (the copy of the
    matrix into the reference's containers is not timed); `omp_iters` and
    `iters` bound the sample."""
    import oracle
    if not os.path.exists(oracle.LIB_PATH):
        return None
    h = A_dev.to_host(rows=False)
    A = oracle.CSR(np.arange(n, dtype=np.int32), h["row_offsets"], h["cols"], h["vals"])
    b = b_dev.to_numpy()
    del h
    threads = int(os.environ.get("OMP_NUM_THREADS", os.cpu_count() or 1))

    def rate(r):
        its = r["num_iters"]
        return its / r["times"][4], r["times"][2] / (its + 1)

    po = oracle.cg_solve_omp(A, b, np.zeros(n), max_iter=omp_iters, threads=threads)
    ps = oracle.cg_solve(A, b, np.zeros(n), max_iter=iters, want_times=True)
    po_rate, po_mv = rate(po)
    ps_rate, ps_mv = rate(ps)
    port = {"value": po_rate, "cores": po["threads"], "spmv_GBs": spmv_bytes(n, nnz) / po_mv / 1e9,
            "serial": {"value": ps_rate, "cores": 1,
                       "spmv_GBs": spmv_bytes(n, nnz) / ps_mv / 1e9}}
    cpu = cpu_model()
    if not (oracle.ref_cg_available(omp=True) and oracle.ref_cg_available(omp=False)):
        return {"value": po_rate, "unit": "CG iterations/s", "cores": po["threads"],
                "kind": "port", "cpu": cpu,
                "sample": f"{po['num_iters']} of 200 FP64 CG iterations on the same 300^3 matrix "
                          f"(oracle restatement of openmp/src cg_solve, {po['threads']} threads)",
                "spmv_GBs": port["spmv_GBs"], "serial": port["serial"]}
    ro = oracle.ref_cg(A, b, max_iter=omp_iters, omp=True, threads=threads)
    rs = oracle.ref_cg(A, b, max_iter=iters, omp=False)
    ro_rate, ro_mv = rate(ro)
    rs_rate, rs_mv = rate(rs)
    return {
        "value": ro_rate, "unit": "CG iterations/s", "cores": ro["threads"], "kind": "reference",
        "cpu": cpu,
        "sample": f"{ro['num_iters']} of 200 FP64 CG iterations on the same 300^3 matrix "
                  f"(openmp/src cg_solve compiled from the reference sources, {ro['threads']} "
                  f"threads, {ro['times'][4]:.1f} s)",
        "spmv_GBs": spmv_bytes(n, nnz) / ro_mv / 1e9,
        "serial": {"value": rs_rate, "cores": 1, "spmv_GBs": spmv_bytes(n, nnz) / rs_mv / 1e9,
                   "sample": f"{rs['num_iters']} iterations of ref/src cg_solve "
                             f"({rs['times'][4]:.1f} s)"},
        "port": port,
        "port_over_reference": {"omp": po_rate / ro_rate, "serial": ps_rate / rs_rate},
    }


def bench_batched(mfe, ctx):
    """64 boxes, sides uniform on [16, 96] (seed 0): assembly + FP64 CG to
    1e-10 together.  Equivalent bytes per problem and
    iteration: 12 B per stored SELL entry + 88 B per row (p update, x gather,
    Ap, x/r update), plus nothing for assembly (not counted); the packed values
    move fewer."""
    from minife_amd.workloads import batch_boxes
    B = mfe.Batch(batch_boxes(0), ctx)
    B.solve(max_iter=5000, rel_tol=1e-10)  # warm (code objects, first touch)
    out = B.solve(max_iter=5000, rel_tol=1e-10)
    byts = 0
    for p in range(B.nprob):
        inf = B.info(p)
        byts += int(out["iters"][p]) * (12 * inf["stored"] + 88 * inf["rows"])
    tot = B.info()
    slow = int(np.argmax(out["problem_seconds"]))
    slowest = {"problem": slow, "dims": [int(v) for v in B.dims[slow]],
               "iters": int(out["iters"][slow]), "workgroups": B.info(slow)["workgroups"],
               "seconds": float(out["problem_seconds"][slow]),
               "phase_seconds": {k: round(float(v), 5)
                                 for k, v in zip(B.PHASES, out["phase_seconds"][slow])}}
    res = {"workload": "64 boxes, sides U[16,96] seed 0, assemble + FP64 CG to 1e-10 together",
           "seconds": out["seconds"], "problems": B.nprob, "workgroups": tot["workgroups"],
           "rows": tot["rows"], "nnz": tot["nnz"], "iters_total": int(out["iters"].sum()),
           "iters_max": int(out["iters"].max()),
           "max_rel_residual": float(out["rel_residual"].max()),
           "cg_equiv_GBs": byts / out["seconds"] / 1e9, "slowest_problem": slowest}
    B.close()
    return res


def bench_multi_rhs(mfe, ctx):
    """128^3 with 16 right-hand sides (N(0,1) per free node, seed 1): simultaneous
    CG over the autotuned CSR x 16 SpMM, against 16 single-vector solves."""
    from minife_amd.workloads import multi_rhs_sources
    N, K = 128, 16
    mesh = mfe.simple_mesh_description([0, N, 0, N, 0, N])
    A = mfe.CSRMatrix(ctx)
    assert mfe.generate_matrix_structure(mesh, A) == 0
    b = mfe.Vector(A.nrows, ctx)
    mfe.assemble_FE_data(mesh, A, b)
    mfe.impose_dirichlet(0.0, A, b, N + 1, N + 1, N + 1, mesh.bc_rows_0)
    mfe.impose_dirichlet(1.0, A, b, N + 1, N + 1, N + 1, mesh.bc_rows_1)
    mfe.make_local_matrix(A)
    n, nnz = A.shape
    Bh = multi_rhs_sources(n, K, 1)
    Bh[np.union1d(mesh.bc_rows_0, mesh.bc_rows_1), :] = 0.0
    Bd = mfe.Vector.from_numpy(Bh.ravel(), ctx)
    tun = mfe.spmm_tune(A, K)
    X = mfe.Vector(n * K, ctx)
    mfe.cg_solve_multi(A, Bd, X, K, max_iter=5000, rel_tol=1e-10)  # warm (graph capture)
    X.fill(0.0)
    r = mfe.cg_solve_multi(A, Bd, X, K, max_iter=5000, rel_tol=1e-10)
    # the same 16 systems one at a time with the single-vector CG
    t_single = 0.0
    its_single = 0
    xs = mfe.Vector(n, ctx)
    for k in range(K):
        bk = mfe.Vector.from_numpy(np.ascontiguousarray(Bh[:, k]), ctx)
        xs.fill(0.0)
        ctx.synchronize()
        t0 = time.perf_counter()
        rk = mfe.cg_solve(A, bk, xs, max_iter=5000, tolerance=1e-10, relative=True)
        t_single += time.perf_counter() - t0
        its_single += rk.num_iters
    ms = tun["ms"][tun["tile"]]
    # CSR-equivalent bytes of one SpMM (values, columns, row offsets, X and Y once)
    spmm_bytes = 12 * nnz + 4 * (n + 1) + 2 * 8 * K * n
    direct = [v for v, t in zip(tun["ms"], tun["tiles"]) if not t["staged"]]
    staged = [v for v, t in zip(tun["ms"], tun["tiles"]) if t["staged"] and np.isfinite(v)]
    def best(kind):
        v = [m for m, t in zip(tun["ms"], tun["tiles"]) if t["kind"] == kind and np.isfinite(m)]
        return min(v) if v else None
    return {"workload": "128^3, 16 RHS N(0,1) per free node seed 1, FP64 CG to 1e-10 per column",
            "seconds": r.seconds, "iters_min": int(r.iters.min()), "iters_max": int(r.iters.max()),
            "max_rel_residual": float(r.rel_residual.max()),
            "single_rhs_seconds": t_single, "single_rhs_iters": its_single,
            "speedup_vs_single": t_single / r.seconds,
            "spmm_tile": tun["tiles"][tun["tile"]], "spmm_ms": ms,
            "spmm_GBs": spmm_bytes / (ms * 1e-3) / 1e9,
            "best_direct_ms": min(direct), "best_staged_ms": min(staged) if staged else None,
            "best_box_ms": best("box"),
            "tuner_ms": [round(v, 4) if np.isfinite(v) else None for v in tun["ms"]]}


def bench_adjoint(mfe):
    """128^3 differentiable solve: loss and dL/dkappa (forward CG, adjoint CG,
    element-gradient kernel), kappa = exp(N(0, 0.5^2)) seed 2, target from seed 3."""
    from minife_amd import adjoint
    from minife_amd.workloads import kappa_field
    N = 128
    ne = N ** 3
    ut = adjoint.solve_u(N, N, N, kappa_field(ne, 3))
    kappa = kappa_field(ne, 2)
    adjoint.loss_and_gradient(N, N, N, kappa, ut)  # warm
    t0 = time.perf_counter()
    L, g, _ = adjoint.loss_and_gradient(N, N, N, kappa, ut)
    dt = time.perf_counter() - t0
    return {"workload": "128^3 kappa=exp(N(0,0.25)) seed 2, L=0.5||u-u_t||^2, FP64, rel tol 1e-13",
            "seconds": dt, "loss": L, "grad_norm": float(np.linalg.norm(g))}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=5)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--n", type=int, default=300, help="elements per side")
    ap.add_argument("--iters", type=int, default=200, help="CG iterations per step")
    ap.add_argument("--spmv-reps", type=int, default=50)
    ap.add_argument("--cpu-iters", type=int, default=10, help="serial CPU baseline iterations")
    ap.add_argument("--cpu-omp-iters", type=int, default=50,
                    help="OpenMP CPU baseline iterations (all host cores)")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-tol-run", action="store_true")
    ap.add_argument("--no-extras", action="store_true",
                    help="skip the batched, multi-RHS and adjoint workloads")
    ap.add_argument("--only", choices=["batched", "multi_rhs", "adjoint"],
                    help="run just this extra workload and print its JSON (for profiling)")
    args = ap.parse_args()
    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) != 1:
        print("bench.py measures one GPU: the library has no multi-GPU path (the sharding "
              "design is described, not built); run with --gpus 1.", file=sys.stderr)
        sys.exit(2)

    import minife_amd as mfe

    ctx = mfe.Context(0)
    info = ctx.device_info()
    log(f"device {info}")
    if args.only:
        fn = {"batched": lambda: bench_batched(mfe, ctx),
              "multi_rhs": lambda: bench_multi_rhs(mfe, ctx),
              "adjoint": lambda: bench_adjoint(mfe)}[args.only]
        print(json.dumps({args.only: fn(), "device": info["name"]}), flush=True)
        return
    N = args.n
    ne = N ** 3

    # ---- assembly (structure -> elements -> Dirichlet), timed by phase ------
    mesh = mfe.simple_mesh_description([0, N, 0, N, 0, N])
    A = mfe.CSRMatrix(ctx)
    t0 = time.perf_counter()
    assert mfe.generate_matrix_structure(mesh, A) == 0
    ctx.synchronize()
    t_struct = time.perf_counter() - t0
    n, nnz = A.shape
    b = mfe.Vector(n, ctx)
    t0 = time.perf_counter()
    mfe.assemble_FE_data(mesh, A, b)
    ctx.synchronize()
    t_asm = time.perf_counter() - t0
    t0 = time.perf_counter()
    mfe.impose_dirichlet(0.0, A, b, N + 1, N + 1, N + 1, mesh.bc_rows_0)
    mfe.impose_dirichlet(1.0, A, b, N + 1, N + 1, N + 1, mesh.bc_rows_1)
    ctx.synchronize()
    t_bc = time.perf_counter() - t0
    mfe.make_local_matrix(A)
    log(f"assembled n={n} nnz={nnz}: struct {t_struct:.3f}s, FE {t_asm:.3f}s, BC {t_bc:.3f}s")
    t0 = time.perf_counter()
    plan = mfe.spmv_plan(A)
    t_plan = time.perf_counter() - t0
    log(f"spmv plan {plan} built in {t_plan:.3f}s")

    # ---- CG steps ----------------------------------------------------------
    x = mfe.Vector(n, ctx)
    for w in range(args.warmup):
        x.fill(0.0)
        r = mfe.cg_solve(A, b, x, max_iter=args.iters)
        log(f"warmup {w}: iters {r.num_iters} normr {r.normr:.6e}")
    ctx.synchronize()
    iters_total = 0
    t0 = time.perf_counter()
    for s in range(args.steps):
        x.fill(0.0)
        r = mfe.cg_solve(A, b, x, max_iter=args.iters)
        iters_total += r.num_iters
    ctx.synchronize()
    dt = time.perf_counter() - t0
    it_s = iters_total / dt
    log(f"timed {args.steps} steps: {iters_total} iterations in {dt:.3f}s -> {it_s:.1f} it/s, "
        f"final normr {r.normr:.6e}")

    # ---- SpMV kernel rate (the CG's kernel and matvec_std's) ------------------
    xs = mfe.Vector.from_numpy(np.linspace(0.0, 1.0, n), ctx)
    ys = mfe.Vector(n, ctx)
    mfe.time_matvec(A, xs, ys, variant=1, reps=3)
    ms_cg = mfe.time_matvec(A, xs, ys, variant=1, reps=args.spmv_reps)
    ms_std = mfe.time_matvec(A, xs, ys, variant=0, reps=args.spmv_reps)
    ms_32 = mfe.time_matvec(A, xs, ys, variant=2, reps=args.spmv_reps)
    if plan["kernel"] == "box-sym-packed":  # the FP32 copy's packed form, now that it exists
        plan["pack_fp32"] = mfe.spmv_plan(A)["pack_fp32"]
    ms_csr = mfe.time_matvec(A, xs, ys, variant=3, reps=args.spmv_reps)
    ms_csr32 = mfe.time_matvec(A, xs, ys, variant=4, reps=args.spmv_reps)
    staged = plan["kernel"] == "sell64-staged-x"
    box = plan["kernel"] in ("box", "box-sym", "box-sym-packed")
    ms_sell = mfe.time_matvec(A, xs, ys, variant=6, reps=args.spmv_reps) if staged else None
    dims = (N + 1, N + 1, N + 1)
    byt = plan_bytes(n, nnz, plan, dims=dims)
    byt32 = plan_bytes(n, nnz, plan, 4, dims=dims)
    staged_cmp = None
    if box:
        # the staged-x SELL-64 kernel on the same matrix (the format uploaded
        # matrices without the box structure use)
        ms_sx = mfe.time_matvec(A, xs, ys, variant=7, reps=args.spmv_reps)
        ms_sx32 = mfe.time_matvec(A, xs, ys, variant=8, reps=args.spmv_reps)
        staged_cmp = {"fp64_ms": ms_sx, "fp64_GBs": spmv_bytes(n, nnz) / (ms_sx * 1e-3) / 1e9,
                      "fp32_ms": ms_sx32, "box_speedup_fp64": ms_sx / ms_cg,
                      "box_speedup_fp32": ms_sx32 / ms_32}
        log(f"staged-x SELL-64 on the same matrix: fp64 {ms_sx:.4f} ms, fp32 {ms_sx32:.4f} ms; "
            f"box layout {ms_sx / ms_cg:.3f}x / {ms_sx32 / ms_32:.3f}x faster")
        if plan["kernel"] == "box-sym-packed":
            # the symmetric layout with every upper value at full width
            ms_64 = mfe.time_matvec(A, xs, ys, variant=11, reps=args.spmv_reps)
            b64 = boxsym_bytes(dims, plan)
            ms_64_32 = mfe.time_matvec(A, xs, ys, variant=12, reps=args.spmv_reps)
            staged_cmp["box_sym_full_values"] = {
                "fp64_ms": ms_64, "kernel_bytes_per_launch": b64,
                "kernel_bytes_GBs": b64 / (ms_64 * 1e-3) / 1e9, "packed_speedup": ms_64 / ms_cg,
                "fp32_ms": ms_64_32, "packed_speedup_fp32": ms_64_32 / ms_32}
            log(f"symmetric layout with full-width upper values: fp64 {ms_64:.4f} ms "
                f"({b64 / (ms_64 * 1e-3) / 1e9:.0f} GB/s of its bytes), fp32 {ms_64_32:.4f} ms; "
                f"packed form {ms_64 / ms_cg:.3f}x / {ms_64_32 / ms_32:.3f}x faster")
        if plan["kernel"] in ("box-sym", "box-sym-packed"):
            ms_full = mfe.time_matvec(A, xs, ys, variant=9, reps=args.spmv_reps)
            ms_full32 = mfe.time_matvec(A, xs, ys, variant=10, reps=args.spmv_reps)
            fb = box_bytes(dims, plan)
            staged_cmp["box_27_slots"] = {
                "fp64_ms": ms_full, "fp32_ms": ms_full32, "kernel_bytes_per_launch": fb,
                "kernel_bytes_GBs": fb / (ms_full * 1e-3) / 1e9,
                "sym_speedup_fp64": ms_full / ms_cg, "sym_speedup_fp32": ms_full32 / ms_32}
            log(f"box layout with 27 slots: fp64 {ms_full:.4f} ms, fp32 {ms_full32:.4f} ms "
                f"({fb / (ms_full * 1e-3) / 1e9:.0f} GB/s of its bytes)")
    kname = KERNEL_NAMES[plan["kernel"]]
    # rates: algorithmic SpMV bytes (CSR operator, x and y once) / time; the
    # kernel_* figures divide the bytes of the plan's format instead
    gbs_cg = byt / (ms_cg * 1e-3) / 1e9
    alg_gbs_cg = spmv_bytes(n, nnz) / (ms_cg * 1e-3) / 1e9
    gbs_std = spmv_bytes(n, nnz) / (ms_std * 1e-3) / 1e9
    gbs_32 = spmv_bytes(n, nnz, 4) / (ms_32 * 1e-3) / 1e9
    gbs_csr = spmv_bytes(n, nnz) / (ms_csr * 1e-3) / 1e9
    gbs_csr32 = spmv_bytes(n, nnz, 4) / (ms_csr32 * 1e-3) / 1e9
    sell_cmp = None
    if staged:
        sb = sell_bytes(n, plan)
        sell_cmp = {"fp64_ms": ms_sell, "fp64_GBs": spmv_bytes(n, nnz) / (ms_sell * 1e-3) / 1e9,
                    "kernel_bytes_per_launch": sb,
                    "kernel_bytes_GBs": sb / (ms_sell * 1e-3) / 1e9,
                    "staged_x_speedup": ms_sell / ms_cg}
        log(f"plain SELL-64 (no staged x) {ms_sell:.4f} ms -> {sell_cmp['fp64_GBs']:.1f} GB/s; "
            f"staged x is {ms_sell / ms_cg:.3f}x faster")
    log(f"spmv ({plan['kernel']}, cg kernel) {ms_cg:.4f} ms -> {alg_gbs_cg:.1f} GB/s algorithmic "
        f"({gbs_cg:.1f} GB/s of its own bytes); matvec_std "
        f"{ms_std:.4f} ms -> {gbs_std:.1f} GB/s; fp32 {ms_32:.4f} ms -> {gbs_32:.1f} GB/s; "
        f"csr kernels: fp64 {ms_csr:.4f} ms ({gbs_csr:.1f} GB/s), fp32 {ms_csr32:.4f} ms "
        f"({gbs_csr32:.1f} GB/s)")

    # ---- time to ||r||/||b|| <= 1e-10 ----------------------------------------
    tol_run = None
    if not args.no_tol_run:
        bnorm = float(np.sqrt(mfe.dot(b, b)))
        res = mfe.Vector(n, ctx)

        def true_rel(xv):
            # ||b - A x|| / ||b|| in FP64 on the GPU
            mfe.matvec(A, xv, res)
            mfe.waxpby(1.0, b, -1.0, res, res)
            return float(np.sqrt(mfe.dot(res, res))) / bnorm

        # FP64 plain CG to ||r||/||b|| <= 1e-10 (warm run first, then timed).  CG
        # stops on its recursive residual; when the true one is still above the
        # target the solve is restarted from the current x (cg_solve's first step
        # recomputes r = b - A x), as a user needing the true residual would.
        for timed in (False, True):
            x.fill(0.0)
            ctx.synchronize()
            t0 = time.perf_counter()
            its64, restarts = 0, 0
            while True:
                r2 = mfe.cg_solve(A, b, x, max_iter=5000, tolerance=1e-10, relative=True)
                its64 += r2.num_iters
                if r2.num_iters == 0 or true_rel(x) <= 1e-10 or restarts >= 5:
                    break
                restarts += 1
            tt = time.perf_counter() - t0
        x64 = x.to_numpy()
        # mixed: FP32 inner CG to 1e-5 + FP64 refinement to 1e-10
        xm = mfe.Vector(n, ctx)
        for timed in (False, True):
            xm.fill(0.0)
            ctx.synchronize()
            t0 = time.perf_counter()
            rm = mfe.cg_solve_mixed(A, b, xm, inner_tol=1e-5, outer_tol=1e-10)
            tm = time.perf_counter() - t0
        xmh = xm.to_numpy()
        # mixed, keeping the FP32 CG's direction across refinements
        xk = mfe.Vector(n, ctx)
        for timed in (False, True):
            xk.fill(0.0)
            ctx.synchronize()
            t0 = time.perf_counter()
            rk = mfe.cg_solve_mixed(A, b, xk, inner_tol=0.1, outer_tol=1e-10,
                                    keep_direction=True)
            tk = time.perf_counter() - t0
        xkh = xk.to_numpy()
        # all residuals recomputed in FP64 on the GPU
        bh = b.to_numpy()
        mfe.matvec(A, x, res)
        rel64 = float(np.linalg.norm(bh - res.to_numpy())) / bnorm
        mfe.matvec(A, xm, res)
        relm = float(np.linalg.norm(bh - res.to_numpy())) / bnorm
        mfe.matvec(A, xk, res)
        relk = float(np.linalg.norm(bh - res.to_numpy())) / bnorm
        err = float(np.linalg.norm(xmh - x64) / np.linalg.norm(x64))
        errk = float(np.linalg.norm(xkh - x64) / np.linalg.norm(x64))
        tol_run = {"fp64_s": tt, "fp64_iters": its64, "fp64_restarts": restarts,
                   "fp64_true_rel_residual": rel64,
                   "mixed_s": tm, "mixed_outer": rm.outer_iters, "mixed_inner": rm.inner_iters,
                   "mixed_true_rel_residual": relm, "mixed_converged": rm.converged,
                   "mixed_rel_err_vs_fp64": err, "speedup_mixed_vs_fp64": tt / tm,
                   "mixed_keep_direction": {
                       "inner_tol": 0.1, "s": tk, "outer": rk.outer_iters, "inner": rk.inner_iters,
                       "true_rel_residual": relk, "converged": rk.converged,
                       "rel_err_vs_fp64": errk, "speedup_vs_fp64": tt / tk}}
        log(f"time to 1e-10: fp64 {tt:.3f}s ({its64} its, {restarts} restarts, true rel "
            f"{rel64:.2e}); mixed "
            f"{tm:.3f}s ({rm.outer_iters} outer, {rm.inner_iters} inner, true rel {relm:.2e}), "
            f"|x_mixed-x_fp64|/|x_fp64| = {err:.2e}; keep-direction {tk:.3f}s ({rk.outer_iters} "
            f"outer, {rk.inner_iters} inner, true rel {relk:.2e}, err {errk:.2e})")
        del xk
        del res

    extras = {}
    if not args.no_extras:
        del x
        extras["batched"] = bench_batched(mfe, ctx)
        log(f"batched: {extras['batched']}")
        extras["multi_rhs"] = bench_multi_rhs(mfe, ctx)
        log(f"multi-rhs: {extras['multi_rhs']}")
        extras["adjoint"] = bench_adjoint(mfe)
        log(f"adjoint: {extras['adjoint']}")

    cpu = None
    if not args.no_cpu_baseline:
        log("cpu baseline ...")
        cpu = cpu_baseline(A, b, n, nnz, args.cpu_iters, args.cpu_omp_iters)
        if cpu:
            log(f"cpu baseline {cpu['value']:.3f} it/s ({cpu['sample']})")

    form = {v: k for k, v in mfe.PACK_FORMS.items()}.get(plan.get("pack"), 0)
    wpk = "true" if plan.get("wpack") and n >= PACKED_BOUNDARY_ROWS else "false"
    traffic = measured_traffic(N, CG_KERNEL_PROFILE_NAMES.get(plan["kernel"], "").format(
        form=form, wpk=wpk))
    # Assembly (the element loop, perform_element_loop): bounded by the FP64
    # arithmetic of the element computation and by HBM for the values read
    # and written once (accumulating onto A's existing entries) and b
    asm_flops = FLOPS_PER_ELEMENT * ne
    asm_bytes = 16 * nnz + 16 * n
    t_flop = asm_flops / (FP64_NOFMA_PEAK_TFLOPS * 1e12)
    t_hbm = asm_bytes / (HBM_PEAK_GBS * 1e9)
    asm_roof = {"bound": "fp64-valu" if t_flop >= t_hbm else "hbm",
                "flops": asm_flops, "flops_per_element": FLOPS_PER_ELEMENT,
                "peak_TFLOPs": FP64_NOFMA_PEAK_TFLOPS, "bytes": asm_bytes,
                "hbm_bound_s": t_hbm, "flop_bound_s": t_flop,
                "achieved_TFLOPs": asm_flops / t_asm / 1e12,
                "hbm_frac": t_hbm / t_asm, "frac": max(t_flop, t_hbm) / t_asm}
    out = {
        "metric": "CG iters/s + SpMV HBM GB/s at 300^3 FP64; time-to-1e-10 resid, mixed vs FP64",
        "value": it_s,
        "unit": "CG iterations/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": 1e3 * dt / args.steps,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic (miniFE hex8 box, unit conductivity, Q=1, u=1 on x=1)",
        "config": {"workload": f"miniFE {N}x{N}x{N} hex8 box, FP64 CSR assembled on GPU, "
                               f"unpreconditioned CG {args.iters} iterations",
                   "nx": N, "ny": N, "nz": N, "nrows": n, "nnz": nnz,
                   "cg_iters_per_step": args.iters},
        # achieved: the algorithmic bytes of one FP64 SpMV (12 nnz + 4(n+1) + 16n,
        # the CSR operator read once, x read once, y written once; independent of
        # the storage format) over the CG SpMV kernel's mean launch time;
        # kernel_bytes: what this kernel's format moves by the same accounting
        # physical_frac: the counter-measured HBM bytes of one launch (traffic)
        # over the same time; kernel_bytes_frac: the format's own bytes
        "roofline": {"bound": "hbm", "achieved": alg_gbs_cg, "peak": HBM_PEAK_GBS, "unit": "GB/s",
                     "frac": alg_gbs_cg / HBM_PEAK_GBS,
                     "traffic": traffic,
                     "physical_frac": (traffic / (ms_cg * 1e-3) / 1e9 / HBM_PEAK_GBS
                                       if traffic else None),
                     "kernel": kname + (f"<double,false,kDot,packed {plan['pack']}>" if plan["kernel"] == "box-sym-packed"
                                        else "<double,false,kDot>") + " (CG SpMV + p.Ap partials)",
                     "bytes_per_launch": spmv_bytes(n, nnz), "avg_ms": ms_cg,
                     "kernel_bytes_per_launch": byt, "kernel_bytes_GBs": gbs_cg,
                     "kernel_bytes_frac": gbs_cg / HBM_PEAK_GBS},
        # the CG iteration against the fused minimum per iteration: one CSR SpMV
        # (12 nnz + 4(n+1) + 16n) plus x, p, r, Ap read and x, r, p written (56n)
        "cg_iteration": {"fused_min_bytes": spmv_bytes(n, nnz) + 56 * n,
                         "GBs": it_s * (spmv_bytes(n, nnz) + 56 * n) / 1e9,
                         "frac_of_peak": it_s * (spmv_bytes(n, nnz) + 56 * n) / 1e9 / HBM_PEAK_GBS,
                         "ms": 1e3 / it_s},
        "spmv_GBs": alg_gbs_cg,
        "spmv_std_GBs": gbs_std,
        "spmv_kernel_bytes": {"fp64": byt, "fp64_GBs": gbs_cg, "fp32": byt32,
                              "fp32_GBs": byt32 / (ms_32 * 1e-3) / 1e9},
        # FP32 SpMV: the FP32 CSR operator's algorithmic bytes (8 nnz + 4(n+1) + 8n)
        # over the mixed solve's inner kernel time, an effective rate; the bytes
        # the kernel moves are in spmv_kernel_bytes.fp32
        "spmv_fp32": {"ms": ms_32, "effective_GBs": gbs_32},
        "spmv_plan": dict(plan, build_s=t_plan),
        "spmv_csr_kernels": {"fp64_ms": ms_csr, "fp64_GBs": gbs_csr, "fp32_ms": ms_csr32,
                             "fp32_GBs": gbs_csr32},
        "spmv_sell_kernel": sell_cmp,
        "spmv_staged_x_kernel": staged_cmp,
        "assembly": {"struct_s": t_struct, "fe_s": t_asm, "dirichlet_s": t_bc,
                     "elements_per_s": ne / t_asm, "roofline": asm_roof},
        "time_to_1e-10": tol_run,
        "cpu_baseline": cpu,
        **extras,
        "device": info["name"],
    }
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
