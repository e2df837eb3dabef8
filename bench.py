"""Benchmark of the Krylov engine on one MI355X.

Default workload (the metric: CG solves/sec to 1e-6 relative residual, learned +
mixed precision vs plain): dense RBF kernel systems K + noise I on 16384 points in
[0,1]^4 (lengthscale ~ LogU[0.05,1], noise ~ LogU[1e-4,1e-1]), 8 N(0,1) right-hand
sides each.  A step is one pass of FP64-residual iterative refinement around FP32 PCG
with the learned rank-64 preconditioner (trained here, on the GPU) over every system;
value = right-hand sides whose FP64-checked relative residual is <= 1e-6, per second.
"plain" is the same refinement around unpreconditioned FP32 CG on the same systems.

    python bench.py [--steps K] [--warmup W]
                    [--workload learned_cg|kron_cg|dense_cg|batched_cg|lanczos|hutch|slq|csr|copy]

Prints one JSON line with the metric, a roofline object for the dominant kernel
(measured with HIP events on the engine's stream) and a CPU baseline (the CPU torch
restatement of the reference algorithm, timed on a bounded sample).
"""
import argparse
import json
import os
import sys
import time

import numpy as np
import torch

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

import cola_amd as ca  # noqa: E402
import cola_amd._native as N  # noqa: E402
from cola_amd.linalg import run_batched_cg  # noqa: E402

METRIC = "CG solves/sec to 1e-6 rel. residual: learned+mixed-prec vs plain; HBM GB/s"
HBM_PEAK = 8000.0  # GB/s
# HBM bytes per kron64_pass_a<float> launch at 64^3 x 16 rhs, from rocprofv3 --pmc FETCH_SIZE (x2.0) plus
# WRITE_SIZE (x1.0), the factors a 1 GiB stream copy reads on the same counters (profiles/kron64_cg_64cubed_hbm_traffic.md)
PASS_A_TRAFFIC_BYTES = (16651.2 + 16222.7) * 1024
FP32_MFMA_PEAK = 157.3  # TFLOP/s
# HBM bytes per dense_f32_lds_kernel<8,4> launch (16384^2 fp32 matrix, 8 rhs): rocprofv3 --pmc FETCH_SIZE (x2.0)
# plus WRITE_SIZE (x1.0), the factors a 1 GiB stream copy reads on the same counters
# (profiles/dense_matvec_16384x8_hbm_traffic.md)
DENSE8_TRAFFIC_BYTES = (526424.10 * 2.0 + 512.13) * 1024
# HBM bytes per symmetric 8-rhs product (dense_sym_kernel<8> + dense_sym_reduce<8>) on the same matrix,
# same counters and factors (profiles/dense_sym_matvec_16384x8_hbm_traffic.md)
DENSE8_SYM_TRAFFIC_BYTES = ((266626.35 + 18589.0) * 2.0 + (36925.76 + 512.0)) * 1024


def dense_product_roof(op, n, B, t):
    """Roofline object of one dense n x n, B-rhs product of `op` timed at t seconds per apply: the
    symmetric product (CK_OP_SYMMETRIC) reads the 128-column strips on and above the diagonal
    (n (n + 128) / 2 entries), the full product all n^2; both read X and write Y once."""
    sym = bool(op.flags & N.CK_OP_SYMMETRIC)
    mat = 4 * n * (n + 128) // 2 if sym else 4 * n * n
    nbytes = mat + 2 * 4 * n * B
    kernel = (f"dense_sym_kernel<8> + dense_sym_reduce<8> (upper 128-column strips, {B} rhs)" if sym
              else f"dense_f32_lds_kernel<8,4> ({B} rhs)")
    traffic = DENSE8_SYM_TRAFFIC_BYTES if sym else DENSE8_TRAFFIC_BYTES
    return {"bound": "hbm", "kernel": kernel, "achieved": nbytes / t / 1e9, "peak": HBM_PEAK, "unit": "GB/s",
            "frac": nbytes / t / 1e9 / HBM_PEAK, "traffic": traffic, "launch_us": t * 1e6,
            "algorithmic_bytes_per_launch": nbytes}


def rbf_factor(t, ell):
    return torch.exp(-(t[:, None] - t[None, :])**2 / (2 * ell**2))


def kron_workload(dev, n1=64, nrhs=16, seed=0):
    g = torch.Generator().manual_seed(seed)
    facs = [rbf_factor(torch.sort(torch.rand(n1, generator=g)).values, 0.1) for _ in range(3)]
    b = torch.randn(n1**3, nrhs, generator=g)
    K = ca.Kronecker(*[ca.Dense(f.to(dev)) for f in facs])
    A = ca.PSD(K + 0.01 * ca.I_like(K))
    return A, facs, b


def kron_apply_f64(facs, X, shift=float(np.float32(0.01))):
    """FP64 (K1 x K2 x K3 + shift I) X on the device, for the residual check only.  The default
    shift is 0.01 as the operator stores it (fp32): the check uses the matrix the solver was given."""
    dims = [f.shape[0] for f in facs]
    ev = X.double().reshape(*dims, -1)
    for i, f in enumerate(facs):
        M = f.double().to(X.device)
        front = torch.movedim(ev, i, 0)
        shape = front.shape
        ev = torch.movedim((M @ front.reshape(shape[0], -1)).reshape(shape), 0, i)
    return ev.reshape(X.shape[0], -1) + shift * X.double()


def time_kernel(fn, reps=50):
    """Average duration of fn's launches (HIP events on the current stream)."""
    fn()
    torch.cuda.synchronize()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record()
    for _ in range(reps):
        fn()
    e1.record()
    torch.cuda.synchronize()
    return e0.elapsed_time(e1) / reps * 1e-3  # seconds


def cpu_threads():
    try:
        return len(os.sched_getaffinity(0))
    except AttributeError:
        return os.cpu_count()


def bench_kron_cg(args, dev):
    from cola_amd.linalg.mixed import HipMixedCG, KroneckerEigInverse, MixedSolver
    A, facs, b = kron_workload(dev)
    n, B = b.shape
    bd = b.to(dev)
    s = N.stream_ptr(dev)

    # ---- engine: FP64-residual refinement around FP32 PCG (Kronecker eigenbasis preconditioner)
    torch.cuda.synchronize()
    t_setup = time.perf_counter()
    P = KroneckerEigInverse([f.to(dev) for f in facs], 1.0, 0.01)
    inner_tol = 1e-3 if args.inner_tol is None else args.inner_tol
    alg = HipMixedCG(tol=1e-6, inner_tol=inner_tol, P=P, chunk=args.chunk, graph=not args.no_graph)
    solver = MixedSolver(A, B, alg)
    # one-time set-up of the repeated solve, whatever --warmup is: the first call records the
    # schedule (refinements x inner steps), the second captures it as one HIP graph
    for _ in range(2):
        solver.solve(bd)
    torch.cuda.synchronize()
    t_setup = time.perf_counter() - t_setup
    for _ in range(args.warmup):
        x, info = solver.solve(bd)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        x, info = solver.solve(bd)
    torch.cuda.synchronize()
    dt = (time.perf_counter() - t0) / args.steps
    # independent FP64 check of the returned (FP64) solution
    res = (kron_apply_f64(facs, x) - bd.double()).norm(dim=0) / bd.double().norm(dim=0)
    res_x64 = float(info["rel_residual_f64"].max())
    if not (float(res.max()) <= 1e-6):
        raise RuntimeError(f"mixed solver missed the FP64 1e-6 target: {float(res.max()):.3e}")

    # ---- plain FP32 CG (the drop-in CG with the reference's defaults: tol 1e-6, 1000-step cap)
    run_batched_cg(A, bd, None, 1000, 1e-6, None, chunk=16)
    torch.cuda.synchronize()
    t1 = time.perf_counter()
    xp, _, kp, _ = run_batched_cg(A, bd, None, 1000, 1e-6, None, chunk=16)
    torch.cuda.synchronize()
    dtp = time.perf_counter() - t1
    resp = (kron_apply_f64(facs, xp) - bd.double()).norm(dim=0) / bd.double().norm(dim=0)
    plain = {"solves_per_s": B / dtp, "ms_per_solve_block": dtp * 1e3, "cg_steps": int(kp),
             "max_fp64_rel_residual": float(resp.max()), "reaches_1e-6": bool(resp.max() <= 1e-6)}

    # ---- roofline: the fused mode-2/3 Kronecker pass (one kernel), timed alone on the solve's block shape
    ld = (n + 63) // 64 * 64
    Xb = torch.randn(B, ld, device=dev)
    Yb = torch.empty_like(Xb)
    K2, K3 = [f.to(dev).contiguous() for f in facs[1:]]
    t_a = time_kernel(lambda: N.call("ck_kron_apply_last2_f32", N.ptr(K2), N.ptr(K3), B, N.ptr(Xb), ld, N.ptr(Yb),
                                      ld, s))
    flops_a = 2 * 2 * 64 * n * B  # two mode products
    bytes_a = 2 * 4 * n * B  # read the slab, write the result
    op, keep = A.hip_op()
    wb = N.q("ck_op_workspace_bytes", op, B)
    work = torch.empty(wb // 4, device=dev)
    t_mv = time_kernel(lambda: N.call("ck_op_apply", op, B, N.ptr(Xb), ld, N.ptr(Yb), ld, N.ptr(work), wb, s))
    roof = {"bound": "mfma", "kernel": "kron64_pass_a<float, false> (fused mode-2/3 Kronecker pass)",
            "achieved": flops_a / t_a / 1e12, "peak": FP32_MFMA_PEAK, "unit": "TFLOP/s",
            "frac": flops_a / t_a / 1e12 / FP32_MFMA_PEAK, "traffic": PASS_A_TRAFFIC_BYTES,
            "launch_us": t_a * 1e6, "algorithmic_flops_per_launch": flops_a,
            "algorithmic_bytes_per_launch": bytes_a, "achieved_gbs": bytes_a / t_a / 1e9,
            "full_kron_matvec_us": t_mv * 1e6, "full_kron_matvec_tflops": 3 * 2 * 64 * n * B / t_mv / 1e12}

    out = {"metric": METRIC, "value": B / dt, "unit": "solves/s", "n_gpus": 1, "steps": args.steps,
           "warmup": args.warmup, "ms_per_step": dt * 1e3, "higher_is_better": True, "scaling": "weak",
           "vs_baseline": None, "dtype": "f32 (inner CG, MFMA) + f64 (refinement residuals)",
           "data": "synthetic (seeded RBF Kronecker factors, N(0,1) rhs)",
           "config": {"workload": "kron_cg: K1xK2xK3+0.01I, N=64^3=262144, 16 rhs, to FP64-checked 1e-6",
                      "method": "FP64-residual iterative refinement around FP32 PCG, Kronecker eigenbasis preconditioner",
                      "hip_graph": alg.graph, "inner_tol": alg.inner_tol,
                      "global_batch": B, "seq_len": n, "parallelism": "single GPU",
                      "refinements": info["refinements"], "inner_cg_steps": info["inner_iterations"],
                      "max_fp64_rel_residual_solver": res_x64, "max_fp64_rel_residual_bench_check": float(res.max()),
                      "setup_s": t_setup, "plain_fp32_cg": plain,
                      "speedup_vs_plain_per_solve": (dtp / dt)},
           "roofline": roof}
    if not args.no_cpu_baseline:
        out["cpu_baseline"] = cpu_baseline_kron(facs, b, 1000, 1e-6)
    return out


def cpu_baseline_kron(facs, b, k_steps, tol, iters=640):
    """The CPU torch restatement of cola's run_batched_cg with Kronecker._matmat (what
    cola.linalg.inv(PSD(A)) @ B runs), timed for `iters` CG steps on the full 16-rhs
    system and scaled to the k_steps (the 1000-step default cap) of one call."""
    from oracle import cg as ocg
    from oracle import operators as oop
    torch.set_num_threads(cpu_threads())
    mm = oop.shifted(lambda V: oop.kron_matmat(facs, V), 0.01)
    ocg.run_batched_cg(mm, b, None, 2, tol, None)  # warm-up
    t0 = time.perf_counter()
    _, _, kk, _ = ocg.run_batched_cg(mm, b, None, iters, tol, None)
    dt = (time.perf_counter() - t0) / max(kk, 1)
    solve_s = dt * k_steps
    return {"value": b.shape[1] / solve_s, "unit": "solves/s", "cores": cpu_threads(), "kind": "port",
            "sample": f"{kk} CG steps of the 16-rhs 64^3 Kronecker system ({dt * 1e3:.1f} ms/step, fp32 torch), "
                      f"scaled to the {int(k_steps)}-step cap of one reference CG call (which does not reach 1e-6 "
                      "on this system)"}


def bench_copy(args, dev):
    """STREAM-style copy of 1 GiB buffers (4x the 256 MB Infinity Cache): the measured HBM peak."""
    n = 1 << 28
    src = torch.ones(n, device=dev)
    dst = torch.empty_like(src)
    s = N.stream_ptr(dev)
    t = time_kernel(lambda: N.call("ck_stream_copy_f32", n, N.ptr(src), N.ptr(dst), s), reps=max(args.steps, 10))
    gbs = 2 * 4 * n / t / 1e9
    return {"metric": "HBM copy bandwidth (read+write)", "value": gbs, "unit": "GB/s", "n_gpus": 1,
            "steps": max(args.steps, 10), "warmup": 1, "ms_per_step": t * 1e3, "higher_is_better": True,
            "scaling": "weak", "vs_baseline": None, "dtype": "f32", "data": "synthetic",
            "config": {"workload": "copy 1 GiB -> 1 GiB (ck_stream_copy_f32)", "bytes_per_launch": 8 * n},
            "roofline": {"bound": "hbm", "achieved": gbs, "peak": HBM_PEAK, "unit": "GB/s", "frac": gbs / HBM_PEAK,
                         "traffic": None}}


def laplacian_op(dev, m=1024, shift=1e-3):
    """5-point Dirichlet Laplacian on an m x m grid (CSR, int32) plus shift * I, built on the device."""
    n = m * m
    idx = torch.arange(n, device=dev)
    y, x = idx // m, idx % m
    rows, cols, vals = [], [], []
    for dy, dx, v in ((-1, 0, -1.0), (0, -1, -1.0), (0, 0, 4.0), (0, 1, -1.0), (1, 0, -1.0)):
        ok = (y + dy >= 0) & (y + dy < m) & (x + dx >= 0) & (x + dx < m)
        r = idx[ok]
        rows.append(r)
        cols.append(r + dy * m + dx)
        vals.append(torch.full((r.numel(), ), v, device=dev))
    A = ca.Sparse(torch.cat(vals), torch.cat(rows), torch.cat(cols), (n, n))
    return A + shift * ca.I_like(A), A


def laplacian_eigs(m, shift):
    j = np.arange(1, m + 1)
    lam = 2.0 - 2.0 * np.cos(np.pi * j / (m + 1))
    return np.sort((lam[:, None] + lam[None, :]).ravel() + shift)


def bench_csr(args, dev):
    """CSR SpMV bandwidth and plain FP32 CG on the 2-D Laplacian + 1e-3 I (the Lanczos and Hutchinson operator, and a
    4096^2 grid whose 0.7 GB of matrix data exceeds the 256 MB Infinity Cache)."""
    from cola_amd.linalg.cg import run_batched_cg as rcg
    s = N.stream_ptr(dev)
    out_sizes = {}
    for m in (1024, 4096):
        op, A = laplacian_op(dev, m=m)
        n = m * m
        got = op.hip_op()
        if got is None:
            raise RuntimeError("the shifted CSR Laplacian did not lower to an engine operator")
        cop, keep = got
        nnz = int(A.data.numel())
        per_b = {}
        for B in (1, 16):
            ld = (n + 63) // 64 * 64
            Xb = torch.randn(B, ld, device=dev)
            Yb = torch.empty_like(Xb)
            wb = N.q("ck_op_workspace_bytes", cop, B)
            work = torch.empty(max(wb, 4) // 4, device=dev)
            t = time_kernel(lambda: N.call("ck_op_apply", cop, B, N.ptr(Xb), ld, N.ptr(Yb), ld, N.ptr(work), wb, s))
            byts = 8 * nnz + 4 * (n + 1) + 8 * n * B  # values + column indices, row pointers, x read, y written
            per_b[B] = {"us": t * 1e6, "algorithmic_bytes": byts, "gbs": byts / t / 1e9, "frac": byts / t / 1e9 / HBM_PEAK}
        out_sizes[m] = {"n": n, "nnz": nnz, "spmv": per_b}
    # plain FP32 CG with the reference's defaults (tol 1e-6, normalised rhs, 1000-step cap), 1 rhs, 1024^2 grid
    op, A = laplacian_op(dev, m=1024)
    n = 1024 * 1024
    b = torch.randn(n, 1, generator=torch.Generator().manual_seed(0)).to(dev)
    for _ in range(max(1, args.warmup)):
        x, r, k, info = rcg(op, b, None, 1000, 1e-6, None, chunk=64)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    reps = max(1, args.steps // 2)
    for _ in range(reps):
        x, r, k, info = rcg(op, b, None, 1000, 1e-6, None, chunk=64)
    torch.cuda.synchronize()
    dt = (time.perf_counter() - t0) / reps
    import scipy.sparse as sp
    Ah = sp.csr_matrix((A.data.cpu().double().numpy(), A.indices.cpu().numpy(), A.indptr.cpu().numpy()), shape=(n, n))
    xh, bh = x.cpu().double().numpy()[:, 0], b.cpu().double().numpy()[:, 0]
    res = float(np.linalg.norm(Ah @ xh + 1e-3 * xh - bh) / np.linalg.norm(bh))
    steps = int(k)
    spmv = out_sizes[1024]["spmv"][1]
    # per CG step: the SpMV plus fused p.Ap, the x/r update (6 vectors) and the p update (3 vectors)
    step_bytes = spmv["algorithmic_bytes"] + 4 * n * (1 + 6 + 3)
    big = out_sizes[4096]["spmv"][16]
    return {"metric": "CSR SpMV GB/s and plain FP32 CG solves/s (2-D Laplacian + 1e-3 I)", "value": big["gbs"],
            "unit": "GB/s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup, "ms_per_step": big["us"] / 1e3,
            "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "f32 values, int32 indices",
            "data": "synthetic (5-point stencil)",
            "config": {"workload": "csr: SpMV on 1024^2 and 4096^2 grids (1 and 16 vectors); plain CG on 1024^2",
                       "grids": out_sizes,
                       "cg_1024sq": {"solves_per_s": 1 / dt, "ms_per_solve": dt * 1e3, "cg_steps": steps,
                                     "fp64_rel_residual": res, "us_per_step": dt / max(steps, 1) * 1e6,
                                     "step_algorithmic_bytes": step_bytes,
                                     "step_effective_gbs": step_bytes / (dt / max(steps, 1)) / 1e9}},
            "roofline": {"bound": "hbm", "kernel": "CSR SpMV, 4096^2 grid, 16 vectors (matrix data > Infinity Cache)",
                         "achieved": big["gbs"], "peak": HBM_PEAK, "unit": "GB/s", "frac": big["frac"],
                         "traffic": None, "launch_us": big["us"], "algorithmic_bytes_per_launch": big["algorithmic_bytes"]},
            **({} if args.no_cpu_baseline else {"cpu_baseline": cpu_baseline_csr_cg(A, b, steps)})}


def _cpu_laplacian_matmat(A, shift=1e-3):
    """The reference's CPU operator apply for the shifted CSR Laplacian: torch's sparse CSR
    product (Sparse._matmat, operators.py:77-78; torch_fns.py:79-80) plus shift * V."""
    torch.set_num_threads(cpu_threads())
    n = A.shape[0]
    M = torch.sparse_csr_tensor(A.indptr.cpu().to(torch.int64), A.indices.cpu().to(torch.int64), A.data.cpu(),
                                size=(n, n))
    return lambda V: M @ V + shift * V


def cpu_baseline_csr_cg(A, b, steps_gpu):
    """The oracle's run_batched_cg (cola's CG restated, FP32 torch) on the CPU with the CSR
    apply, the same rhs, tolerance 1e-6 and cap 1000: one whole solve (a few seconds)."""
    from oracle import cg as ocg
    mm = _cpu_laplacian_matmat(A)
    bc = b.cpu()
    ocg.run_batched_cg(mm, bc, None, 2, 1e-6, None)
    t0 = time.perf_counter()
    _, _, k, _ = ocg.run_batched_cg(mm, bc, None, 1000, 1e-6, None)
    dt = time.perf_counter() - t0
    return {"value": 1 / dt, "unit": "solves/s", "cores": cpu_threads(), "kind": "port",
            "sample": f"one whole plain CG solve on the 1024^2 Laplacian ({int(k)} steps, the GPU run took "
                      f"{int(steps_gpu)}), {dt * 1e3 / max(int(k), 1):.2f} ms per step, torch sparse CSR"}


def cpu_baseline_lanczos(A, s0):
    """The oracle's Lanczos with full double Gram-Schmidt (lanczos.py:235-296 restated, FP32
    torch) and its eigh/Ritz-vector step, the whole 120-step run on the 1024^2 Laplacian, on the
    CPU (about half a minute to a minute of host time: its steps sweep all m + 2 basis columns,
    as the reference's do)."""
    from oracle import lanczos as olz
    mm = _cpu_laplacian_matmat(A)
    n = A.shape[0]
    t0 = time.perf_counter()
    olz.lanczos_eigs(mm, n, s0.cpu(), 120, 1e-7, torch.float32, torch.float64)
    dt = time.perf_counter() - t0
    return {"value": 1 / dt, "unit": "eigensolves/s", "cores": cpu_threads(), "kind": "port",
            "sample": f"one whole 120-step eigensolve ({dt:.1f} s), torch sparse CSR apply, FP64 eigh of T"}


def cpu_baseline_hutch(A, reps=3):
    """The oracle's Hutchinson estimate with 64 Rademacher probes (diag_trace.py restated) on the
    CPU: one 64-column CSR product and the probe sums, `reps` estimates."""
    from oracle import hutch as oh
    mm = _cpu_laplacian_matmat(A)
    n = A.shape[0]
    g = torch.Generator().manual_seed(0)
    t0 = time.perf_counter()
    for _ in range(reps):
        Z = (torch.randint(0, 2, (n, 64), generator=g) * 2 - 1).float()
        oh.trace_from_probes(mm, Z)
    dt = (time.perf_counter() - t0) / reps
    return {"value": 1 / dt, "unit": "estimates/s", "cores": cpu_threads(), "kind": "port",
            "sample": f"{reps} estimates of 64 probes each ({dt * 1e3:.0f} ms per estimate, probes drawn on the host)"}


def cpu_baseline_slq(facs, probes=8):
    """The oracle's SLQ (slq.py:37-52 restated: batched Lanczos with full re-orthogonalisation,
    eigh of T, quadrature) with the Kronecker apply on the CPU, for `probes` of the 32 Rademacher
    probes, scaled to 32."""
    from oracle import operators as oop
    from oracle import unary as ou
    torch.set_num_threads(cpu_threads())
    mm = oop.shifted(lambda V: oop.kron_matmat(facs, V), 0.01)
    n = 64**3
    g = torch.Generator().manual_seed(5)
    Z = (torch.randint(0, 2, (n, probes), generator=g) * 2 - 1).float()
    t0 = time.perf_counter()
    ou.slq_fwd(mm, n, torch.log, Z, 30, 1e-6, torch.float32, torch.float64)
    dt = (time.perf_counter() - t0) * 32 / probes
    return {"value": 1 / dt, "unit": "logdets/s", "cores": cpu_threads(), "kind": "port",
            "sample": f"{probes} of the 32 probes x 30 steps ({dt * probes / 32:.1f} s), scaled to 32 probes"}


def bench_dense_cg(args, dev):
    """A = X X^T/256 + 0.1 I, N=1024, one N(0,1) rhs (seed 0), CG to the reference tolerance: the
    persistent fused solve (one launch per solve) and the chained-launch path on the same system."""
    g = torch.Generator().manual_seed(0)
    X = torch.randn(1024, 256, generator=g)
    b = torch.randn(1024, generator=g)
    A = X @ X.T / 256 + 0.1 * torch.eye(1024)
    op = ca.PSD(ca.Dense(A.to(dev)))
    bd = b.to(dev)[:, None]

    def timed(fused):
        for _ in range(1 + args.warmup):  # one set-up call (workspaces, first lowering), then the warmup
            out = run_batched_cg(op, bd, None, 1000, 1e-6, None, chunk=32, fused=fused)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(args.steps):
            out = run_batched_cg(op, bd, None, 1000, 1e-6, None, chunk=32, fused=fused)
        torch.cuda.synchronize()
        return (time.perf_counter() - t0) / args.steps, out

    dt, (x, r, k, info) = timed(True)
    dtc, (xc, rc, kc, ic) = timed(False)
    res = float((A.double() @ x.cpu().double()[:, 0] - b.double()).norm() / b.double().norm())
    # GPU time of the solve alone (the reset and solve kernels back to back, HIP events on the
    # engine's stream) for the roofline line
    from cola_amd.linalg._engine import lower
    from cola_amd.linalg.cg import _fused_buffers
    aop = lower(op)
    state, work, *_ = _fused_buffers(dev, 1024, 1, 1000)
    xr = torch.empty((2, 1024, 1), dtype=torch.float32, device=dev)
    t_kernel = time_kernel(lambda: N.call("ck_cg_fused", aop[0], None, 1, N.ptr(bd), bd.stride(0), bd.stride(1), None, 0,
                                          0, N.ptr(xr[0]), 1, 1, N.ptr(xr[1]), 1, 1, N.ptr(state), 1e-6, 1000,
                                          N.ptr(work), work.numel() * 8, 0, 0, 0, 0, N.stream_ptr(dev)), reps=20)
    step_bytes = 4 * 1024 * 1024 + 8 * 4 * 1024  # A once per step plus the vector streams
    ach = int(k) * step_bytes / t_kernel / 1e9
    from oracle import cg as ocg
    torch.set_num_threads(cpu_threads())
    t1 = time.perf_counter()
    reps = 0
    while time.perf_counter() - t1 < 2.0:
        xo, io = ocg.cg(lambda V: A @ V, b[:, None], tol=1e-6, max_iters=1000)
        reps += 1
    dto = (time.perf_counter() - t1) / reps
    return {"metric": "CG solves/sec (dense N=1024, 1 rhs, reference tol 1e-6)", "value": 1 / dt,
            "unit": "solves/s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup, "ms_per_step": dt * 1e3,
            "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "f32",
            "data": "synthetic (seeded X, rhs)",
            "config": {"workload": "dense_cg: A = X X^T/256 + 0.1 I, N=1024, 1 rhs, tol 1e-6 (persistent fused CG)",
                       "cg_steps": int(k), "oracle_steps": int(io["iterations"] - 1), "fp64_rel_residual": res,
                       "chained_launch_solves_per_s": 1 / dtc, "chained_cg_steps": int(kc),
                       "solve_gpu_us": t_kernel * 1e6, "us_per_cg_step_gpu": t_kernel * 1e6 / max(int(k), 1)},
            "roofline": {"bound": "hbm", "kernel": "fused_cg_kernel<1, 4, 2, true> (whole solve, A rows held in registers)",
                         "achieved": ach, "peak": HBM_PEAK, "unit": "GB/s", "frac": ach / HBM_PEAK, "traffic": None,
                         "algorithmic_bytes_per_step": step_bytes,
                         "note": "latency-bound: one grid-wide exchange per step; A stays in registers"},
            "cpu_baseline": {"value": 1 / dto, "unit": "solves/s", "cores": cpu_threads(), "kind": "port",
                             "sample": f"{reps} full solves of the oracle's CG (fp32 torch) in 2 s"}}


def bench_lanczos(args, dev):
    """Lanczos top-32 of the 1024^2-grid Laplacian + 1e-3 I, 120 steps, full CGS2."""
    from cola_amd.linalg import HipLanczos, eig
    from cola_amd.linalg.lanczos import run_lanczos
    op, A = laplacian_op(dev)
    op = ca.SelfAdjoint(op)
    n = op.shape[0]
    g = torch.Generator().manual_seed(42)
    s0 = torch.randn(n, generator=g).to(dev)
    alg = HipLanczos(start_vector=s0, max_iters=120, tol=1e-7)
    for _ in range(1 + args.warmup):  # one set-up call, then the warmup
        vals, vecs = eig(op, 32, "LM", alg)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    reps = max(1, args.steps // 5)
    for _ in range(reps):
        vals, vecs = eig(op, 32, "LM", alg)
    torch.cuda.synchronize()
    dt = (time.perf_counter() - t0) / reps
    exact = laplacian_eigs(1024, 1e-3)[-32:]
    err = float(np.abs(np.sort(vals.cpu().double().numpy()) - exact).max())
    # algorithmic bytes: SpMV (values, columns, rowptr, x, y) + the i basis vectors read three
    # times per step (project; the fused apply + second project, whose second read is served
    # by the caches; apply) + the w traffic
    spmv = 4 * (2 * 5238784 + (n + 1) + 2 * n)
    reorth = sum(3 * i * 4 * n + 2 * 2 * 4 * n for i in range(1, 121))
    total = 120 * spmv + reorth
    # the engine's block re-orthogonalisation (S = 16): same start, same accuracy bar
    S = 16
    balg = HipLanczos(start_vector=s0, max_iters=120, tol=1e-7, reorth="block", block=S)
    for _ in range(1 + args.warmup):
        bvals, _ = eig(op, 32, "LM", balg)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(reps):
        bvals, _ = eig(op, 32, "LM", balg)
    torch.cuda.synchronize()
    bdt = (time.perf_counter() - t0) / reps
    # bytes: SpMV + the window passes (three reads of the window's columns) + per completed block
    # two passes of (project: old + S columns; apply: old columns + S columns read and written)
    bwin = 0
    for i in range(1, 121):
        c0 = (i // S) * S + 1
        jlo = max(1, c0 - 1)
        bwin += 3 * (i - jlo + 1) * 4 * n + 2 * 2 * 4 * n
    bblk = sum(2 * 4 * n * (2 * (i - S) + 3 * S) for i in range(2 * S, 121, S))
    bflops = sum(2 * 2 * 2 * (i - S) * 16 * n for i in range(2 * S, 121, S))
    btotal = 120 * spmv + bwin + bblk
    block_line = {"value": 1 / bdt, "unit": "eigensolves/s", "ms_per_step": bdt * 1e3, "block": S,
                  "max_rel_err_top32_vs_fp64_oracle_same_start": _golden_rel(
                      "lanczos_laplacian_1024sq", "top32_ritz_fp64", bvals.cpu().numpy()),
                  "algorithmic_bytes": btotal, "block_pass_mfma_flops": bflops,
                  "roofline": {"bound": "hbm", "achieved": btotal / bdt / 1e9, "peak": HBM_PEAK, "unit": "GB/s",
                               "frac": btotal / bdt / 1e9 / HBM_PEAK, "traffic": None}}
    return {"metric": "Lanczos eigensolves/sec (2-D Laplacian 1024^2, 120 steps, CGS2, top-32)",
            "value": 1 / dt, "unit": "eigensolves/s", "ms_per_step": dt * 1e3, "dtype": "f32 (+f64 tridiagonal)",
            "block_reorth": block_line,
            "config": {"workload": "lanczos", "n": n, "nnz": 5238784, "steps": 120,
                       "max_abs_err_top32_vs_closed_form": err,
                       "max_rel_err_top32_vs_fp64_oracle_same_start": _golden_rel(
                           "lanczos_laplacian_1024sq", "top32_ritz_fp64", vals.cpu().numpy()),
                       "algorithmic_bytes": total,
                       "effective_gbs": total / dt / 1e9},
            "roofline": {"bound": "hbm", "achieved": total / dt / 1e9, "peak": HBM_PEAK, "unit": "GB/s",
                         "frac": total / dt / 1e9 / HBM_PEAK, "traffic": None},
            **({} if args.no_cpu_baseline else {"cpu_baseline": cpu_baseline_lanczos(A, s0)})}


def bench_hutch(args, dev):
    """Hutchinson trace of the Laplacian + 1e-3 I with 64 packed Rademacher probes."""
    from cola_amd.linalg import hutch_trace_csr
    op, A = laplacian_op(dev)
    n = op.shape[0]
    for _ in range(1 + args.warmup):  # one set-up call (workspace, first lowering), then the warmup
        tr = hutch_trace_csr(op, 64, seed=0)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for i in range(args.steps):
        tr = hutch_trace_csr(op, 64, seed=i)
    torch.cuda.synchronize()
    dt = (time.perf_counter() - t0) / args.steps
    exact = 4.001 * n
    byts = 4 * 2 * 5238784 + 4 * (n + 1)  # values, columns, rowptr (probe words are recomputed in the pass)
    # roofline: the device pass alone (popcount trace with in-pass probe words + final sum), HIP events
    import ctypes
    hop, keep = op.hip_op()
    wb = N.q("ck_trace_workspace_bytes", n)
    work = torch.empty(wb // 8 + 1, dtype=torch.float64, device=dev)
    out = torch.empty(1, dtype=torch.float64, device=dev)
    s = N.stream_ptr(dev)

    def passes():
        N.call("ck_trace_csr_rademacher_seeded", hop, 1, ctypes.c_uint64(7), N.ptr(out), N.ptr(work), wb, s)
    t_k = time_kernel(passes, reps=50)
    return {"metric": "Hutchinson trace estimates/sec (64 Rademacher probes, CSR 1024^2 Laplacian)",
            "value": 1 / dt, "unit": "estimates/s", "ms_per_step": dt * 1e3, "dtype": "f32 values, popcount probes",
            "config": {"workload": "hutch", "estimate": float(tr), "exact": exact,
                       "rel_err": abs(float(tr) - exact) / exact, "expected_std_rel": 361.9 / exact,
                       "algorithmic_bytes": byts, "device_us": t_k * 1e6},
            "roofline": {"bound": "hbm", "kernel": "trace_stream<SeededWords> + trace_bits_final",
                         "achieved": byts / t_k / 1e9, "peak": HBM_PEAK, "unit": "GB/s",
                         "frac": byts / t_k / 1e9 / HBM_PEAK, "traffic": None},
            **({} if args.no_cpu_baseline else {"cpu_baseline": cpu_baseline_hutch(A)})}


def bench_slq(args, dev):
    """SLQ logdet of K1xK2xK3 + 0.01 I, 32 Rademacher probes x 30 steps, FP64 tridiagonal."""
    from cola_amd.linalg import HipSLQ, logdet
    A, facs, _ = kron_workload(dev)
    alg = HipSLQ(num_probes=32, max_iters=30, key=5)
    for _ in range(1 + args.warmup):  # one set-up call, then the warmup
        est = logdet(A, alg)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        est = logdet(A, alg)
    torch.cuda.synchronize()
    dt = (time.perf_counter() - t0) / args.steps
    lam = [torch.linalg.eigvalsh(f.double()) for f in facs]
    exact = float(torch.log((lam[0][:, None, None] * lam[1][None, :, None] * lam[2][None, None, :]) + 0.01).sum())
    # algorithmic bytes: per step the 32-probe Kronecker apply (read and write 32 vectors of 64^3)
    # and each probe's re-orthogonalisation (three reads of its i basis vectors, w traffic)
    vb = 4 * 64**3
    slq_bytes = sum(2 * 32 * vb + 32 * (3 * i + 4) * vb for i in range(1, 31))
    return {"metric": "SLQ log-determinants/sec (64^3 Kronecker, 32 probes x 30 steps)",
            "value": 1 / dt, "unit": "logdets/s", "ms_per_step": dt * 1e3, "dtype": "f32 (+f64 tridiagonal)",
            "config": {"workload": "slq", "estimate_abs": float(est), "exact": exact,
                       "rel_err_vs_abs_exact": abs(float(est) - abs(exact)) / abs(exact),
                       "rel_err_vs_fp64_oracle_same_probes": _golden_rel("slq_kron64", "logdet_fp64", float(est)),
                       "note": "cola's logdet returns |tr log A| (logdet.py:111-117)", "algorithmic_bytes": slq_bytes},
            "roofline": {"bound": "hbm", "kernel": "whole SLQ run (Kronecker applies + re-orthogonalisation), wall time",
                         "achieved": slq_bytes / dt / 1e9, "peak": HBM_PEAK, "unit": "GB/s",
                         "frac": slq_bytes / dt / 1e9 / HBM_PEAK, "traffic": None},
            **({} if args.no_cpu_baseline else {"cpu_baseline": cpu_baseline_slq([f.cpu() for f in facs])})}


def _golden_rel(section, key, got):
    """Relative difference from the FP64 oracle value stored in tests/golden/full_config.json
    for this exact workload (None when the fixture is absent)."""
    path = os.path.join(os.path.dirname(os.path.abspath(__file__)), "tests", "golden", "full_config.json")
    if not os.path.exists(path):
        return None
    ref = np.asarray(json.load(open(path))[section][key], dtype=np.float64)
    got = np.sort(np.asarray(got, dtype=np.float64)) if ref.ndim else abs(float(got))
    return float(np.max(np.abs(got - np.abs(ref)) / np.abs(ref)))


def dense_rel_residual(K, shift, x, b):
    """max_j ||b_j - (K + shift I) x_j|| / ||b_j|| in FP64 with K as stored (fp32), on the engine."""
    from cola_amd._blocks import ld_of
    n, B = x.shape
    ld = ld_of(n)
    X = torch.zeros((B, ld), dtype=torch.float64, device=K.device)
    X[:, :n] = x.T.double()
    Y = torch.empty_like(X)
    N.call("ck_dense_apply_f64acc", n, N.ptr(K), K.stride(0), 1.0, shift, B, N.ptr(X), ld, N.ptr(Y), ld,
           N.stream_ptr(K.device))
    bd = b.T.double()
    return ((Y[:, :n] - bd).norm(dim=1) / bd.norm(dim=1)).cpu().numpy()


def bench_learned_cg(args, dev):
    """Dense RBF systems on 16384 points in [0,1]^4 (lengthscale ~ LogU[0.05,1], noise ~
    LogU[1e-4,1e-1], 8 N(0,1) rhs each).  value: solves/s at an FP64-checked relative residual
    of 1e-6 of the learned (or, when it measurably captures less, pivoted-Cholesky) rank-64
    preconditioner inside FP64-residual iterative refinement around FP32 PCG.  "plain": the same
    refinement around unpreconditioned FP32 CG -- the reference's CG, which alone does not reach
    1e-6 on these systems (its FP32 runs are reported too)."""
    from cola_amd.linalg import learned as L
    from cola_amd.linalg.cg import cg
    n, B = args.n, 8
    # --- training: top-64 Lanczos eigenvectors of seeded instances, Adam on the engine
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    insts = L.make_training_set(range(args.train_instances), args.train_n, m=64, ell_range=(0.05, 1.0), device=dev)
    torch.cuda.synchronize()
    t_data = time.perf_counter() - t0
    net = L.PointMLP(4, 64, device=dev, seed=0)
    probe = insts[:min(64, len(insts))]
    loss0 = L.mean_loss(net, probe)
    t1 = time.perf_counter()
    losses = L.train(net, insts, epochs=args.train_epochs, lr=2e-3, seed=0)
    torch.cuda.synchronize()
    t_train = time.perf_counter() - t1
    loss1 = L.mean_loss(net, probe)
    del insts, probe
    # --- held-out test systems and their preconditioners (construction timed apart)
    systems = []
    for j in range(args.systems):
        X, ell, noise = L.sample_instance(100000 + j, n)
        Xd = X.to(dev)
        torch.cuda.synchronize()
        ts = time.perf_counter()
        K = L.rbf_matrix(Xd, ell)
        Kop = ca.Dense(K)
        A = ca.PSD(Kop + noise * ca.I_like(Kop))
        torch.cuda.synchronize()
        t_op = time.perf_counter() - ts
        b = torch.randn(n, B, generator=torch.Generator().manual_seed(200000 + j)).to(dev)
        torch.cuda.synchronize()
        ts = time.perf_counter()
        Pl = L.LearnedPreconditioner(K, Xd, net, noise)
        torch.cuda.synchronize()
        t_pl = time.perf_counter() - ts
        Pc = L.PivotedCholeskyPreconditioner(K, 64, noise)
        P, rep = L.select_preconditioner(K, Xd, noise, candidates={"learned": Pl, "pivoted_cholesky": Pc}, A=A)
        torch.cuda.synchronize()
        systems.append({"K": K, "X": Xd, "A": A, "b": b, "shift": float(np.float32(noise)), "ell": ell, "noise": noise,
                        "Pl": Pl, "Pc": Pc, "P": P, "choice": rep["choice"], "operator_s": t_op, "learned_build_s": t_pl,
                        "select_s": time.perf_counter() - ts})

    def fp32_run(sd, P):
        """The reference's CG (FP32, cap 1000) with a 10x tighter recursive target, so that its true
        residual has a chance to reach the FP64-checked tolerance."""
        torch.cuda.synchronize()
        t = time.perf_counter()
        x, info = cg(sd["A"], sd["b"], P=P, tol=args.tol / 10, max_iters=1000, chunk=16)
        torch.cuda.synchronize()
        dt = time.perf_counter() - t
        res = dense_rel_residual(sd["K"], sd["shift"], x, sd["b"])
        return {"steps": int(info["iterations"]) - 1, "s": dt, "max_res": float(res.max()),
                "solved": int((res <= args.tol).sum())}

    per = []
    for sd in systems:
        row = {"ell": sd["ell"], "noise": sd["noise"], "choice": sd["choice"], "operator_s": sd["operator_s"],
               "learned_build_s": sd["learned_build_s"], "select_s": sd["select_s"],
               "resid_trace_learned": sd["Pl"].residual_trace, "resid_trace_pivchol": sd["Pc"].residual_trace,
               "fp32_only": {name: fp32_run(sd, P) for name, P in (("plain", None), ("pivchol", sd["Pc"]),
                                                                   ("learned", sd["Pl"]))}}
        per.append(row)
    itol = 1e-4 if args.inner_tol is None else args.inner_tol
    refined = {}
    for name, pick, reps in (("learned", lambda sd: sd["P"], args.steps), ("plain", lambda sd: None, min(args.steps, 3)),
                             ("pivchol", lambda sd: sd["Pc"], min(args.steps, 3))):
        refined[name] = timed_refined(systems, [pick(sd) for sd in systems], B, args, itol, reps)
        for row, r in zip(per, refined[name]["per_system"]):
            row[name + "_refined"] = r
    head, plain = refined["learned"], refined["plain"]
    total_rhs = B * len(systems)
    value = head["solved"] / head["s"]
    plain_rate = plain["solved"] / plain["s"]
    # --- roofline: the dense 8-rhs matvec (K + noise I) the solves spend their time in, timed with
    # HIP events on the engine's stream
    from cola_amd._blocks import ld_of
    ld = ld_of(n)
    Xb = torch.randn(B, ld, device=dev)
    Yb = torch.empty_like(Xb)
    op, keep = systems[0]["A"].hip_op()
    wb = N.q("ck_op_workspace_bytes", op, B)
    work = torch.empty(max(wb, 4) // 4, device=dev)
    t_mv = time_kernel(lambda: N.call("ck_op_apply", op, B, N.ptr(Xb), ld, N.ptr(Yb), ld, N.ptr(work), wb,
                                      N.stream_ptr(dev)), reps=20)
    roof = dense_product_roof(op, n, B, t_mv)
    roof["kernel"] += ", K + noise I"
    sketch = bench_sketch(systems[0], net, n, dev)
    out = {"metric": METRIC, "value": value, "unit": "solves/s", "n_gpus": 1, "steps": args.steps,
           "warmup": args.warmup, "ms_per_step": head["s"] * 1e3, "higher_is_better": True, "scaling": "weak",
           "vs_baseline": None,
           "dtype": "f32 (matvec, PCG) + f64 (refinement residuals, Woodbury core) + bf16 MFMA (preconditioner sketch)",
           "data": "synthetic (seeded points, lengthscales, noise, N(0,1) rhs; network trained here on seeded instances)",
           "config": {"workload": f"learned_cg: {len(systems)} dense RBF systems, N={n} points in [0,1]^4, "
                                  f"lengthscale~LogU[0.05,1], noise~LogU[1e-4,1e-1], {B} rhs each, to FP64-checked "
                                  f"{args.tol:g}",
                      "global_batch": total_rhs, "seq_len": n, "parallelism": "single GPU",
                      "step": f"one pass of refined PCG over all {len(systems)} systems ({total_rhs} rhs), "
                              f"{args.streams} systems in flight at once",
                      "streams": args.streams,
                      "rhs_solved": head["solved"], "rhs_total": total_rhs, "inner_tol": itol,
                      "plain_refined_solves_per_s": plain_rate, "plain_refined_rhs_solved": plain["solved"],
                      "ratio_vs_plain": value / plain_rate if plain_rate > 0 else None,
                      "pivchol_refined_solves_per_s": refined["pivchol"]["solved"] / refined["pivchol"]["s"],
                      "inner_steps_total": {k: v["inner_steps"] for k, v in refined.items()},
                      "training": {"instances": args.train_instances, "points": args.train_n,
                                   "epochs": args.train_epochs, "lanczos_data_s": t_data, "train_s": t_train,
                                   "energy_loss_before": loss0, "energy_loss_after": loss1,
                                   "last_step_loss": float(losses[-1]) if len(losses) else None},
                      "systems": per},
           "roofline": roof, "sketch_bf16": sketch}
    if not args.no_cpu_baseline:
        out["cpu_baseline"] = cpu_baseline_refined(systems, B, args.tol, itol, head["per_system"])
    del systems, per
    torch.cuda.empty_cache()
    if not args.no_kron:
        # the structured Kronecker workload (64^3, 16 rhs) as a labelled sub-object
        ka = argparse.Namespace(**vars(args))
        ka.no_cpu_baseline, ka.inner_tol = True, None
        kr = bench_kron_cg(ka, dev)
        out["kron_cg"] = {"value": kr["value"], "unit": kr["unit"], "ms_per_step": kr["ms_per_step"],
                          "config": kr["config"], "roofline": kr["roofline"]}
    return out


def bench_sketch(sd, net, n, dev):
    """The preconditioner's sketch product K G (n x n by n x 64) on BF16 MFMA (K as a bf16
    pair, ck_sketch_bf16) against the FP32 operator apply on 64 columns, both timed with HIP
    events, and the learned preconditioner's build time either way."""
    from cola_amd._blocks import ld_of
    from cola_amd.linalg import learned as L
    k, ld = 64, ld_of(n)
    K = sd["K"]
    G = torch.randn(k, ld, device=dev)
    G16 = torch.empty((k, ld), dtype=torch.int16, device=dev)
    Gr = torch.zeros((k, ld), device=dev)
    Y = torch.zeros((k, ld), device=dev)
    s = N.stream_ptr(dev)
    N.call("ck_round_bf16", n, k, N.ptr(G), ld, N.ptr(G16), ld, N.ptr(Gr), ld, s)
    t16 = time_kernel(lambda: N.call("ck_sketch_bf16", n, k, N.ptr(K), K.stride(0), 1.0, 0.0, N.ptr(G16), ld, None, 0,
                                     N.ptr(Y), ld, 1, s), reps=10)
    op, keep = ca.Dense(K).hip_op()
    wb = N.q("ck_op_workspace_bytes", op, k)
    work = torch.empty(max(wb, 4) // 4, device=dev)
    t32 = time_kernel(lambda: N.call("ck_op_apply", op, k, N.ptr(G), ld, N.ptr(Y), ld, N.ptr(work), wb, s), reps=5)
    builds = {}
    for name, flag in (("bf16_mfma", True), ("fp32", False)):
        torch.cuda.synchronize()
        t = time.perf_counter()
        L.LearnedPreconditioner(K, sd["X"], net, sd["noise"], bf16_sketch=flag)
        torch.cuda.synchronize()
        builds[name] = (time.perf_counter() - t) * 1e3
    by = 4 * n * n + 2 * k * n + 4 * k * n
    flops = 2 * 2 * n * n * k  # two bf16 products (hi, lo) per element
    return {"kernel": "sketch_bf16_kernel<64, split> (K G, K as bf16 hi + lo, FP32 accumulation)",
            "launch_us": t16 * 1e6, "achieved_GBps": by / t16 / 1e9, "frac_hbm": by / t16 / 1e9 / HBM_PEAK,
            "mfma_TFLOPs": flops / t16 / 1e12, "frac_bf16_mfma": flops / t16 / 1e12 / 2500.0,
            "fp32_apply_64cols_us": t32 * 1e6, "speedup_vs_fp32": t32 / t16,
            "learned_build_ms": builds}


def timed_refined(systems, precs, B, args, itol, reps):
    """FP64-residual refinement around FP32 (P)CG on every system: one set-up call per solver
    (it records the refinement schedule), args.warmup untimed passes, then `reps` timed passes
    over all systems, args.streams systems in flight at once (solve_concurrent); every rhs is
    checked in FP64 afterwards."""
    from cola_amd.linalg.mixed import HipMixedCG, MixedSolver, solve_concurrent
    solvers = []
    for sd, P in zip(systems, precs):
        alg = HipMixedCG(tol=args.tol, inner_tol=itol, inner_max_iters=1000, max_refinements=args.max_refinements,
                         P=P, chunk=args.chunk)
        solvers.append(MixedSolver(sd["A"], B, alg))
    rhs = [sd["b"] for sd in systems]
    for sv, b in zip(solvers, rhs):
        sv.solve(b)
    for _ in range(args.warmup):
        solve_concurrent(solvers, rhs, args.streams)
    torch.cuda.synchronize()
    t = time.perf_counter()
    infos = []
    for _ in range(max(1, reps)):
        infos = solve_concurrent(solvers, rhs, args.streams)
    torch.cuda.synchronize()
    dt = (time.perf_counter() - t) / max(1, reps)
    solved, steps, per = 0, 0, []
    for (x, info), sd in zip(infos, systems):
        res = dense_rel_residual(sd["K"], sd["shift"], x, sd["b"])
        solved += int((res <= args.tol).sum())
        steps += int(sum(info["inner_iterations"]))
        per.append({"refinements": info["refinements"], "inner_steps": [int(k) for k in info["inner_iterations"]],
                    "max_res": float(res.max()), "solved": int((res <= args.tol).sum())})
    del solvers
    return {"s": dt, "solved": solved, "inner_steps": steps, "per_system": per, "timed_passes": max(1, reps)}


def cpu_baseline_refined(systems, B, tol, itol, per_system, max_refinements=30):
    """The reference algorithm on the host: the oracle's run_batched_cg (cola's CG restated in
    torch, FP32) with the same preconditioner (its Woodbury apply in torch), inside the same FP64
    refinement.  The sample is one converging solve (FP64-checked) of the system that needed the
    fewest inner steps on the GPU; its time per inner CG step and per FP64 residual is scaled by
    the inner steps and refinements every system took on the GPU, which gives the time the same
    converging solves of the whole workload take on the host."""
    from oracle import cg as ocg
    torch.set_num_threads(cpu_threads())
    cost = [sum(r["inner_steps"]) for r in per_system]
    j = int(np.argmin(cost))
    sd = systems[j]
    K = sd["K"].cpu()
    K64 = K.double()  # residual operator (the matrix as stored, FP64 arithmetic): set-up, not timed
    b64 = sd["b"].cpu().double()
    s = sd["shift"]
    P = sd["P"]
    prec = None
    if P is not None:
        F64, core, ps = P.F.cpu().double(), P.core_inv.cpu(), P.s

        def prec(V):
            t = F64.T @ V.double()
            return ((V.double() - F64 @ (core @ t)) / ps).float()
    x64 = torch.zeros(K.shape[0], B, dtype=torch.float64)
    t_res = t_cg = 0.0
    steps = refinements = 0
    for _ in range(max_refinements):
        t0 = time.perf_counter()
        r = b64 - (K64 @ x64 + s * x64)
        rel = float((r.norm(dim=0) / b64.norm(dim=0)).max())
        t_res += time.perf_counter() - t0
        if rel <= tol:
            break
        t0 = time.perf_counter()
        d, _, k, _ = ocg.run_batched_cg(lambda V: K @ V + s * V, r.float(), None, 1000, itol, prec)
        t_cg += time.perf_counter() - t0
        steps += int(k)
        refinements += 1
        x64 += d.double()
    res = ((K64 @ x64 + s * x64) - b64).norm(dim=0) / b64.norm(dim=0)
    solved = int((res <= tol).sum())
    per_step = t_cg / max(steps, 1)
    per_res = t_res / (refinements + 1)
    total = sum(sum(r["inner_steps"]) * per_step + (r["refinements"] + 1) * per_res for r in per_system)
    return {"value": B * len(systems) / total, "unit": "solves/s", "cores": cpu_threads(), "kind": "port",
            "sample": f"one converging solve of system {j} ({B} rhs, {solved} reached {tol:g} FP64-checked): the oracle's "
                      f"CG (FP32 torch) with the same preconditioner, {steps} inner steps in {refinements} refinements, "
                      f"{per_step * 1e3:.1f} ms per CG step and {per_res * 1e3:.1f} ms per FP64 residual on "
                      f"{cpu_threads()} host threads ({t_cg + t_res:.1f} s), scaled to the inner steps and refinements "
                      f"of all {len(systems)} systems' GPU solves"}


def bench_dense_matvec(args, dev):
    """The dense 8-rhs matvec of the learned_cg workload alone (one 16384-point RBF system of
    it, K + noise I): the launch rocprofv3 counter passes measure."""
    from cola_amd._blocks import ld_of
    from cola_amd.linalg import learned as L
    n, B = args.n, 8
    X, ell, noise = L.sample_instance(100000, n)
    K = L.rbf_matrix(X.to(dev), ell)
    Kop = ca.Dense(K)
    A = ca.PSD(Kop + noise * ca.I_like(Kop))
    ld = ld_of(n)
    Xb = torch.randn(B, ld, device=dev)
    Yb = torch.empty_like(Xb)
    op, keep = A.hip_op()
    wb = N.q("ck_op_workspace_bytes", op, B)
    work = torch.empty(max(wb, 4) // 4, device=dev)
    reps = max(args.steps, 10)
    t = time_kernel(lambda: N.call("ck_op_apply", op, B, N.ptr(Xb), ld, N.ptr(Yb), ld, N.ptr(work), wb,
                                   N.stream_ptr(dev)), reps=reps)
    roof = dense_product_roof(op, n, B, t)
    # the same product without the symmetry flag (the whole matrix read), for comparison
    full = N.CkOp.from_buffer_copy(op)
    full.flags = 0
    t_full = time_kernel(lambda: N.call("ck_op_apply", full, B, N.ptr(Xb), ld, N.ptr(Yb), ld, N.ptr(work), wb,
                                        N.stream_ptr(dev)), reps=reps)
    return {"metric": "dense 8-rhs matvec products/s (K + noise I, K 16384^2 fp32)", "value": 1.0 / t,
            "unit": "products/s", "n_gpus": 1, "steps": reps, "warmup": 1, "ms_per_step": t * 1e3,
            "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "f32", "data": "synthetic",
            "config": {"workload": f"dense_matvec: {n}^2 fp32 RBF matrix + noise I, {B} rhs",
                       "algorithmic_bytes_per_launch": roof["algorithmic_bytes_per_launch"],
                       "full_product_us": t_full * 1e6,
                       "full_product_gbs": (4 * n * n + 2 * 4 * n * B) / t_full / 1e9},
            "roofline": roof}


def gp_systems(nsys, dev, bf16=True):
    """512 (nsys) RBF systems: n_i ~ U{256..4096} (generator seed 0), system i from manual_seed(i):
    points U[0,1]^3, lengthscale LogU[0.05,0.5], one N(0,1) rhs; noise 1e-2."""
    from cola_amd.linalg.batched import BatchedSystems
    sizes = torch.randint(256, 4097, (nsys, ), generator=torch.Generator().manual_seed(0)).tolist()
    pts, ells, rhs = [], [], []
    for i, n in enumerate(sizes):
        g = torch.Generator().manual_seed(i)
        pts.append(torch.rand(n, 3, generator=g))
        u = float(torch.rand(1, generator=g, dtype=torch.float64))
        ells.append(float(np.exp(np.log(0.05) + u * (np.log(0.5) - np.log(0.05)))))
        rhs.append(torch.randn(n, generator=g))
    sy = BatchedSystems.rbf(pts, ells, 1e-2, dev, bf16=bf16)
    b = sy.concat([r.to(dev) for r in rhs])
    return sy, b, sizes, ells, pts


def bench_batched_cg(args, dev):
    """512 uneven dense GP systems; FP64 refinement to 1e-8 around batched PCG (bf16 storage
    where it contracts, per-system learned / pivoted-Cholesky rank-64 preconditioners) vs plain FP32 CG."""
    from cola_amd.linalg import learned as L
    from cola_amd.linalg.batched import BatchedCG, BatchedMixedSolver, BatchedPrecond, autotune, time_matvec
    nsys = args.systems_batched
    tol = args.batched_tol
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    sy, b, sizes, ells, pts = gp_systems(nsys, dev)
    torch.cuda.synchronize()
    t_build = time.perf_counter() - t0
    t1 = time.perf_counter()
    rows, tune = autotune(sy, np.ones(nsys, dtype=bool), max_iters=1000)
    t_tune = time.perf_counter() - t1
    # preconditioners: rank-64 pivoted Cholesky and a 3-input network trained on the engine
    torch.cuda.synchronize()
    t2 = time.perf_counter()
    pcc = BatchedPrecond.pivoted_cholesky(sy, 64)
    torch.cuda.synchronize()
    t_pc = time.perf_counter() - t2
    t3 = time.perf_counter()
    insts = L.make_training_set(range(args.batched_train), 1024, m=64, din=3, ell_range=(0.05, 0.5), device=dev)
    net = L.PointMLP(3, 64, device=dev, seed=0)
    losses = L.train(net, insts, epochs=args.train_epochs, lr=2e-3, seed=0)
    torch.cuda.synchronize()
    t_train = time.perf_counter() - t3
    del insts
    t4 = time.perf_counter()
    pcl = BatchedPrecond.learned(sy, pts, net)
    torch.cuda.synchronize()
    t_pl = time.perf_counter() - t4
    best = BatchedPrecond.best_of(pcc, pcl)

    # correction-solve tolerance 3e-5: the hardest systems' FP32 floor (~6e-4 after a correction)
    # sets the refinement count either way; tighter inner solves cost steps, looser ones a 4th pass
    itol = 3e-5 if args.inner_tol is None else args.inner_tol

    def run(P, label):
        solver = BatchedMixedSolver(sy, rows_per_tile=rows, inner_max_iters=1000, bf16=True, precond=P)
        # one-time set-up, whatever --warmup is (the first call screens bf16 storage and
        # builds the solver's launch state)
        solver.solve(b, tol=tol, inner_tol=itol, chunk=args.chunk_batched)
        for _ in range(args.warmup):
            solver.solve(b, tol=tol, inner_tol=itol, chunk=args.chunk_batched)
        torch.cuda.synchronize()
        t = time.perf_counter()
        for _ in range(args.steps):
            x, info = solver.solve(b, tol=tol, inner_tol=itol, chunk=args.chunk_batched)
        torch.cuda.synchronize()
        dt = (time.perf_counter() - t) / args.steps
        rel = solver.residual(np.ones(nsys, dtype=bool))  # FP64 residual of the returned x
        return solver, x, {"s": dt, "solved": int((rel <= tol).sum()), "solves_per_s": int((rel <= tol).sum()) / dt,
                           "refinements": info["refinements"],
                           "inner_iterations_total": int(info["inner_iterations"].sum()),
                           "bf16_systems_final": info["bf16_systems_final"], "max_rel_residual": float(rel.max()),
                           "history_max_rel": info["history"],
                           "per_refinement_active_steps_bf16": info["per_refinement"]}

    variants = {}
    solver, x, variants["best"] = run(best, "best")
    # a-priori bf16 admissibility: 2 ||K_bf16 - K||_2 (power-iteration estimate) against 5% of the shift
    ratio = 2.0 * solver.bf16_norm_estimate / sy.shift.cpu().numpy().astype(np.float64)
    screen = {"admitted": int(solver.admissible.sum()), "threshold": 0.05,
              "ratio_2norm_over_shift_min_median_max": [float(ratio.min()), float(np.median(ratio)), float(ratio.max())]}
    for name, P in (("pivoted_cholesky", pcc), ("learned", pcl), ("none", None)):
        variants[name] = run(P, name)[2]
    head = variants["best"]
    # independent spot check of three systems with a dense FP64 product
    s32 = float(np.float32(1e-2))
    spot = []
    for s_ in [0, nsys // 2, nsys - 1]:
        A = sy.matrix(s_).double() + s32 * torch.eye(sizes[s_], dtype=torch.float64, device=dev)
        bs = sy.segment(b, s_).double()
        spot.append(float((A @ sy.segment(x, s_) - bs).norm() / bs.norm()))
    # plain FP32 batched CG on the same systems (fp32 storage, no preconditioner)
    plain = BatchedCG(sy, rows, 1000)
    plain.solve(b, tol_rel=tol / 10, chunk=args.chunk_batched)
    torch.cuda.synchronize()
    t5 = time.perf_counter()
    xp, kp = plain.solve(b, tol_rel=tol / 10, chunk=args.chunk_batched)
    torch.cuda.synchronize()
    dtp = time.perf_counter() - t5
    solver.x64.copy_(xp.double())
    relp = solver.residual(np.ones(nsys, dtype=bool))
    plain_res = {"s": dtp, "solved_1e-8": int((relp <= tol).sum()), "solved_1e-6": int((relp <= 1e-6).sum()),
                 "iterations_total": int(kp.sum()), "max_rel_residual": float(relp.max()),
                 "solves_per_s_1e-8": int((relp <= tol).sum()) / dtp}
    # roofline: the batched matvec over all systems, fp32 storage
    bcg = BatchedCG(sy, rows, 1000)
    t_mv = time_matvec(bcg, reps=5)
    mbytes = float(np.sum(sy.sizes * sy.lda * 4)) + 8.0 * float(sy.sizes.sum())
    roof = {"bound": "hbm", "kernel": f"bcg_matvec<{rows // 4}> (all {nsys} systems, fp32, one launch)",
            "achieved": mbytes / t_mv / 1e9, "peak": HBM_PEAK, "unit": "GB/s", "frac": mbytes / t_mv / 1e9 / HBM_PEAK,
            "traffic": None, "launch_us": t_mv * 1e6, "algorithmic_bytes_per_launch": mbytes}
    sum_n2 = int(np.sum(sy.sizes.astype(np.int64)**2))
    return {"metric": "batched GP solves/sec to 1e-8 (FP64-checked): learned/pivoted-Cholesky PCG + bf16/FP64 "
                      "refinement vs plain FP32 CG",
            "value": head["solves_per_s"], "unit": "solves/s", "n_gpus": 1, "steps": args.steps,
            "warmup": args.warmup, "ms_per_step": head["s"] * 1e3, "higher_is_better": True, "scaling": "weak",
            "vs_baseline": None, "dtype": "bf16/f32 storage + f32 accumulate (inner PCG), f64 (residuals, Woodbury)",
            "data": "synthetic (seeded points, lengthscales, rhs)",
            "config": {"workload": f"batched_cg: {nsys} RBF systems n~U{{256..4096}} in [0,1]^3, noise 1e-2, 1 rhs, "
                                   f"to FP64-checked {tol:g}",
                       "sum_n2": sum_n2, "build_s": t_build, "autotune_s": t_tune, "rows_per_tile": rows,
                       "autotune_us": {str(k): v * 1e6 for k, v in tune.items()},
                       "pivchol_build_s": t_pc, "learned": {"train_instances": args.batched_train, "train_s": t_train,
                                                            "build_s": t_pl, "last_loss": float(losses[-1]),
                                                            "systems_choosing_learned": int(best.pick.sum())},
                       "inner_tol": itol, "variants": variants, "bf16_screen": screen, "spot_check_fp64": spot, "plain_fp32": plain_res,
                       "speedup_vs_plain_time": dtp / head["s"]},
            "roofline": roof}


def cpu_baseline_dense(sd, n, B, k_steps, tol, iters=130):
    """The oracle's plain CG (the reference algorithm, torch on the host) on the first system:
    `iters` steps timed (about 10 s on 16 host threads), scaled to the steps the engine's plain
    CG took."""
    from oracle import cg as ocg
    torch.set_num_threads(cpu_threads())
    K = sd["K"].cpu()
    b = sd["b"].cpu()
    s = sd["shift"]
    mm = lambda V: K @ V + s * V  # noqa: E731
    t = time.perf_counter()
    ocg.cg(mm, b, tol=1e-30, max_iters=iters)
    per_step = (time.perf_counter() - t) / iters
    total = per_step * max(k_steps, 1)
    return {"value": B / total, "unit": "solves/s", "cores": cpu_threads(), "kind": "port",
            "sample": f"{iters} CG steps of the first {n}-point system x {B} rhs ({per_step * 1e3:.1f} ms/step), "
                      f"scaled to the {k_steps} steps plain CG takes on it"}


def workloads():
    """--workload name -> bench function."""
    return {"learned_cg": bench_learned_cg, "kron_cg": bench_kron_cg, "dense_cg": bench_dense_cg,
            "batched_cg": bench_batched_cg, "lanczos": bench_lanczos, "hutch": bench_hutch, "slq": bench_slq,
            "csr": bench_csr, "copy": bench_copy, "dense_matvec": bench_dense_matvec}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=10)
    ap.add_argument("--warmup", type=int, default=2)
    ap.add_argument("--workload", default="learned_cg")
    ap.add_argument("--tol", type=float, default=1e-6)
    ap.add_argument("--chunk", type=int, default=8)
    ap.add_argument("--inner-tol", type=float, default=None,
                    help="correction-solve tolerance (default 1e-3 for kron_cg, where one eigenbasis-preconditioned "
                         "step reaches it, 3e-5 for batched_cg, 1e-4 for learned_cg)")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-kron", action="store_true", help="leave out the Kronecker sub-object of learned_cg")
    ap.add_argument("--no-graph", action="store_true", help="launch the refinement schedule eagerly (no HIP graph)")
    ap.add_argument("--n", type=int, default=16384, help="points per system (learned_cg)")
    ap.add_argument("--systems", type=int, default=8, help="held-out systems (learned_cg)")
    ap.add_argument("--streams", type=int, default=2,
                    help="systems solved at once on their own streams (learned_cg; 1 = one after another)")
    ap.add_argument("--max-refinements", type=int, default=30, help="refinement cap (learned_cg)")
    ap.add_argument("--train-instances", type=int, default=2000)
    ap.add_argument("--train-n", type=int, default=1024)
    ap.add_argument("--train-epochs", type=int, default=4)
    ap.add_argument("--systems-batched", type=int, default=512, help="systems (batched_cg)")
    ap.add_argument("--batched-tol", type=float, default=1e-8)
    ap.add_argument("--chunk-batched", type=int, default=16)
    ap.add_argument("--batched-train", type=int, default=1000, help="training instances of the 3-D network")
    args = ap.parse_args()
    if args.gpus != 1:
        print(json.dumps({"error": "this engine runs on one GPU; --gpus > 1 is not supported"}))
        sys.exit(2)
    dev = torch.device("cuda:0")
    N.load()
    fn = workloads()[args.workload]
    out = fn(args, dev)
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
