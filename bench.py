#!/usr/bin/env python3
"""Benchmark of the Pauli-operator path on one MI355X.

Default workload (the headline): 20 qubits, 2000 random Pauli terms
(labels uniform over {I,X,Y,Z}, complex N(0,1) coefficients): one step is the
full CSR build (2^20 rows x G distinct x masks, uint64 indices, complex128
values) followed by one complex128 CSR matvec on a normalised random state.
`value` is whole-step throughput in CSR nonzeros per second; inputs are
resident in device memory when timing starts.

Also reported (same JSON line, key "extra"), unless --no-extra: the 24-qubit
Heisenberg ring matrix-free apply on 8 states, FP64 vs mixed precision (GB/s,
% of HBM peak, speedup, error vs FP64); the 256-operator uneven batch; the
28-qubit k-local apply; the reference's giant Hamiltonians (H10, H11, H12, HJ);
the eigensolver-step operations; the box's plain copy/fill/read rates.

roofline: the dominant kernel's algorithmic bytes per launch / its mean
duration from HIP events on the launch stream.  cpu_baseline: the oracle's C
restatement of qrusty's RowwiseUnsafeChunked/1000 build + spmat_dot_densevec
on a bounded sample of rows, on every host core this process may use (capped
at the CPU share the environment grants, OMP_NUM_THREADS); the core count, the
CPU model and the sampled fraction are recorded.
"""
from __future__ import annotations

import argparse
import ctypes
import json
import os
import shutil
import statistics
import sys
import time

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, HERE)

HBM_PEAK_GBPS = 8000.0


def log(msg):
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def load_traffic(kernel: str, workload: str):
    path = os.path.join(HERE, "profiles", "traffic.json")
    try:
        with open(path) as f:
            t = json.load(f)
        e = t.get(f"{kernel}@{workload}")
        return None if e is None else e["traffic_bytes"]
    except (OSError, ValueError, KeyError, TypeError):
        return None


def cpu_info() -> dict:
    """The host CPUs this process may use: every core of its affinity mask,
    capped at the CPU share the machine grants one GPU job when the
    environment states one (OMP_NUM_THREADS), plus nproc and the CPU model."""
    try:
        affinity = len(os.sched_getaffinity(0))
    except AttributeError:
        affinity = os.cpu_count() or 1
    share = os.environ.get("OMP_NUM_THREADS", "")
    threads = min(affinity, int(share)) if share.isdigit() and int(share) > 0 else affinity
    model = ""
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    model = line.split(":", 1)[1].strip()
                    break
    except OSError:
        pass
    return {"threads": max(1, threads), "affinity_cpus": affinity, "nproc": os.cpu_count(),
            "omp_num_threads": share or None, "cpu_model": model}


# ---------------------------------------------------------------------------
def bench_csr(args, torch, qa):
    from qrusty_amd import _lib as L
    from qrusty_amd import workloads

    nq, T = 20, 2000
    labels, coeffs = workloads.random_op(nq, T, seed=workloads.SEED_CFG2)
    op = qa.SparsePauliOp([qa.Pauli(l) for l in labels], coeffs)
    h = op._handle(L.QR_PHASE_ROWWISE)
    N, G, nnz = 1 << nq, h.G, h.nnz
    log(f"csr workload: n={nq} T={T} G={G} nnz={nnz} ({24 * nnz / 1e9:.1f} GB CSR)")
    dev = torch.device("cuda", 0)
    indptr = torch.empty(N + 1, dtype=torch.int64, device=dev)
    indices = torch.empty(nnz, dtype=torch.int64, device=dev)
    data = torch.empty(nnz, dtype=torch.complex128, device=dev)
    x = torch.from_numpy(workloads.random_states(N, 1, seed=workloads.SEED_CFG2 + 1)[0]).to(dev)
    y = torch.empty(N, dtype=torch.complex128, device=dev)
    stream = torch.cuda.current_stream()
    sh = ctypes.c_void_p(stream.cuda_stream)
    P = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731

    def step(ev=None):
        if ev:
            ev[0].record(stream)
        L.check(L.lib.qr_csr_build(h.h, P(indptr), P(indices), P(data), sh))
        if ev:
            ev[1].record(stream)
        L.check(L.lib.qr_csr_matvec(N, N, nnz, P(indptr), P(indices), P(data), P(x), P(y), sh))
        if ev:
            ev[2].record(stream)

    for _ in range(args.warmup):
        step()
    torch.cuda.synchronize()
    evs = [[torch.cuda.Event(enable_timing=True) for _ in range(3)] for _ in range(args.steps)]
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for k in range(args.steps):
        step(evs[k])
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    build_ms = [e[0].elapsed_time(e[1]) for e in evs]
    mv_ms = [e[1].elapsed_time(e[2]) for e in evs]
    ms_per_step = 1e3 * wall / args.steps
    b_build = 24 * nnz + 8 * (N + 1)
    b_mv = 24 * nnz + 8 * (N + 1) + 32 * N
    bm, mm = statistics.mean(build_ms), statistics.mean(mv_ms)
    res = {
        "workload": "csr_build+matvec n=20 T=2000 random", "N": N, "T": T, "G": G, "nnz": nnz,
        "ms_per_step": ms_per_step, "value": nnz / (ms_per_step / 1e3),
        "build_ms": bm, "matvec_ms": mm,
        "build_nnz_per_s": nnz / (bm / 1e3), "build_GBps": b_build / bm / 1e6,
        "matvec_GBps": b_mv / mm / 1e6,
    }
    res["build_pct_hbm"] = 100 * res["build_GBps"] / HBM_PEAK_GBPS
    res["matvec_pct_hbm"] = 100 * res["matvec_GBps"] / HBM_PEAK_GBPS
    # the kernels that run here: k_csr_build_words and k_csr_matvec_staged (rows
    # of 256+ entries)
    dom = ("k_csr_build_words", bm, b_build) if bm >= mm else ("k_csr_matvec_staged", mm, b_mv)
    res["roofline"] = {
        "kernel": dom[0], "bound": "hbm", "achieved": dom[2] / dom[1] / 1e6, "peak": HBM_PEAK_GBPS,
        "unit": "GB/s", "frac": dom[2] / dom[1] / 1e6 / HBM_PEAK_GBPS,
        "traffic": load_traffic(dom[0], "n20_T2000"),
        "algorithmic_bytes": dom[2], "mean_ms": dom[1],
    }
    log(f"build {bm:.3f} ms ({res['build_GBps']:.0f} GB/s), matvec {mm:.3f} ms "
        f"({res['matvec_GBps']:.0f} GB/s), step {ms_per_step:.3f} ms")

    # invariant check of the timed output on sampled rows (no oracle): each
    # row holds the columns r ^ x_g in ascending order, and y is the row dot x
    if not args.no_check:
        import numpy as np
        xm = np.empty(h.T, dtype=np.uint64)
        L.check(L.lib.qr_op_terms(h.h, xm.ctypes.data_as(L.u64p), None, None))
        gx = np.unique(xm)
        rows = np.random.default_rng(1).choice(N, size=64, replace=False)
        sel = torch.from_numpy(rows).to(dev)
        ind_h = indices.view(N, G)[sel].cpu().numpy().view(np.uint64)
        dat_h = data.view(N, G)[sel].cpu().numpy()
        xh = x.cpu().numpy()
        ok = bool(np.array_equal(indptr[sel].cpu().numpy(), rows * G))
        for i, r in enumerate(rows):
            ok &= bool(np.array_equal(ind_h[i], np.sort(np.uint64(r) ^ gx)))
        yr = np.einsum("ij,ij->i", dat_h, xh[ind_h.astype(np.int64)])
        ok &= bool(np.allclose(y[sel].cpu().numpy(), yr, rtol=1e-12, atol=1e-14))
        res["invariants_sampled_rows_ok"] = ok
    del indices, data
    torch.cuda.empty_cache()
    return res, (labels, coeffs)


def cpu_baseline_csr(labels, coeffs, target_s=4.0):
    """Oracle (C restatement of RowwiseUnsafeChunked/1000 + spmat_dot_densevec)
    on a bounded sample of rows; median of 3 runs after 1 warm-up."""
    from oracle import oracle as orc
    from qrusty_amd import workloads
    p = orc.Params(labels, coeffs)
    info = cpu_info()
    nthr = info["threads"]
    x = workloads.random_states(p.N, 1, seed=workloads.SEED_CFG2 + 1)[0]

    def run(rows):
        t0 = time.perf_counter()
        ip, ind, dat = orc.build_csr(p, 0, rows, step=1000, nthreads=nthr)
        orc.spmat_dot_densevec(ip, ind, dat, x, nthreads=nthr)
        return time.perf_counter() - t0, len(ind)

    rows = 4096
    t, _ = run(rows)
    rows = int(min(p.N, max(4096, rows * target_s / max(t, 1e-3))))
    rows = (rows // 1000) * 1000 or 1000
    run(rows)  # warm-up
    times = []
    for _ in range(3):
        t, nnz = run(rows)
        times.append(t)
    med = statistics.median(times)
    return {"value": nnz / med, "unit": "nnz/s", "cores": nthr, "kind": "port",
            "sample": f"rows 0..{rows} of 2^20 ({nnz} nnz, {100 * rows / p.N:.1f}% of the rows): "
                      f"RowwiseUnsafeChunked/1000 build + spmat_dot_densevec, median of 3 after "
                      f"1 warm-up, {nthr} threads",
            "full_row_set": rows == p.N, "rows_timed": rows, "rows_total": p.N,
            "median_s": med, "host": info}


# ---------------------------------------------------------------------------
def bench_apply_one(args, torch, qa, precision):
    """24-qubit Heisenberg ring, 8 states, one precision only: `steps` applies
    with <psi|H|psi> after `warmup` untimed ones (a short program for profiler
    counter passes: every dispatch of the apply kernel is the same call)."""
    from qrusty_amd import _lib as L
    from qrusty_amd import workloads
    nq, nvec = 24, 8
    labels, coeffs = workloads.heisenberg_ring(nq, seed=workloads.SEED_CFG3)
    op = qa.SparsePauliOp([qa.Pauli(l) for l in labels], coeffs)
    h = op._handle(L.QR_PHASE_ROWWISE)
    N = 1 << nq
    mixed = precision == "mixed"
    dt = torch.complex64 if mixed else torch.complex128
    prec = L.QR_PREC_MIXED if mixed else L.QR_PREC_FP64
    g = torch.Generator(device="cuda")
    g.manual_seed(workloads.SEED_CFG3 + 1)
    x = torch.randn(nvec, N, dtype=dt, device="cuda", generator=g)
    x /= torch.linalg.vector_norm(x, dim=1, keepdim=True)
    y = torch.empty_like(x)
    e = torch.empty(2 * nvec, dtype=torch.float64, device="cuda")
    stream = torch.cuda.current_stream()
    sh = ctypes.c_void_p(stream.cuda_stream)
    P = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    call = lambda: L.check(L.lib.qr_pauli_apply(h.h, prec, nvec, P(x), P(y), P(e), sh))  # noqa: E731
    for _ in range(args.warmup):
        call()
    a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    torch.cuda.synchronize()
    a.record(stream)
    for _ in range(args.steps):
        call()
    b.record(stream)
    torch.cuda.synchronize()
    ms = a.elapsed_time(b) / args.steps
    byts = nvec * N * 2 * (8 if mixed else 16)
    log(f"apply {precision}: {ms:.3f} ms ({byts / ms / 1e6:.0f} GB/s)")
    return {"workload": f"heisenberg ring n=24, 8 states, {precision} apply + <psi|H|psi>",
            "ms": ms, "GBps": byts / ms / 1e6, "pct_hbm": 100 * byts / ms / 1e6 / HBM_PEAK_GBPS,
            "algorithmic_bytes": byts}


def bench_apply(args, torch, qa):
    """24-qubit Heisenberg ring, 8 states: FP64 vs mixed matrix-free apply."""
    import numpy as np
    from qrusty_amd import _lib as L
    from qrusty_amd import workloads

    nq, nvec = 24, 8
    labels, coeffs = workloads.heisenberg_ring(nq, seed=workloads.SEED_CFG3)
    op = qa.SparsePauliOp([qa.Pauli(l) for l in labels], coeffs)
    h = op._handle(L.QR_PHASE_ROWWISE)
    N = 1 << nq
    dev = torch.device("cuda", 0)
    x64 = torch.from_numpy(workloads.random_states(N, nvec, seed=workloads.SEED_CFG3 + 1)).to(dev)
    x32 = x64.to(torch.complex64)
    y64 = torch.empty_like(x64)
    y32 = torch.empty_like(x32)
    e64 = torch.empty(2 * nvec, dtype=torch.float64, device=dev)
    e32 = torch.empty(2 * nvec, dtype=torch.float64, device=dev)
    stream = torch.cuda.current_stream()
    sh = ctypes.c_void_p(stream.cuda_stream)
    P = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731

    def timed(prec, xt, yt, et, reps):
        for _ in range(2):
            L.check(L.lib.qr_pauli_apply(h.h, prec, nvec, P(xt), P(yt), P(et), sh))
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        torch.cuda.synchronize()
        a.record(stream)
        for _ in range(reps):
            L.check(L.lib.qr_pauli_apply(h.h, prec, nvec, P(xt), P(yt), P(et), sh))
        b.record(stream)
        torch.cuda.synchronize()
        return a.elapsed_time(b) / reps

    reps = max(3, args.steps)
    ms64 = timed(L.QR_PREC_FP64, x64, y64, e64, reps)
    ms32 = timed(L.QR_PREC_MIXED, x32, y32, e32, reps)

    # expectation only: y is never written (algorithmic bytes nvec*N*s_in)
    def timed_expect(prec, xt, et, reps):
        L.check(L.lib.qr_pauli_apply(h.h, prec, nvec, P(xt), None, P(et), sh))
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        torch.cuda.synchronize()
        a.record(stream)
        for _ in range(reps):
            L.check(L.lib.qr_pauli_apply(h.h, prec, nvec, P(xt), None, P(et), sh))
        b.record(stream)
        torch.cuda.synchronize()
        return a.elapsed_time(b) / reps

    ee = torch.empty_like(e32)
    ms32_e = timed_expect(L.QR_PREC_MIXED, x32, ee, reps)
    ms64_e = timed_expect(L.QR_PREC_FP64, x64, ee, reps)
    b64 = nvec * N * 32
    b32 = nvec * N * 16
    ry = (torch.linalg.vector_norm((y32.to(torch.complex128) - y64).reshape(-1)) /
          torch.linalg.vector_norm(y64.reshape(-1))).item()
    E64 = e64.cpu().numpy().view(np.complex128)
    E32 = e32.cpu().numpy().view(np.complex128)
    rE = float(np.max(np.abs(E32 - E64) / np.abs(E64)))
    # |dE| against the scale of the sum, ||psi|| ||H psi|| (the states are
    # normalised): the error measure that cancellation in E does not inflate
    nHpsi = torch.linalg.vector_norm(y64, dim=1).cpu().numpy()
    rE_norm = float(np.max(np.abs(E32 - E64) / nHpsi))
    # the same FP64 path on the complex64-rounded states: separates the kernel's
    # arithmetic error from the rounding of psi itself (|E| of a traceless H in
    # a random state is small, so the latter dominates the relative error)
    xr = x32.to(torch.complex128)
    er = torch.empty_like(e64)
    L.check(L.lib.qr_pauli_apply(h.h, L.QR_PREC_FP64, nvec, P(xr), P(y64), P(er), sh))
    torch.cuda.synchronize()
    ER = er.cpu().numpy().view(np.complex128)
    rE_kernel = float(np.max(np.abs(E32 - ER) / np.abs(ER)))
    rE_input = float(np.max(np.abs(ER - E64) / np.abs(E64)))
    res = {
        "workload": "heisenberg ring n=24, 8 states, matrix-free apply + <psi|H|psi>",
        "G": h.G, "T": h.T,
        "fp64_ms": ms64, "fp64_GBps": b64 / ms64 / 1e6, "fp64_pct_hbm": 100 * b64 / ms64 / 1e6 / HBM_PEAK_GBPS,
        "mixed_ms": ms32, "mixed_GBps": b32 / ms32 / 1e6, "mixed_pct_hbm": 100 * b32 / ms32 / 1e6 / HBM_PEAK_GBPS,
        "mixed_speedup_vs_fp64": ms64 / ms32,
        "mixed_rel_err_y_vs_fp64": ry, "mixed_rel_err_expect_vs_fp64": rE,
        "mixed_rel_err_expect_vs_fp64_same_rounded_input": rE_kernel,
        "expect_rel_change_from_rounding_psi_to_c64": rE_input,
        "mixed_err_expect_over_norm_Hpsi": rE_norm,
        "expect_only_fp64_ms": ms64_e, "expect_only_mixed_ms": ms32_e,
        "expect_only_mixed_pct_hbm": 100 * (b32 // 2) / ms32_e / 1e6 / HBM_PEAK_GBPS,
        "algorithmic_bytes": {"fp64": b64, "mixed": b32},
    }
    log(f"apply fp64 {ms64:.3f} ms ({res['fp64_GBps']:.0f} GB/s) mixed {ms32:.3f} ms "
        f"({res['mixed_GBps']:.0f} GB/s) speedup {ms64 / ms32:.2f}x err y {ry:.2e} E {rE:.2e} "
        f"(kernel only {rE_kernel:.2e}, from rounding psi {rE_input:.2e}; "
        f"|dE|/||H psi|| {rE_norm:.2e}); expectation only: fp64 {ms64_e:.3f} ms, mixed {ms32_e:.3f} ms")
    return res


def bench_batch(args, torch, qa):
    """256 operators of 8..18 qubits and 10..5000 random terms (log-uniform):
    every CSR built and applied to one state each, in one graph launch."""
    import numpy as np
    from qrusty_amd import workloads

    specs = workloads.uneven_batch(256, workloads.SEED_CFG4)
    ops = [qa.SparsePauliOp([qa.Pauli(l) for l in lab], co) for lab, co in specs]
    b = qa.Batch(ops, keep_csr=True)
    nnz = sum(h.nnz for h in b._h)
    rows = sum(1 << h.num_qubits for h in b._h)
    log(f"batch workload: {len(ops)} operators, {rows} rows, nnz={nnz} ({24 * nnz / 1e9:.1f} GB CSR)")
    b.set_states([workloads.random_states(1 << h.num_qubits, 1, seed=workloads.SEED_CFG4 + k)[0]
                  for k, h in enumerate(b._h)])
    t0 = time.perf_counter()
    best = b.tune()
    tune_s = time.perf_counter() - t0
    log(f"batch tuned in {tune_s:.1f} s: {best}")
    stream = torch.cuda.current_stream()
    for _ in range(args.warmup):
        b.run()
    torch.cuda.synchronize()
    ev = [torch.cuda.Event(enable_timing=True) for _ in range(args.steps + 1)]
    ev[0].record(stream)
    for k in range(args.steps):
        b.run()
        ev[k + 1].record(stream)
    torch.cuda.synchronize()
    ms = [ev[k].elapsed_time(ev[k + 1]) for k in range(args.steps)]
    m = statistics.mean(ms)
    # algorithmic bytes: CSR written (24 B/nnz + indptr), then y = A x (x read,
    # y written).  The split form's matvec pass reads every CSR back, the fused
    # form none.  Operators of more than 2^21 entries run the single-operator
    # kernels.
    split = bool(best.get("split", 0))
    big = [k for k, h in enumerate(b._h) if h.nnz > 1 << 21]
    nnz_big = sum(b._h[k].nnz for k in big)
    nnz_reread = nnz if split else 0
    byts = 24 * nnz + 8 * (rows + len(ops)) + 24 * nnz_reread + 32 * rows
    res = {"workload": "batch of 256 uneven random operators (8..18 qubits, 10..5000 terms): "
                       "CSR build + one matvec each, one graph launch",
           "operators": len(ops), "rows": rows, "nnz": nnz, "ms_per_step": m,
           "nnz_per_s": nnz / (m / 1e3), "GBps": byts / m / 1e6,
           "pct_hbm": 100 * byts / m / 1e6 / HBM_PEAK_GBPS, "tuning": best, "tune_s": tune_s,
           "single_operator_route": {"operators": len(big), "nnz_frac": nnz_big / nnz},
           "csr_read_back_nnz": nnz_reread}
    if not args.no_check:
        # invariant check: every operator's indptr is r*G and one sampled row per
        # operator holds sorted r ^ x_g
        from qrusty_amd import _lib as L
        ok = True
        rng = np.random.default_rng(2)
        for k, h in enumerate(b._h):
            N, G = 1 << h.num_qubits, h.G
            ip, ind, _ = b.csr(k)
            r = int(rng.integers(N))
            xm = np.empty(h.T, dtype=np.uint64)
            L.check(L.lib.qr_op_terms(h.h, xm.ctypes.data_as(L.u64p), None, None))
            got = ind[r * G:(r + 1) * G].cpu().numpy().view(np.uint64)
            ok &= bool(np.array_equal(got, np.sort(np.uint64(r) ^ np.unique(xm))))
            ok &= int(ip[N].item()) == N * G
        res["invariants_ok"] = ok
    log(f"batch {m:.3f} ms/step, {res['nnz_per_s']:.3e} nnz/s, {res['GBps']:.0f} GB/s")
    del b
    torch.cuda.empty_cache()
    return res


def bench_large_apply(args, torch, qa):
    """28 qubits, 10000 k-local terms (weights 1..4, real N(0,1) coefficients),
    one 4 GiB complex128 state: mixed apply + <psi|H|psi> (the headline form
    of this case) and the FP64 apply for reference."""
    import numpy as np
    from qrusty_amd import _lib as L
    from qrusty_amd import workloads

    nq, T = 28, 10000
    labels, coeffs = workloads.k_local_op(nq, T, seed=workloads.SEED_CFG5)
    op = qa.SparsePauliOp([qa.Pauli(l) for l in labels], coeffs)
    h = op._handle(L.QR_PHASE_ROWWISE)
    N = 1 << nq
    g = torch.Generator(device="cuda")
    g.manual_seed(workloads.SEED_CFG5 + 1)
    x64 = torch.randn(N, dtype=torch.complex128, device="cuda", generator=g)
    x64 /= torch.linalg.vector_norm(x64)
    x32 = x64.to(torch.complex64)
    y64, y32 = torch.empty_like(x64), torch.empty_like(x32)
    e64 = torch.empty(2, dtype=torch.float64, device="cuda")
    e32 = torch.empty(2, dtype=torch.float64, device="cuda")
    stream = torch.cuda.current_stream()
    sh = ctypes.c_void_p(stream.cuda_stream)
    P = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731

    def timed(prec, xt, yt, et, reps):
        L.check(L.lib.qr_pauli_apply(h.h, prec, 1, P(xt), P(yt), P(et), sh))
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        torch.cuda.synchronize()
        a.record(stream)
        for _ in range(reps):
            L.check(L.lib.qr_pauli_apply(h.h, prec, 1, P(xt), P(yt), P(et), sh))
        b.record(stream)
        torch.cuda.synchronize()
        return a.elapsed_time(b) / reps

    reps = max(2, min(args.steps, 5))
    ms32 = timed(L.QR_PREC_MIXED, x32, y32, e32, reps)
    ms64 = timed(L.QR_PREC_FP64, x64, y64, e64, reps)
    ny = torch.linalg.vector_norm(y64).item()
    ry = torch.linalg.vector_norm(y32.to(torch.complex128) - y64).item() / ny
    E64 = complex(*e64.cpu().numpy())
    E32 = complex(*e32.cpu().numpy())
    b32, b64 = N * 16, N * 32
    res = {
        "workload": "k-local n=28 T=10000 (weights 1..4), 1 state: mixed apply + <psi|H|psi>",
        "T": h.T, "G": h.G, "mixed_ms": ms32, "fp64_ms": ms64,
        "mixed_GBps": b32 / ms32 / 1e6, "mixed_pct_hbm": 100 * b32 / ms32 / 1e6 / HBM_PEAK_GBPS,
        "fp64_GBps": b64 / ms64 / 1e6, "mixed_speedup_vs_fp64": ms64 / ms32,
        "sign_evals_per_s_mixed": N * h.T / (ms32 / 1e3),
        "group_macs_per_s_mixed": N * h.G / (ms32 / 1e3),
        "mixed_rel_err_y_vs_fp64": ry,
        "expect_fp64": [E64.real, E64.imag], "expect_mixed": [E32.real, E32.imag],
        "mixed_abs_err_expect": abs(E32 - E64),
        "mixed_err_expect_over_norm_Hpsi": abs(E32 - E64) / ny,
    }
    log(f"k-local 28q: mixed {ms32:.1f} ms ({res['mixed_GBps']:.0f} GB/s), fp64 {ms64:.1f} ms, "
        f"err y {ry:.2e}, |dE| {abs(E32 - E64):.2e} (|E| {abs(E64):.2e}, ||Hpsi|| {ny:.2e})")
    del x64, x32, y64, y32
    torch.cuda.empty_cache()
    return res


def bench_giant(args, torch, qa):
    """The reference's giant Hamiltonians, the operators its timing script
    builds with RowwiseUnsafeChunked/1000 (pyqrusty/tests/perf_giant.py:33-40;
    data from pyqrusty/tests/H_fixtures.py in tests/golden): the whole CSR
    build where it fits in device memory (H10 64 GB, HJ 90 GB), else every row
    built through a reused window of about 16 GB (H11 382 GB, H12 327 GB);
    the matrix-free apply of each to one state (mixed and FP64); the CPU port
    of RowwiseUnsafeChunked/1000 on a bounded sample of rows."""
    import numpy as np
    from oracle import oracle as orc
    from qrusty_amd import _lib as L
    with open(os.path.join(HERE, "tests", "golden", "hamiltonians.json")) as f:
        ham = json.load(f)
    stream = torch.cuda.current_stream()
    sh = ctypes.c_void_p(stream.cuda_stream)
    P = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    nthr = cpu_info()["threads"]
    out = {}

    def timed(fn, reps):
        fn()
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        torch.cuda.synchronize()
        a.record(stream)
        for _ in range(reps):
            fn()
        b.record(stream)
        torch.cuda.synchronize()
        return a.elapsed_time(b) / reps

    for name in ("H10", "H11", "H12", "HJ"):
        h_ = ham[f"py_{name}"]
        labels = h_["labels"]
        coeffs = [complex(a, b) for a, b in h_["coeffs"]]
        op = qa.SparsePauliOp([qa.Pauli(l) for l in labels], coeffs)
        h = op._handle(L.QR_PHASE_ROWWISE)
        nq, G = h.num_qubits, h.G
        N = 1 << nq
        nnz = N * G
        res = {"num_qubits": nq, "terms": h.T, "groups": G, "nnz": nnz,
               "csr_GB": 24 * nnz / 1e9}
        # operator tables: host path (qr_op_create) against the device path
        # (qr_op_create_device), best of 3 after one untimed device call
        arr = (ctypes.c_char_p * len(labels))(*[s_.encode() for s_ in labels])
        cbuf = np.ascontiguousarray(np.asarray(coeffs, dtype=np.complex128)).view(np.float64)

        def create(device):
            hh = ctypes.c_void_p()
            t0 = time.perf_counter()
            if device:
                L.check(L.lib.qr_op_create_device(arr, cbuf.ctypes.data_as(L.f64p), len(labels),
                                                  L.QR_PHASE_ROWWISE, sh, ctypes.byref(hh)))
            else:
                L.check(L.lib.qr_op_create(arr, cbuf.ctypes.data_as(L.f64p), len(labels),
                                           L.QR_PHASE_ROWWISE, ctypes.byref(hh)))
            dt = time.perf_counter() - t0
            L.lib.qr_op_destroy(hh)
            return dt
        create(True)
        res["create_host_ms"] = 1e3 * min(create(False) for _ in range(3))
        res["create_device_ms"] = 1e3 * min(create(True) for _ in range(3))
        window = 16 << 30
        if 24 * nnz + 8 * (N + 1) <= 120 << 30:
            ip = torch.empty(N + 1, dtype=torch.int64, device="cuda")
            ix = torch.empty(nnz, dtype=torch.int64, device="cuda")
            dv = torch.empty(nnz, dtype=torch.complex128, device="cuda")
            ms = timed(lambda: L.check(L.lib.qr_csr_build(h.h, P(ip), P(ix), P(dv), sh)), 3)
            res["csr_build"] = "whole"
            del ip, ix, dv
        else:
            W = max(16, (window // (24 * G)) // 16 * 16)
            ix = torch.empty(W * G, dtype=torch.int64, device="cuda")
            dv = torch.empty(W * G, dtype=torch.complex128, device="cuda")

            def sweep():
                for r0 in range(0, N, W):
                    L.check(L.lib.qr_csr_build_rows(h.h, r0, min(N, r0 + W), P(ix), P(dv), sh))
            ms = timed(sweep, 2)
            res["csr_build"] = f"every row through a window of {W} rows ({24 * W * G / 2**30:.1f} GiB)"
            del ix, dv
        torch.cuda.empty_cache()
        res.update({"build_ms": ms, "build_nnz_per_s": nnz / (ms / 1e3),
                    "build_GBps": (24 * nnz + 8 * (N + 1)) / ms / 1e6})
        res["build_pct_hbm"] = 100 * res["build_GBps"] / HBM_PEAK_GBPS
        g = torch.Generator(device="cuda")
        g.manual_seed(23)
        x64 = torch.randn(N, dtype=torch.complex128, device="cuda", generator=g)
        x64 /= torch.linalg.vector_norm(x64)
        x32 = x64.to(torch.complex64)
        y64, y32 = torch.empty_like(x64), torch.empty_like(x32)
        e = torch.empty(2, dtype=torch.float64, device="cuda")
        for prec, xt, yt, key, sz in ((L.QR_PREC_MIXED, x32, y32, "mixed", 8),
                                      (L.QR_PREC_FP64, x64, y64, "fp64", 16)):
            ms_a = timed(lambda: L.check(L.lib.qr_pauli_apply(h.h, prec, 1, P(xt), P(yt), P(e), sh)), 3)
            res[f"apply_{key}_ms"] = ms_a
            res[f"apply_{key}_GBps"] = 2 * sz * N / ms_a / 1e6
        res["apply_mixed_rel_err_y"] = (torch.linalg.vector_norm(y32.to(torch.complex128) - y64) /
                                        torch.linalg.vector_norm(y64)).item()
        del x64, x32, y64, y32
        torch.cuda.empty_cache()
        # CPU port of RowwiseUnsafeChunked/1000 on the first rows
        p = orc.Params(labels, coeffs)
        rows = 1000
        t0 = time.perf_counter()
        orc.build_csr(p, 0, rows, step=1000, nthreads=nthr)
        t1 = time.perf_counter() - t0
        rows = int(min(N, max(1000, rows * 2.0 / max(t1, 1e-3)))) // 1000 * 1000 or 1000
        t0 = time.perf_counter()
        _, ind, _ = orc.build_csr(p, 0, rows, step=1000, nthreads=nthr)
        tc = time.perf_counter() - t0
        res["cpu_port_build_nnz_per_s"] = len(ind) / tc
        res["cpu_port_sample"] = f"rows 0..{rows} of 2^{nq}, {nthr} threads, one run"
        res["gpu_over_cpu_build"] = res["build_nnz_per_s"] / res["cpu_port_build_nnz_per_s"]
        del ind
        out[name] = res
        log(f"giant {name}: n={nq} T={h.T} G={G} build {ms:.2f} ms ({res['build_GBps']:.0f} GB/s, "
            f"{res['build_nnz_per_s']:.3e} nnz/s; CPU port {res['cpu_port_build_nnz_per_s']:.3e}), "
            f"apply mixed {res['apply_mixed_ms']:.3f} ms, fp64 {res['apply_fp64_ms']:.3f} ms; "
            f"tables host {res['create_host_ms']:.2f} ms, device {res['create_device_ms']:.2f} ms")
    return out


def bench_vec(args, torch, qa):
    """Eigensolver-step operations on the device: axpby and precond2 on
    2^27-element complex128 vectors (48 B per element: two reads, one write),
    and SpMat.diagonal of the 24-qubit Heisenberg CSR (2^24 rows, G = 25)."""
    from qrusty_amd import _lib as L
    from qrusty_amd import workloads

    n = 1 << 27
    g = torch.Generator(device="cuda")
    g.manual_seed(7)
    x = torch.randn(n, dtype=torch.complex128, device="cuda", generator=g)
    y = torch.randn(n, dtype=torch.complex128, device="cuda", generator=g)
    z = torch.empty_like(x)
    stream = torch.cuda.current_stream()
    sh = ctypes.c_void_p(stream.cuda_stream)
    P = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    a = (ctypes.c_double * 2)(0.3, -1.7)
    b = (ctypes.c_double * 2)(-2.5, 0.25)
    e = (ctypes.c_double * 2)(0.25, -0.5)

    def timed(fn, reps):
        fn()
        ev = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        torch.cuda.synchronize()
        ev[0].record(stream)
        for _ in range(reps):
            fn()
        ev[1].record(stream)
        torch.cuda.synchronize()
        return ev[0].elapsed_time(ev[1]) / reps

    reps = max(3, args.steps)
    t_axpby = timed(lambda: L.check(L.lib.qr_axpby(n, a, P(x), b, P(y), P(z), sh)), reps)
    t_pre = timed(lambda: L.check(L.lib.qr_precond2(n, P(x), P(y), e, 1e-14, P(z), sh)), reps)
    del x, y, z
    labels, coeffs = workloads.heisenberg_ring(24, seed=workloads.SEED_CFG3)
    sop = qa.SparsePauliOp([qa.Pauli(l) for l in labels], coeffs)
    m = sop.to_matrix_mode("Hip")
    ip, ix, dv = m.device_arrays()
    N = 1 << 24
    # the build of that CSR (24 B per entry written; its diagonal group has 48
    # terms, the other 24 groups 2)
    h = sop._handle(0)
    t_build = timed(lambda: L.check(L.lib.qr_csr_build(h.h, P(ip), P(ix), P(dv), sh)), reps)
    d = torch.empty(N, dtype=torch.complex128, device="cuda")
    t_diag = timed(lambda: L.check(L.lib.qr_csr_diagonal(N, N, dv.numel(), P(ip), P(ix), P(dv),
                                                         P(d), sh)), reps)
    # CSR matvec of the same matrix (one complex128 state): the "24-qubit
    # Heisenberg matvec" in CSR form, next to the matrix-free apply
    xs = torch.randn(N, dtype=torch.complex128, device="cuda", generator=g)
    ys = torch.empty_like(xs)
    t_mv = timed(lambda: L.check(L.lib.qr_csr_matvec(N, N, dv.numel(), P(ip), P(ix), P(dv), P(xs),
                                                     P(ys), sh)), reps)
    mv_bytes = 24 * dv.numel() + 8 * (N + 1) + 32 * N
    del xs, ys
    # H - e*I (a_spmat_p_b_spmat): count pass + indptr scan, then the fill pass
    eip = torch.arange(N + 1, dtype=torch.int64, device="cuda")
    eix = torch.arange(N, dtype=torch.int64, device="cuda")
    edv = torch.ones(N, dtype=torch.complex128, device="cuda")
    one = (ctypes.c_double * 2)(1.0, 0.0)
    ipo = torch.empty(N + 1, dtype=torch.int64, device="cuda")
    nnz = ctypes.c_uint64()
    common = (N, one, dv.numel(), P(ip), P(ix), P(dv), e, N, P(eip), P(eix), P(edv))
    L.check(L.lib.qr_csr_add_count(*common, P(ipo), ctypes.byref(nnz), sh))
    ixo = torch.empty(nnz.value, dtype=torch.int64, device="cuda")
    dvo = torch.empty(nnz.value, dtype=torch.complex128, device="cuda")
    t_cnt = timed(lambda: L.check(L.lib.qr_csr_add_count(*common, P(ipo), ctypes.byref(nnz), sh)),
                  reps)
    t_fill = timed(lambda: L.check(L.lib.qr_csr_add_fill(*common, P(ipo), P(ixo), P(dvo), sh)), reps)
    # algorithmic bytes: both inputs (indices + values) and indptrs read once,
    # the sum written once
    nin = dv.numel() + N
    sp_bytes = 24 * nin + 16 * (N + 1) + 24 * nnz.value + 8 * (N + 1)
    res = {"workload": "axpby / precond2 on 2^27 complex128; diagonal and H - e*I of the "
                       "24-qubit Heisenberg CSR",
           "axpby_ms": t_axpby, "axpby_GBps": 48 * n / t_axpby / 1e6,
           "precond2_ms": t_pre, "precond2_GBps": 48 * n / t_pre / 1e6,
           "diagonal_ms": t_diag, "diagonal_rows_per_s": N / (t_diag / 1e3),
           "heisenberg24_csr_build_ms": t_build,
           "heisenberg24_csr_build_GBps": (24 * dv.numel() + 8 * (N + 1)) / t_build / 1e6,
           "heisenberg24_csr_matvec_ms": t_mv, "heisenberg24_csr_matvec_GBps": mv_bytes / t_mv / 1e6,
           "heisenberg24_csr_matvec_frac": mv_bytes / t_mv / 1e6 / HBM_PEAK_GBPS,
           "spadd_count_ms": t_cnt, "spadd_fill_ms": t_fill, "spadd_nnz_in": nin,
           "spadd_nnz_out": nnz.value, "spadd_GBps": sp_bytes / (t_cnt + t_fill) / 1e6}
    log(f"vec: axpby {t_axpby:.3f} ms ({res['axpby_GBps']:.0f} GB/s), precond2 {t_pre:.3f} ms "
        f"({res['precond2_GBps']:.0f} GB/s), diagonal {t_diag:.3f} ms ({res['diagonal_rows_per_s']:.3e} rows/s), "
        f"H-eI count {t_cnt:.3f} + fill {t_fill:.3f} ms ({res['spadd_GBps']:.0f} GB/s algorithmic), "
        f"Heisenberg-24 CSR build {t_build:.3f} ms ({res['heisenberg24_csr_build_GBps']:.0f} GB/s), "
        f"Heisenberg-24 CSR matvec {t_mv:.3f} ms ({res['heisenberg24_csr_matvec_GBps']:.0f} GB/s, "
        f"{100 * res['heisenberg24_csr_matvec_frac']:.1f}% of HBM peak)")
    del m, ip, ix, dv, d, eip, eix, edv, ipo, ixo, dvo
    torch.cuda.empty_cache()
    return res


def bench_io(args, torch, qa):
    """CSR files of the 20-qubit Heisenberg ring CSR (2^20 rows, G = 21, 2.2e7
    entries) in the temporary directory: raw format write / read (24 B per
    entry + indptr) and MatrixMarket write / read (text), plain; raw with
    gzip.  Times include the device <-> host streaming; files are removed."""
    import tempfile
    from qrusty_amd import workloads
    labels, coeffs = workloads.heisenberg_ring(20, seed=workloads.SEED_CFG3)
    m = qa.SparsePauliOp([qa.Pauli(l) for l in labels], coeffs).to_matrix_mode("Hip")
    nnz = m.nnz()
    raw_bytes = 24 * nnz + 8 * ((1 << 20) + 1) + 2 + 6 * 8
    res = {"workload": "CSR files of the 20-qubit Heisenberg ring (2^20 rows, 2.2e7 entries)",
           "nnz": nnz}
    d = tempfile.mkdtemp()

    def clock(fn):
        torch.cuda.synchronize()
        t = time.perf_counter()
        out = fn()
        torch.cuda.synchronize()
        return time.perf_counter() - t, out

    try:
        for name, path in [("raw", os.path.join(d, "h.bin")), ("raw_gz", os.path.join(d, "h.bin.gz"))]:
            tw, _ = clock(lambda: m.raw_write(path))
            tr, back = clock(lambda: qa.SpMat.raw_read(path))
            assert all(torch.equal(a.view(torch.int64), b.view(torch.int64))
                       for a, b in zip(m.device_arrays(), back.device_arrays()))
            res[f"{name}_write_s"], res[f"{name}_read_s"] = tw, tr
            res[f"{name}_file_bytes"] = os.path.getsize(path)
            res[f"{name}_write_GBps"] = raw_bytes / tw / 1e9
            res[f"{name}_read_GBps"] = raw_bytes / tr / 1e9
            os.remove(path)
            del back
        path = os.path.join(d, "h.mtx")
        tw, _ = clock(lambda: m.matrixmarket_write(path))
        size = os.path.getsize(path)
        tr, back = clock(lambda: qa.SpMat.matrixmarket_read(path))
        assert all(torch.equal(a.view(torch.int64), b.view(torch.int64))
                   for a, b in zip(m.device_arrays(), back.device_arrays()))
        os.remove(path)
        res.update({"mm_write_s": tw, "mm_read_s": tr, "mm_file_bytes": size,
                    "mm_write_entries_per_s": nnz / tw, "mm_read_entries_per_s": nnz / tr,
                    "mm_write_MBps": size / tw / 1e6, "mm_read_MBps": size / tr / 1e6})
    finally:
        shutil.rmtree(d, ignore_errors=True)
    log(f"io: raw write {res['raw_write_GBps']:.2f} GB/s read {res['raw_read_GBps']:.2f} GB/s; "
        f"raw.gz write {res['raw_gz_write_GBps']:.2f} read {res['raw_gz_read_GBps']:.2f} GB/s; "
        f"mtx write {res['mm_write_MBps']:.0f} MB/s ({res['mm_write_entries_per_s']:.3e} entries/s) "
        f"read {res['mm_read_MBps']:.0f} MB/s")
    return res


def bench_copy(args, torch):
    """Plain device-to-device copy of 2 GiB (torch copy_): the calibration
    kernel whose known bytes scale the HBM counters FETCH_SIZE / WRITE_SIZE.
    Also the rates a write-only fill and a read-only reduction reach on 16 GiB,
    the practical ceilings for the CSR build (writes) and matvec (reads)."""
    def timed(f, steps):
        for _ in range(args.warmup):
            f()
        torch.cuda.synchronize()
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(steps):
            f()
        b.record()
        torch.cuda.synchronize()
        return a.elapsed_time(b) / steps

    n = 1 << 28  # float64 elements = 2 GiB
    src = torch.ones(n, dtype=torch.float64, device="cuda")
    dst = torch.empty_like(src)
    ms = timed(lambda: dst.copy_(src), args.steps)
    res = {"workload": "device copy 2 GiB", "bytes_read": 8 * n, "bytes_written": 8 * n,
           "ms": ms, "GBps": 16 * n / ms / 1e6}
    del src, dst
    big = torch.empty(1 << 31, dtype=torch.float64, device="cuda")  # 16 GiB
    ms_fill = timed(lambda: big.fill_(1.0), max(2, args.steps))
    ms_sum = timed(lambda: big.sum(), max(2, args.steps))
    res["fill_16GiB_GBps"] = 8 * big.numel() / ms_fill / 1e6
    res["read_sum_16GiB_GBps"] = 8 * big.numel() / ms_sum / 1e6
    del big
    torch.cuda.empty_cache()
    log(f"copy {ms:.3f} ms ({res['GBps']:.0f} GB/s); fill {res['fill_16GiB_GBps']:.0f} GB/s, "
        f"read (sum) {res['read_sum_16GiB_GBps']:.0f} GB/s")
    return res


def main():
    ap = argparse.ArgumentParser(description=__doc__, formatter_class=argparse.RawDescriptionHelpFormatter)
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=5)
    ap.add_argument("--warmup", type=int, default=2)
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline")
    ap.add_argument("--no-extra", action="store_true", help="skip the Heisenberg apply workload")
    ap.add_argument("--no-check", action="store_true", help="skip the sampled parity check")
    ap.add_argument("--only", choices=["csr", "apply", "apply-mixed", "apply-fp64", "batch", "large",
                                       "giant", "vec", "io", "copy"],
                    default=None, help="one section; io (files) runs only when named")
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py: runs on one GPU only; launches over several GPUs are not "
              "implemented (the path's sharding exists as a design, not as code).", file=sys.stderr)
        sys.exit(2)

    import torch
    import qrusty_amd as qa
    if not torch.cuda.is_available():
        print("bench.py needs a GPU", file=sys.stderr)
        sys.exit(1)
    torch.cuda.set_device(0)

    if args.only == "copy":
        print(json.dumps({"extra": {"copy": bench_copy(args, torch)}}), flush=True)
        return

    out = {"metric": "CSR nnz/s + Pauli-sum matvec GB/s (% HBM peak); FP64 vs mixed @<=1e-6 rel",
           "n_gpus": 1, "steps": args.steps, "warmup": args.warmup, "higher_is_better": True,
           "scaling": "weak", "vs_baseline": None, "dtype": "c128/u64", "data": "synthetic"}
    extra = {}
    if args.only in (None, "csr"):
        res, (labels, coeffs) = bench_csr(args, torch, qa)
        out.update({"value": res["value"], "unit": "nnz/s", "ms_per_step": res["ms_per_step"],
                    "config": {"workload": res["workload"], "num_qubits": 20, "num_terms": 2000,
                               "groups": res["G"], "nnz": res["nnz"], "seed": "0x51520002"},
                    "roofline": res.pop("roofline")})
        extra["csr"] = res
        if not args.no_cpu:
            log("cpu baseline ...")
            out["cpu_baseline"] = cpu_baseline_csr(labels, coeffs)
            log(f"cpu baseline {out['cpu_baseline']['value']:.3e} nnz/s")
    if args.only in ("apply-mixed", "apply-fp64"):
        a = bench_apply_one(args, torch, qa, args.only.split("-")[1])
        out.update({"value": a["GBps"], "unit": "GB/s", "ms_per_step": a["ms"],
                    "config": {"workload": a["workload"]}})
        extra[args.only] = a
    if args.only in (None, "apply") and not args.no_extra:
        extra["apply"] = bench_apply(args, torch, qa)
        if args.only == "apply":
            a = extra["apply"]
            out.update({"value": a["mixed_GBps"], "unit": "GB/s", "ms_per_step": a["mixed_ms"],
                        "dtype": "c64/fp64", "config": {"workload": a["workload"]}})
    if args.only in (None, "batch") and not args.no_extra:
        extra["batch"] = bench_batch(args, torch, qa)
    if args.only in (None, "large") and not args.no_extra:
        extra["large_apply"] = bench_large_apply(args, torch, qa)
    if args.only in (None, "giant") and not args.no_extra:
        extra["giant"] = bench_giant(args, torch, qa)
    if args.only in (None, "vec") and not args.no_extra:
        extra["vec"] = bench_vec(args, torch, qa)
    if args.only == "io":
        extra["io"] = bench_io(args, torch, qa)
    if args.only is None and not args.no_extra:
        # the rates this box sustains for plain streams, and the CSR kernels
        # as a fraction of them (next to the fraction of the 8 TB/s peak)
        cp = bench_copy(args, torch)
        extra["copy"] = cp
        if "csr" in extra:
            extra["csr"]["build_frac_of_fill"] = extra["csr"]["build_GBps"] / cp["fill_16GiB_GBps"]
            extra["csr"]["matvec_frac_of_read"] = extra["csr"]["matvec_GBps"] / cp["read_sum_16GiB_GBps"]
            extra["csr"]["matvec_frac_of_copy"] = extra["csr"]["matvec_GBps"] / cp["GBps"]
    out["extra"] = extra
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
