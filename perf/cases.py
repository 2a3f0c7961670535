"""Workloads of the Pauli-operator framework, each through its public entry points.

A case is one call sequence of a user's program on one operator:

    build         op.to_matrix_mode(): the rowwise CSR matrix
    build_matvec  the CSR and one y = A x with it
    matvec        y = A x with a CSR that the program holds
    apply         y = H x without a matrix; in FP64 with <x|H|x> from the same pass
    expectation   <x|H|x> without a matrix (one state, as in a variational loop)
    davidson      the steps around the matvec of a Davidson iteration: the residual
                  A v - e v, its diagonal preconditioning, and the shifted matrix A - e I
    batch         several uneven operators built and applied in one launch

and the operator is of one of four families:

    random        labels uniform over {I, X, Y, Z}: every group of terms that share an
                  x mask is one term or a few; complex coefficients
    heisenberg    a nearest-neighbour spin ring with fields; real coefficients
    klocal        random terms of weight 1 to 4; real coefficients
    molecule      the Jordan-Wigner form of an electronic-structure Hamiltonian (one- and
                  two-body integrals, spin-blocked orbitals): hundreds of terms in the
                  diagonal and the hopping groups, 4 or 6 in the others

The labels come from the case (a list of terms is what a program is written for), the
coefficients and the states from the seed.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import qrusty_amd as qa
from qrusty_amd import workloads as wl

MODE = "RowwiseUnsafeChunked/1000"
TOL = 1e-3
# most matrix entries of a drawn case, and most products (rows x groups x states)
MOST_NNZ = 2.0e9
MOST_PRODUCTS = 5.0e11


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the smallest everyday call: a 12-qubit operator of 200 terms, matrix and product
        {"name": "build_matvec_random_12q", "what": "build_matvec", "family": "random", "qubits": 12,
         "terms": 200, "labels": 0x51520001},
        # one energy of a variational loop on a small molecule
        {"name": "expectation_molecule_12q", "what": "expectation", "family": "molecule", "qubits": 12,
         "precision": "fp64", "states": 1},
        # the matrix of 2000 random terms on 20 qubits
        {"name": "build_random_20q", "what": "build", "family": "random", "qubits": 20, "terms": 2000,
         "labels": 0x51520002},
        # the matrix of a 10-orbital molecule (20 qubits, 14251 terms)
        {"name": "build_molecule_20q", "what": "build", "family": "molecule", "qubits": 20},
        # the product with long rows (about 2000 entries each), as in an eigensolver's loop
        {"name": "matvec_random_20q", "what": "matvec", "family": "random", "qubits": 20, "terms": 2000,
         "labels": 0x51520002},
        # and with short rows (25 entries each)
        {"name": "matvec_heisenberg_24q", "what": "matvec", "family": "heisenberg", "qubits": 24},
        # a block of states through a spin ring, without a matrix, in both precisions
        {"name": "apply_fp64_heisenberg_24q_8", "what": "apply", "family": "heisenberg", "qubits": 24,
         "precision": "fp64", "states": 8},
        {"name": "apply_mixed_heisenberg_24q_8", "what": "apply", "family": "heisenberg", "qubits": 24,
         "precision": "mixed", "states": 8},
        # the largest state: 28 qubits, 10000 k-local terms
        {"name": "apply_mixed_klocal_28q", "what": "apply", "family": "klocal", "qubits": 28, "terms": 10000,
         "labels": 0x51520005, "precision": "mixed", "states": 1},
        # one state through the 10-orbital molecule, without a matrix
        {"name": "apply_fp64_molecule_20q", "what": "apply", "family": "molecule", "qubits": 20,
         "precision": "fp64", "states": 1},
        # a Davidson iteration's other steps on a 23-site ring
        {"name": "davidson_heisenberg_23q", "what": "davidson", "family": "heisenberg", "qubits": 23},
        # uneven operators (8 to 18 qubits, 10 to 5000 terms) in one launch
        {"name": "batch_random_16", "what": "batch", "family": "random", "operators": 16, "qmin": 8, "qmax": 18,
         "tmin": 10, "tmax": 5000, "labels": 5},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case: what is called, the family, and sizes over the whole range."""
    while True:
        what = rng.choice(["build", "build_matvec", "matvec", "matvec", "apply", "apply", "apply", "expectation",
                           "davidson", "batch"])
        if what == "batch":
            qmin = rng.randint(6, 12)
            c = {"what": what, "family": "random", "operators": rng.randint(2, 16), "qmin": qmin,
                 "qmax": rng.randint(qmin + 1, 18), "tmin": rng.randint(1, 40), "tmax": rng.randint(100, 5000),
                 "labels": rng.randrange(1, 1 << 20)}
            if work(c)["bytes"] > 48 * MOST_NNZ / 2:
                continue
            return c
        if what == "davidson":
            family = rng.choice(["heisenberg", "heisenberg", "molecule"])
        else:
            family = rng.choice(["random", "heisenberg", "klocal", "molecule"])
        c = {"what": what, "family": family, "qubits": rng.randint(8, 26)}
        if family == "molecule":
            c["qubits"] -= c["qubits"] % 2
        if family in ("random", "klocal"):
            c["terms"] = _log_int(rng, 10, 10000)
            c["labels"] = rng.randrange(1, 1 << 20)
        if what in ("apply", "expectation"):
            c["precision"] = "fp64" if what == "expectation" else rng.choice(["fp64", "mixed"])
            c["states"] = 1 if what == "expectation" else rng.randint(1, 8)
        groups = _group_bound(c)
        rows = 1 << c["qubits"]
        nnz = rows * groups
        if what in ("apply", "expectation"):
            # FP64 arithmetic and complex coefficients take about twice the time each
            cost = nnz * c["states"] * (2 if c["precision"] == "fp64" else 1) * (2 if family == "random" else 1)
            if cost > MOST_PRODUCTS or rows * c["states"] > 1 << 28:
                continue
        elif nnz > (MOST_NNZ / 4 if what == "davidson" else MOST_NNZ):
            continue
        return c


def _group_bound(case):
    """About how many distinct x masks (entries per row) the operator has."""
    n = case["qubits"]
    if case["family"] == "heisenberg":
        return n + 1
    if case["family"] == "molecule":
        m = n // 2
        pairs = m * (m - 1) // 2
        return 1 + 2 * pairs + 2 * math.comb(m, 4) + pairs * pairs
    t = case["terms"]
    if case["family"] == "klocal":
        return min(t, 1 + n + math.comb(n, 2) + math.comb(n, 3) + math.comb(n, 4))
    return min(t, 1 << n)


# ---------------------------------------------------------------------------
# operators
# ---------------------------------------------------------------------------
def _molecule(n, rng):
    """Terms of a molecular Hamiltonian on n = 2m spin-blocked orbitals: m alpha (qubits
    0..m-1), m beta, real integrals with magnitudes over several decades."""
    m = n // 2

    def value():
        return float(rng.choice([-1.0, 1.0]) * 10.0 ** rng.uniform(-6.0, -0.5))

    def label(ops, strings):
        chars = ["I"] * n
        for a, b in strings:  # the Z string strictly between two orbitals
            for q in range(a + 1, b):
                chars[n - 1 - q] = "Z"
        for q, c in ops:
            chars[n - 1 - q] = c
        return "".join(chars)

    labels, coeffs = [label([], [])], [-10.0 + value()]
    for p in range(n):
        labels.append(label([(p, "Z")], []))
        coeffs.append(value())
    for p in range(n):
        for q in range(p + 1, n):
            labels.append(label([(p, "Z"), (q, "Z")], []))
            coeffs.append(value())
    for s in (0, m):
        for p in range(s, s + m):
            for q in range(p + 1, s + m):
                # hopping p <-> q, alone and with the density of every other orbital (on an
                # orbital inside the string the two Z cancel)
                for r in [None] + [r for r in range(n) if r not in (p, q)]:
                    c = value()
                    for pair in "YX":
                        chars = list(label([(p, pair), (q, pair)], [(p, q)]))
                        if r is not None:
                            chars[n - 1 - r] = "I" if chars[n - 1 - r] == "Z" else "Z"
                        labels.append("".join(chars))
                        coeffs.append(c)
        # two electrons of one spin: four orbitals, six terms
        for p in range(s, s + m):
            for q in range(p + 1, s + m):
                for r in range(q + 1, s + m):
                    for t in range(r + 1, s + m):
                        a, b = value(), value()
                        for f, c in (("YXXY", a), ("YYYY", a + b), ("XXYY", b), ("YYXX", b), ("XXXX", a + b),
                                     ("XYYX", a)):
                            labels.append(label(list(zip((p, q, r, t), f)), [(p, q), (r, t)]))
                            coeffs.append(c)
    # one of each spin: four orbitals, four terms
    for p in range(m):
        for q in range(p + 1, m):
            for r in range(m, n):
                for t in range(r + 1, n):
                    c = value()
                    for f in ("YYYY", "XXYY", "YYXX", "XXXX"):
                        labels.append(label(list(zip((p, q, r, t), f)), [(p, q), (r, t)]))
                        coeffs.append(c)
    return labels, [complex(c, 0.0) for c in coeffs]


def _operator(case, seed):
    """(labels, coefficients) of the case's operator."""
    rng = np.random.default_rng([seed, case["qubits"]])
    n = case["qubits"]
    if case["family"] == "molecule":
        return _molecule(n, rng)
    if case["family"] == "heisenberg":
        labels = wl.heisenberg_ring(n, 1)[0]
        return labels, [complex(c, 0.0) for c in rng.uniform(-1.0, 1.0, len(labels))]
    if case["family"] == "klocal":
        labels = wl.k_local_op(n, case["terms"], case["labels"])[0]
        return labels, [complex(c, 0.0) for c in rng.standard_normal(len(labels))]
    labels = wl.random_op(n, case["terms"], case["labels"])[0]
    c = rng.standard_normal(len(labels)) + 1j * rng.standard_normal(len(labels))
    return labels, [complex(v) for v in c]


def _batch_operators(case, seed):
    ops = []
    rng = np.random.default_rng([seed, case["operators"]])
    for labels, _ in wl.uneven_batch(case["operators"], case["labels"], case["qmin"], case["qmax"], case["tmin"],
                                     case["tmax"]):
        c = rng.standard_normal(len(labels)) + 1j * rng.standard_normal(len(labels))
        ops.append((labels, [complex(v) for v in c]))
    return ops


def _op(labels, coeffs):
    return qa.SparsePauliOp([qa.Pauli(s) for s in labels], coeffs)


def _states(dim, count, seed, dtype=torch.complex128):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 7919 + 17)
    x = torch.empty((count, dim), dtype=dtype, device="cuda")
    part = torch.float32 if dtype == torch.complex64 else torch.float64
    for k in range(count):
        v = torch.randn((dim, 2), generator=g, dtype=part, device="cuda")
        x[k] = torch.view_as_complex(v / torch.linalg.vector_norm(v))
        del v
    return x[0] if count == 1 else x


# ---------------------------------------------------------------------------
# what is measured
# ---------------------------------------------------------------------------
def prepare(case, seed):
    what = case["what"]
    if what == "batch":
        ops = [_op(labels, coeffs) for labels, coeffs in _batch_operators(case, seed)]
        batch = qa.Batch(ops)
        batch.set_states([_states(1 << op.num_qubits(), 1, seed + k) for k, op in enumerate(ops)])
        return {"what": what, "batch": batch}
    labels, coeffs = _operator(case, seed)
    op = _op(labels, coeffs)
    n = 1 << case["qubits"]
    state = {"what": what, "op": op}
    if what in ("apply", "expectation"):
        dtype = torch.complex64 if case["precision"] == "mixed" else torch.complex128
        state["x"] = _states(n, case["states"], seed, dtype)
        state["precision"] = case["precision"]
        return state
    if what == "build":
        return state
    state["x"] = _states(n, 1, seed)
    if what == "build_matvec":
        return state
    state["m"] = op.to_matrix_mode(MODE)
    if what == "davidson":
        state["e"] = _energy(seed)
        state["Av"] = qa.spmat_dot_densevec(state["m"], state["x"])
        rows = torch.arange(n + 1, dtype=torch.int64, device="cuda")
        ones = torch.ones(n, dtype=torch.complex128, device="cuda")
        state["I"] = qa.SpMat.new_unchecked((n, n), ones, rows[:n].clone(), rows)
    return state


def _energy(seed):
    """An approximate eigenvalue."""
    return -float(np.random.default_rng([seed, 3]).uniform(3.0, 12.0))


def _arrays(m):
    indptr, indices, data = m.device_arrays()
    return {"indptr": indptr, "indices": indices, "data": data}


def run(state):
    what = state["what"]
    if what == "build":
        return _arrays(state["op"].to_matrix_mode(MODE))
    if what == "build_matvec":
        m = state["op"].to_matrix_mode(MODE)
        y = qa.spmat_dot_densevec(m, state["x"])
        return {"m": _arrays(m), "y": y}
    if what == "matvec":
        return {"y": qa.spmat_dot_densevec(state["m"], state["x"])}
    if what == "apply":
        if state["precision"] == "mixed":
            return {"y": state["op"].apply(state["x"], "mixed")}
        y, e = state["op"].apply_and_expectation(state["x"], "fp64")
        return {"y": y, "e": e}
    if what == "expectation":
        return {"e": state["op"].expectation(state["x"], state["precision"])}
    if what == "davidson":
        r = qa.axpby(1.0, state["Av"], -state["e"], state["x"])
        d = qa.precond(state["m"], r, state["e"], TOL)
        s = qa.a_spmat_p_b_spmat(1.0, state["m"], -state["e"], state["I"])
        return {"r": r, "d": d, "s": _arrays(s)}
    batch = state["batch"]
    batch.run()
    return [[batch.csr(k)[0], batch.csr(k)[1], batch.csr(k)[2], batch.y[k]] for k in range(len(batch))]


def _masks(labels):
    """x and z masks and the number of Y of each label."""
    a = np.array([list(s) for s in labels])[:, ::-1]
    bit = np.uint64(1) << np.arange(a.shape[1], dtype=np.uint64)
    ax, ay, az = a == "X", a == "Y", a == "Z"
    x = ((ax | ay) * bit).sum(axis=1, dtype=np.uint64).astype(np.int64)
    z = ((az | ay) * bit).sum(axis=1, dtype=np.uint64).astype(np.int64)
    return x, z, ay.sum(axis=1)


def work(case):
    """Bytes: each input read once, each output written once.  Flops: a complex addition per
    row and term of a build; a complex product and sum per matrix entry of a matvec; per row
    and group of an apply a sum with a real, imaginary or complex factor."""
    if case["what"] == "batch":
        b = f = 0
        for labels, _ in _batch_operators(case, 1):
            rows, nnz = 1 << len(labels[0]), len(np.unique(_masks(labels)[0])) << len(labels[0])
            b += 2 * 24 * nnz + 8 * (rows + 1) + 32 * rows
            f += 2 * len(labels) * rows + 8 * nnz
        return {"bytes": b, "flops": f}
    labels, _ = _operator(case, 1)
    rows, groups = 1 << case["qubits"], len(np.unique(_masks(labels)[0]))
    nnz = rows * groups
    csr = 24 * nnz + 8 * (rows + 1)
    build = {"bytes": csr, "flops": 2 * len(labels) * rows}
    matvec = {"bytes": csr + 32 * rows, "flops": 8 * nnz}
    if case["what"] == "build":
        return build
    if case["what"] == "matvec":
        return matvec
    if case["what"] == "build_matvec":
        return {k: build[k] + matvec[k] for k in build}
    if case["what"] == "davidson":
        # r: two vectors in, one out; d: r and the matrix's diagonal in, one out; s: the
        # matrix and the identity in, the sum out
        return {"bytes": 48 * rows + 48 * rows + 2 * csr + 32 * rows, "flops": 20 * rows + 8 * nnz}
    size = 8 if case["precision"] == "mixed" else 16
    out = 0 if case["what"] == "expectation" else size
    flops = nnz * case["states"] * (8 if case["family"] == "random" else 4)
    return {"bytes": rows * case["states"] * (size + out), "flops": flops}


# ---------------------------------------------------------------------------
# the same results in 64 bits, in plain torch
# ---------------------------------------------------------------------------
def _grouped(labels, coeffs):
    """[(x mask, z masks, coefficients)] by ascending x mask: entry (r, r ^ x) of the operator
    is the sum of (-1)^popcount(r & z) (-i)^#Y c."""
    x, z, ys = _masks(labels)
    c = np.asarray(coeffs) * np.array([1, -1j, -1, 1j])[ys % 4]
    order = np.argsort(x, kind="stable")
    x, z, c = x[order], z[order], c[order]
    heads = np.flatnonzero(np.r_[True, x[1:] != x[:-1]])
    ends = np.r_[heads[1:], len(x)]
    return [(int(x[a]), z[a:b], c[a:b]) for a, b in zip(heads, ends)]


def _signs(width, z):
    """(-1)^popcount(r & z) for r < 2^width: a (2^width, len(z)) matrix."""
    r = torch.arange(1 << width, device="cuda")[:, None] & torch.as_tensor(z, device="cuda")[None, :]
    for s in (16, 8, 4, 2, 1):
        r = r ^ (r >> s)
    return (1 - 2 * (r & 1)).to(torch.float64)


def _apply_exact(groups, n, x):
    """sum over the groups of D(r) x[r ^ mask], r split into high and low halves."""
    lo = n // 2
    hi = n - lo
    single = x.dim() == 1
    xs = x.to(torch.complex128).reshape(-1, 1 << hi, 1 << lo)
    y = torch.zeros_like(xs)
    rh, rl = torch.arange(1 << hi, device="cuda"), torch.arange(1 << lo, device="cuda")
    for mask, z, c in groups:
        a = _signs(hi, z >> lo).to(torch.complex128) * torch.as_tensor(c, device="cuda")
        d = a @ _signs(lo, z & ((1 << lo) - 1)).to(torch.complex128).t().contiguous()
        rows, cols = rh ^ (mask >> lo), rl ^ (mask & ((1 << lo) - 1))
        for k in range(xs.shape[0]):
            y[k].addcmul_(d, xs[k][rows][:, cols])
    return y.reshape(-1) if single else y.reshape(y.shape[0], -1)


def _data_exact(groups, n):
    """Values of the CSR, columns ascending in each row, summed in term order."""
    lo = min(n, 10)
    G = len(groups)
    masks = torch.as_tensor([g[0] for g in groups], device="cuda")
    most = max(len(g[1]) for g in groups)
    # position k of every group that has that many terms
    steps = []
    for k in range(most):
        has = [g for g in range(G) if len(groups[g][1]) > k]
        z = np.array([groups[g][1][k] for g in has])
        c = torch.as_tensor(np.array([groups[g][2][k] for g in has]), device="cuda")
        steps.append((slice(None) if len(has) == G else torch.as_tensor(has, device="cuda"),
                      _signs(lo, z & ((1 << lo) - 1)), _signs(n - lo, z >> lo), c))
    out = torch.empty((1 << n, G), dtype=torch.complex128, device="cuda")
    part = max(1, min(1 << (n - lo), (1 << 25) // (G << lo) or 1))
    low = torch.arange(1 << lo, device="cuda")
    for h0 in range(0, 1 << (n - lo), part):
        h1 = min(h0 + part, 1 << (n - lo))
        v = torch.zeros((h1 - h0, 1 << lo, G), dtype=torch.complex128, device="cuda")
        for has, sl, sh, c in steps:
            v[:, :, has] += sl[None] * (sh[h0:h1] * c)[:, None, :]
        r = ((torch.arange(h0, h1, device="cuda") << lo)[:, None] | low[None, :])[:, :, None]
        order = torch.argsort(r ^ masks, dim=2)
        out[h0 << lo:h1 << lo] = torch.gather(v, 2, order).reshape(-1, G)
    return out.reshape(-1)


def exact(case, seed):
    what = case["what"]
    if what == "batch":
        out = []
        for k, (labels, coeffs) in enumerate(_batch_operators(case, seed)):
            groups, n = _grouped(labels, coeffs), len(labels[0])
            out.append([None, None, _data_exact(groups, n), _apply_exact(groups, n, _states(1 << n, 1, seed + k))])
        return out
    n = case["qubits"]
    groups = _grouped(*_operator(case, seed))
    if what == "build":
        return {"indptr": None, "indices": None, "data": _data_exact(groups, n)}
    if what in ("apply", "expectation"):
        # about 20 passes over the states per group: too long for the largest
        if (len(groups) * case["states"]) << n > 1.5e11:
            return None
        x = _states(1 << n, case["states"], seed,
                    torch.complex64 if case["precision"] == "mixed" else torch.complex128)
        y = _apply_exact(groups, n, x)
        if case["precision"] == "mixed":
            return {"y": y}
        e = (x.conj() * y).sum(dim=-1).cpu().numpy()
        return {"e": e} if what == "expectation" else {"y": y, "e": e}
    x = _states(1 << n, 1, seed)
    y = _apply_exact(groups, n, x)
    if what == "matvec":
        return {"y": y}
    if what == "build_matvec":
        return {"m": {"indptr": None, "indices": None, "data": _data_exact(groups, n)}, "y": y}
    e = _energy(seed)
    r = y - e * x
    G = len(groups)
    data = _data_exact(groups, n).reshape(-1, G)
    rows = torch.arange(1 << n, device="cuda")[:, None]
    masks = torch.as_tensor([g[0] for g in groups], device="cuda")
    # the diagonal's place in row r: as many masks as give a column below r
    at = torch.cat([((rows[k:k + (1 << 20)] ^ masks) < rows[k:k + (1 << 20)]).sum(dim=1, keepdim=True)
                    for k in range(0, 1 << n, 1 << 20)])
    diag = torch.gather(data, 1, at).reshape(-1)
    reg = diag - e
    reg = torch.where(reg.abs() < TOL, torch.full_like(reg, TOL), reg)
    s = None
    if case["family"] == "heisenberg":  # no entry cancels, so none is dropped
        data.scatter_add_(1, at, torch.full_like(at, 1, dtype=torch.complex128) * -e)
        s = data.reshape(-1)
    return {"r": r, "d": r / reg, "s": {"indptr": None, "indices": None, "data": s}}
