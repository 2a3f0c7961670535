"""GPU parity of the apply's launch shapes against the oracle: the thread
groups that share a tile (1, 2, 4), coefficient tables of many parts, and the
window passes of FP64 applies of 2^21 rows and more.

Bars: FP64 1e-12 (normwise, and componentwise against sum |c'||x|): every
coefficient, product and sum is FP64, at most a few thousand terms per row.
Mixed 1e-6: FP64 arithmetic on a state rounded to complex64 (6e-8) and one
rounding of y.
"""
import numpy as np
import pytest

from oracle import oracle as orc

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import qrusty_amd  # noqa: F401
    yield
    torch.cuda.synchronize()
    torch.cuda.empty_cache()


def _op(labels, coeffs):
    import qrusty_amd as qa
    return qa.SparsePauliOp([qa.Pauli(s) for s in labels], coeffs)


def _bound(p, x, rows):
    cabs = np.abs(p.cp.view(np.complex128))
    out = np.zeros((x.shape[0], len(rows)))
    for t in range(p.T):
        out += cabs[t] * np.abs(x[:, (rows ^ p.x[t]).astype(np.int64)])
    return out


def _check(p, op, x, rows, prec):
    ref = orc.apply_rows(p, x, rows)
    y, e = op.apply_and_expectation(x, prec)
    got = y[:, rows.astype(np.int64)]
    if prec == "fp64":
        assert np.linalg.norm(got - ref) <= 1e-12 * np.linalg.norm(ref)
        assert np.all(np.abs(got - ref) <= 1e-12 * _bound(p, x, rows) + 1e-300)
    else:
        assert np.linalg.norm(got - ref) <= 1e-6 * np.linalg.norm(ref)
    # <x|Hx> from the whole y that the same call returned
    eref = np.sum(x.conj() * y, axis=1)
    tol = 1e-12 if prec == "fp64" else 1e-6
    assert np.all(np.abs(e - eref) <= tol * np.linalg.norm(x, axis=1) * np.linalg.norm(y, axis=1))
    assert np.array_equal(op.expectation(x, prec), e)


def _mixed_terms(n, T, seed, z_only=0.3, real=False):
    rng = np.random.default_rng(seed)
    labels = ["".join(rng.choice(list("IZ" if rng.random() < z_only else "IXYZ"), size=n)) for _ in range(T)]
    coeffs = rng.standard_normal(T) + (0 if real else 1j * rng.standard_normal(T))
    return labels, list(coeffs)


@pytest.mark.parametrize("split", ["1", "2", "4"])
@pytest.mark.parametrize("form", ["1", "2"])
@pytest.mark.parametrize("n", [1, 7, 9, 10, 11, 13])
def test_thread_groups(monkeypatch, n, form, split):
    from qrusty_amd import workloads
    monkeypatch.setenv("QR_APPLY_SPLIT", split)
    monkeypatch.setenv("QR_APPLY_FORM", form)
    labels, coeffs = _mixed_terms(n, 1 + 23 * n, 300 + n)
    p, op = orc.Params(labels, coeffs), _op(labels, coeffs)
    x = workloads.random_states(p.N, 3, 400 + n)
    rows = np.arange(p.N, dtype=np.uint64)
    print(f"[gpu] apply thread groups n={n} form={form} split={split}", flush=True)
    _check(p, op, x, rows, "fp64")
    for small in ("0", "1"):
        monkeypatch.setenv("QR_APPLY_SMALL", small)
        _check(p, op, x, rows, "mixed")


@pytest.mark.parametrize("real", [True, False])
@pytest.mark.parametrize("T", [40, 700, 4000])
def test_tables_of_many_parts(monkeypatch, T, real):
    """Groups whose patterns span more dimensions than one table holds: a
    diagonal of up to 4000 Z strings on 13 qubits (every pattern of the tile,
    chunks of their own, a group split at its pattern limit) beside one-term
    groups."""
    from qrusty_amd import workloads
    labels, coeffs = _mixed_terms(13, T, 500 + T, z_only=0.9, real=real)
    p, op = orc.Params(labels, coeffs), _op(labels, coeffs)
    x = workloads.random_states(p.N, 1, 600 + T)
    rows = np.arange(p.N, dtype=np.uint64)
    for form in ("1", "2"):
        monkeypatch.setenv("QR_APPLY_FORM", form)
        print(f"[gpu] apply tables T={T} real={real} form={form}", flush=True)
        _check(p, op, x, rows, "fp64")
        _check(p, op, x, rows, "mixed")


def _ring(n, rng, kind):
    """Nearest-neighbour operators: the Heisenberg ring; the same with XY and
    YX terms (complex coefficients) on an open chain; single X on every site
    with ZZ couplings."""
    labels, coeffs = [], []

    def term(ops, c):
        chars = ["I"] * n
        for q, ch in ops.items():
            chars[n - 1 - q] = ch
        labels.append("".join(chars))
        coeffs.append(c)

    for i in range(n if kind == "ring" else n - 1):
        j = (i + 1) % n
        for a, b in (("X", "X"), ("Y", "Y"), ("Z", "Z")) if kind != "field" else (("Z", "Z"),):
            term({i: a, j: b}, complex(rng.uniform(-1, 1)))
        if kind == "chain":
            term({i: "X", j: "Y"}, complex(rng.uniform(-1, 1)))
            term({i: "Y", j: "X"}, complex(0, rng.uniform(-1, 1)))
    for i in range(n):
        term({i: "X" if kind == "field" else "Z"}, complex(rng.uniform(-1, 1)))
    return labels, coeffs


@pytest.mark.parametrize("kind,n,nvec", [("ring", 21, 5), ("ring", 22, 1), ("chain", 22, 1), ("field", 23, 1)])
def test_window_passes(kind, n, nvec):
    """States of 2^25 bytes and more, whose high neighbour masks run in window
    passes (several at 23 qubits; several launches of states at 5 of 21
    qubits)."""
    from qrusty_amd import workloads
    rng = np.random.default_rng(n)
    labels, coeffs = _ring(n, rng, kind)
    p, op = orc.Params(labels, coeffs), _op(labels, coeffs)
    x = workloads.random_states(p.N, nvec, 700 + n)
    rows = np.unique(np.r_[0, p.N - 1, rng.choice(p.N, size=4096)]).astype(np.uint64)
    print(f"[gpu] apply window passes {kind} n={n} nvec={nvec}", flush=True)
    _check(p, op, x, rows, "fp64")


@pytest.mark.parametrize("n,kind,nvec", [(21, "x", 3), (22, "x", 1), (23, "bonds", 2), (24, "x", 1)])
def test_windows_take_every_group(n, kind, nvec):
    """Operators of high masks alone, without a diagonal: X on the top qubits,
    XX + YY bonds of qubits 17 and up.  Window passes hold all their groups, and
    the first of them writes y."""
    from qrusty_amd import workloads

    def term(ops):
        return "".join(ops.get(n - 1 - k, "I") for k in range(n))

    if kind == "bonds":
        labels = [term({q: p, q + 1: p}) for q in range(17, n - 1) for p in "XY"]
    else:
        labels = [term({q: "X"}) for q in range(17, n)]
    rng = np.random.default_rng(n)
    coeffs = list(rng.uniform(-1, 1, len(labels)).astype(complex))
    p, op = orc.Params(labels, coeffs), _op(labels, coeffs)
    x = workloads.random_states(p.N, nvec, 800 + n)
    rows = np.unique(np.r_[0, p.N - 1, rng.choice(p.N, size=4096)]).astype(np.uint64)
    print(f"[gpu] apply windows only {kind} n={n} nvec={nvec}", flush=True)
    _check(p, op, x, rows, "fp64")


def test_complex64_sum_is_rounded_once():
    """26 qubits, complex64: groups inside a tile and groups of high masks whose
    sums cancel to 1e-6 of either.  On a constant state y is the sum of the
    coefficients times it; one rounding of each part (2^-24) and FP64 before."""
    import qrusty_amd as qa
    from qrusty_amd import workloads
    n = 26
    qubits = [0, 1, 2, 3] + list(range(19, n))
    coeffs = [1 / 12] * 4 + [-1 / 21 + 1e-6 / 7] * 7
    op = qa.SparsePauliOp([qa.Pauli(workloads._label(n, {q: "X"})) for q in qubits], [complex(c) for c in coeffs])
    v = complex(np.float32(0.1), np.float32(0.3))
    print("[gpu] complex64 cancelling sum", flush=True)
    x = torch.full((1, 1 << n), v, dtype=torch.complex64, device="cuda")
    y = op.apply(x, "mixed")
    ref = sum(coeffs) * v
    err = (torch.view_as_real(y).double() - torch.tensor([ref.real, ref.imag], device="cuda")).abs().amax().item()
    assert err <= 1.01 * 2.0**-24 * abs(ref)


@pytest.mark.parametrize("n,terms,nvec,prec", [(20, 70, 2, "fp64"), (22, 70, 1, "fp64"), (20, 40, 1, "fp64"),
                                               (16, 3, 4, "fp64"), (14, 15, 1, "fp64"), (22, 70, 2, "mixed"),
                                               (23, 70, 1, "mixed")])
def test_scattered_partners(n, terms, nvec, prec):
    """Random operators, whose groups have partners of their own far from the
    tile: on both sides of the rule's numbers of partners and rows."""
    from qrusty_amd import workloads
    rng = np.random.default_rng(n + terms)
    labels = ["X" + "".join(rng.choice(list("IXYZ"), size=n - 1)) for _ in range(terms)]
    coeffs = list(rng.standard_normal(terms) + 1j * rng.standard_normal(terms))
    p, op = orc.Params(labels, coeffs), _op(labels, coeffs)
    x = workloads.random_states(p.N, nvec, 900 + n)
    rows = np.unique(np.r_[0, p.N - 1, rng.choice(p.N, size=4096)]).astype(np.uint64)
    print(f"[gpu] apply scattered n={n} terms={terms} nvec={nvec} {prec}", flush=True)
    _check(p, op, x, rows, prec)
