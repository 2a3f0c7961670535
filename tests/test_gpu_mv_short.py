"""CSR matvec of rows of 8 to 64 entries in the mean (k_csr_matvec_short): each
load count per lane, rows that do not fit beside rows that do, row counts around
a wave's eight, columns past the state (skipped), an indptr that descends.
Against numpy within (2 len + 8) eps sum |a||x| per row."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import qrusty_amd  # noqa: F401
    yield
    torch.cuda.synchronize()


@pytest.mark.parametrize("rows,lens", [(1, [16]), (7, [16]), (9, [17]), (64, [24]), (257, [25]), (1000, [32]), (33, [31]),
                                       (513, [0, 40]), (100, [1, 1, 1, 1, 1, 1, 1, 200]), (4000, [5, 20, 33, 16]), (65, [33]), (130, [48]), (70, [49]), (300, [64]), (77, [63, 30, 90]), (41, [8]), (90, [9]), (200, [12, 0, 30])])
@pytest.mark.parametrize("kind", ["valid", "past", "descends"])
def test_short(rows, lens, kind):
    import qrusty_amd as qa
    rng = np.random.default_rng(rows + len(lens))
    cols = 300
    lens = np.resize(lens, rows)
    indptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    ind = np.concatenate([np.sort(rng.choice(cols, size=int(n), replace=False)) for n in lens]).astype(np.uint64)
    data = rng.standard_normal(len(ind)) + 1j * rng.standard_normal(len(ind))
    if kind == "past":
        ind[::7] += np.uint64(10**6)
    if kind == "descends" and rows > 3:
        indptr[rows // 2] = indptr[rows // 2 - 1] // np.uint64(2)
    x = rng.standard_normal(cols) + 1j * rng.standard_normal(cols)
    m = qa.SpMat.new_unchecked((rows, cols), data, ind, indptr)
    print(f"[gpu] short rows={rows} {kind}", flush=True)
    y = qa.spmat_dot_densevec(m, torch.from_numpy(x).cuda()).cpu().numpy()
    for r in range(rows):
        k0, k1 = int(indptr[r]), max(int(indptr[r]), int(indptr[r + 1]))
        c, a = ind[k0:k1], data[k0:k1]
        c, a = c[c < cols].astype(np.int64), a[c < cols]
        bound = (2 * len(c) + 8) * 2.3e-16 * np.sum(np.abs(a) * np.abs(x[c]))
        assert abs(y[r] - np.sum(a * x[c])) <= bound + 1e-300


@pytest.mark.parametrize("n,terms", [(19, 70), (19, 110), (18, 129)])
def test_long_rows_of_large_matrices(n, terms):
    """65 to 128 entries per row from 2^25 entries on (and past both limits):
    the product against the oracle on sampled rows, within 1e-12 of
    sum |c'||x|."""
    import qrusty_amd as qa
    from oracle import oracle as orc
    from qrusty_amd import workloads
    labels, coeffs = workloads.random_op(n, terms, seed=0x6100 + terms)
    p = orc.Params(labels, coeffs)
    op = qa.SparsePauliOp([qa.Pauli(l) for l in labels], coeffs)
    m = op.to_matrix_mode("RowwiseUnsafeChunked/100")
    x = workloads.random_states(p.N, 1, 17)[0]
    print(f"[gpu] matvec n={n} terms={terms}", flush=True)
    y = qa.spmat_dot_densevec(m, torch.from_numpy(x).cuda()).cpu().numpy()
    rows = np.unique(np.concatenate([[0, p.N - 1], np.random.default_rng(3).integers(0, p.N, 200)])).astype(np.uint64)
    ref = orc.apply_rows(p, x, rows)[0]
    bound = sum(abs(c) * np.abs(x[(rows ^ xm).astype(np.int64)]) for c, xm in zip(p.cp.view(np.complex128), p.x))
    assert np.all(np.abs(y[rows.astype(np.int64)] - ref) <= 1e-12 * bound)


@pytest.mark.parametrize("n,mean,dense", [(21, 8.0, 40), (20, 12.0, 600), (19, 25.0, 200), (18, 60.0, 90)])
def test_uneven_rows_of_large_matrices(n, mean, dense):
    """Matrices past 256 MB whose rows vary about their mean, one in 100 with
    `dense` entries: waves that fit beside waves that do not.  Against numpy
    within (2 len + 8) eps sum |a||x| per row."""
    import qrusty_amd as qa
    rng = np.random.default_rng(n)
    rows = 1 << n
    lens = np.where(rng.random(rows) < 0.01, dense, rng.poisson(mean, rows)).astype(np.int64)
    lens[-3:] = [dense, 0, dense]
    indptr = np.concatenate([[0], np.cumsum(lens)])
    nnz = int(indptr[-1])
    which = np.repeat(np.arange(rows), lens)
    k = np.arange(nnz) - indptr[which]
    ind = (which // 1024 * 1024 + k).clip(0, rows + 5)  # (the last past the state)
    data = rng.standard_normal(nnz) + 1j * rng.standard_normal(nnz)
    x = rng.standard_normal(rows) + 1j * rng.standard_normal(rows)
    m = qa.SpMat.new_unchecked((rows, rows), data, ind.astype(np.uint64), indptr.astype(np.uint64))
    print(f"[gpu] uneven rows n={n} mean={mean} dense={dense} nnz={nnz}", flush=True)
    assert 24 * nnz > 1 << 28
    y = qa.spmat_dot_densevec(m, torch.from_numpy(x).cuda()).cpu().numpy()
    prod = np.where(ind < rows, data * x[np.minimum(ind, rows - 1)], 0)
    size = np.where(ind < rows, np.abs(data) * np.abs(x[np.minimum(ind, rows - 1)]), 0)
    starts = np.minimum(indptr[:-1], nnz - 1)
    ref = np.where(lens > 0, np.add.reduceat(prod, starts), 0)
    bound = np.where(lens > 0, np.add.reduceat(size, starts), 0) * (2 * lens + 8) * 2.3e-16
    assert np.all(np.abs(y - ref) <= bound + 1e-300)
