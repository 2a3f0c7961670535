"""diagonal() and precond() where lane groups scan the rows (8 to 48 entries in
the mean): the diagonal on any entry of a row, absent, or in an empty row, rows
longer and shorter than a group's four loads per lane, square and rectangular
shapes; the diagonal exactly, precond as precond2 of it to the last bit."""
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


@pytest.mark.parametrize("rows,cols,lens", [(31, 31, [8]), (64, 64, [9, 16]), (1000, 1000, [24]), (1000, 1000, [16, 0, 40]),
                                            (257, 257, [47]), (300, 300, [200, 1, 1, 1, 1, 1]), (500, 120, [20]),
                                            (120, 500, [33])])
def test_scan(rows, cols, lens):
    import qrusty_amd as qa
    rng = np.random.default_rng(rows + cols)
    lens = np.resize(lens, rows)
    ind, want = [], np.zeros(min(rows, cols), complex)
    for r, n in enumerate(lens):
        c = rng.choice(cols, size=int(n), replace=False)
        if n and r < cols and r % 3 and r not in c:
            c[rng.integers(n)] = r
        ind.append(np.sort(c))
    indptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    indices = np.concatenate(ind).astype(np.uint64)
    data = rng.standard_normal(len(indices)) + 1j * rng.standard_normal(len(indices))
    for r in range(min(rows, cols)):
        at = np.flatnonzero(ind[r] == r)
        if len(at):
            want[r] = data[int(indptr[r]) + at[0]]
    m = qa.SpMat.new_unchecked((rows, cols), data, indices, indptr)
    print(f"[gpu] diagonal scan rows={rows} cols={cols}", flush=True)
    diag = m.diagonal()
    assert np.array_equal(np.asarray(diag), want)
    dx = rng.standard_normal(min(rows, cols)) + 0.5j
    for e, tol in [(0.3 - 0.1j, 1e-3), (0.0, 0.5)]:
        assert np.array_equal(np.asarray(qa.precond(m, dx, e, tol)).view(np.uint64),
                              np.asarray(qa.precond2(want, dx, e, tol)).view(np.uint64))


@pytest.mark.parametrize("rows,mean", [(200, 8), (200, 13), (300, 31), (129, 47)])
def test_scan_of_repeated_columns(rows, mean):
    """Rows in any order that hold their diagonal column more than once: the
    first entry of the row that has it, whichever lanes read them."""
    import qrusty_amd as qa
    from oracle import oracle as orc
    rng = np.random.default_rng(rows + mean)
    indptr = np.arange(rows + 1, dtype=np.uint64) * np.uint64(mean)
    indices = rng.integers(0, rows, (rows, mean))
    for r in range(rows):
        if r % 2:
            indices[r].sort()
        at = (r // 2) % mean  # the pair on every place of the row, on two lanes or one
        indices[r, at] = indices[r, min(at + 1 + r % 5, mean - 1)] = r
        if r % 2:
            indices[r].sort()
    data = rng.standard_normal(rows * mean) + 1j * rng.standard_normal(rows * mean)
    indices = indices.reshape(-1).astype(np.uint64)
    want = orc.csr_diagonal((rows, rows), indptr, indices, data)
    m = qa.SpMat.new_unchecked((rows, rows), data, indices, indptr)
    print(f"[gpu] diagonal scan, repeated columns rows={rows} mean={mean}", flush=True)
    assert np.array_equal(np.asarray(m.diagonal()), want)
