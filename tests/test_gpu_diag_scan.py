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


@pytest.mark.parametrize("rows,lens", [(300, [8, 0, 16, 17, 1, 40]), (65, [31, 32, 33, 0]), (64, [48, 100, 64, 65, 3]),
                                       (1, [9]), (257, [2, 30]), (4096, [12] * 63 + [2000])])
def test_scan_of_uneven_rows(rows, lens):
    """Rows on both sides of what their lanes read at a time, in one wave; some
    that start past the matrix's entries, and end before they start."""
    import qrusty_amd as qa
    from oracle import oracle as orc
    rng = np.random.default_rng(rows + len(lens))
    lens, cols = np.resize(lens, rows), max(rows, 2000)
    indptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    ind = []
    for r, n in enumerate(lens):
        c = rng.choice(cols, size=int(n), replace=False)
        if n and r % 3 and r not in c:
            c[rng.integers(n)] = r
        ind.append(np.sort(c))
    indices = np.concatenate(ind).astype(np.uint64)
    data = rng.standard_normal(len(indices)) + 1j * rng.standard_normal(len(indices))
    print(f"[gpu] diagonal scan, uneven rows={rows} lens={lens[:6]}", flush=True)
    m = qa.SpMat.new_unchecked((rows, cols), data, indices, indptr)
    assert np.array_equal(np.asarray(m.diagonal()), orc.csr_diagonal((rows, cols), indptr, indices, data))
    if rows > 8:
        bad = indptr.copy()
        bad[3], bad[5], bad[-2] = bad[-1] + np.uint64(9), np.uint64(0), np.uint64(1) << np.uint64(40)
        m = qa.SpMat.new_unchecked((rows, cols), data, indices, bad)
        got, want = np.asarray(m.diagonal()), orc.csr_diagonal((rows, cols), indptr, indices, data)
        ok = [r for r in range(6, rows - 3)]
        assert np.array_equal(got[ok], want[ok])
