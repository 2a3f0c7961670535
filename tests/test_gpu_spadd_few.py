"""a*A + b*B where one matrix has few entries per row: bit-exact against the
oracle's merge at the edges of the layout -- rows that fill and overflow their
lanes, none, one or several entries of the short matrix before, between, on
and after the long one's, exact cancellations, -0.0, both argument orders, row
counts around a wave's 64 and the one-block scan's 1024 and 2^14."""
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


def _csr(rows, cols, lens, rng):
    indptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    ind = [np.sort(rng.choice(cols, size=int(n), replace=False)) for n in lens] + [np.zeros(0, np.int64)]
    n = int(indptr[-1])
    data = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    data[rng.random(n) < 0.05] = 0.0
    data.imag[rng.random(n) < 0.2] = -0.0
    return indptr, np.concatenate(ind).astype(np.uint64), data


# rows, columns, lengths of the long matrix's rows, of the short one's
CASES = [(1, 1, [1], [1]), (63, 40, [4], [1]), (64, 40, [5, 8], [1]), (65, 40, [24], [1, 0]),
         (4097, 64, [24], [1]), (1000, 64, [32], [1]), (1000, 64, [33, 20], [0, 1, 2]), (200, 200, [64], [1]),
         (200, 300, [65, 130, 1], [1]), (300, 2000, [981, 3, 0], [5, 0, 1, 0]), (70000, 30, [3], [1]),
         (130, 900, [0, 0, 0, 900], [2, 1, 0]), (1023, 20, [2], [1]), (1025, 20, [0, 5], [1]),
         (16384, 20, [2], [1]), (16385, 20, [2], [1])]


@pytest.mark.parametrize("rows,cols,long,short", CASES)
def test_few(rows, cols, long, short):
    import qrusty_amd as qa
    rng = np.random.default_rng(rows + cols)
    a = _csr(rows, cols, np.resize(long, rows), rng)
    b = _csr(rows, cols, np.resize(short, rows), rng)
    # half of the short matrix's entries on an entry of the long one, some of
    # those its negative
    for r in range(rows):
        lo, hi = int(a[0][r]), int(a[0][r + 1])
        if hi == lo or r % 2:
            continue
        k0, k1 = int(b[0][r]), int(b[0][r + 1])
        pick = np.sort(rng.choice(np.arange(lo, hi), size=min(k1 - k0, hi - lo), replace=False))
        if len(pick) == k1 - k0:
            b[1][k0:k1] = a[1][pick]
            if r % 4 == 0:
                b[2][k0:k1] = -a[2][pick]
    ma, mb = (qa.SpMat.new_unchecked((rows, cols), m[2], m[1], m[0]) for m in (a, b))
    print(f"[gpu] spadd few rows={rows} cols={cols} long={long} short={short}", flush=True)
    for s, t in [(1.0, 1.0), (0.3 - 1.1j, -2.0 + 0.5j), (0.0, 1.0)]:
        for first, second, m1, m2 in [(a, b, ma, mb), (b, a, mb, ma)]:
            _, data, indices, indptr = qa.a_spmat_p_b_spmat(s, m1, t, m2).export()
            ref = orc.csr_add(rows, s, first, t, second)
            assert np.array_equal(indptr, ref[0]) and np.array_equal(indices, ref[1])
            assert np.array_equal(np.asarray(data).view(np.uint64), np.asarray(ref[2]).view(np.uint64))


@pytest.mark.parametrize("rows,cols,long,short", [(300, 9, [8, 2, 5], [1]), (300, 9, [8, 2, 5], [0, 2, 1, 1]),
                                                  (130, 6, [24, 2], [1]), (130, 6, [24, 2], [2, 0]), (130, 40, [64], [1]),
                                                  (130, 12, [300, 900, 2], [1, 3]), (1, 6, [2], [1])])
def test_few_of_any_order(rows, cols, long, short):
    """Rows whose columns do not ascend or come twice: every entry keeps a place
    of its own, those of the merge.  (As many short entries as rows and a whole
    number of long ones per row, or rows too long for the staged tile: the sums
    that lane groups take.)"""
    import qrusty_amd as qa
    rng = np.random.default_rng(rows + cols + len(short))

    def matrix(lens):
        lens = np.resize(lens, rows)
        indptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
        n = int(indptr[-1])
        return indptr, rng.integers(0, cols, n).astype(np.uint64), rng.integers(-1, 2, n) + 1j * rng.integers(-1, 2, n)

    a, b = matrix(long), matrix(short)
    if rows == 1:
        a[1][:], b[1][:], a[2][:], b[2][:] = [5, 2], [3], [1, 2], [4]
    ma, mb = (qa.SpMat.new_unchecked((rows, cols), m[2], m[1], m[0]) for m in (a, b))
    print(f"[gpu] spadd few, any order rows={rows} cols={cols} long={long} short={short}", flush=True)
    for first, second, m1, m2 in [(a, b, ma, mb), (b, a, mb, ma)]:
        _, data, indices, indptr = qa.a_spmat_p_b_spmat(1.0, m1, -1.0, m2).export()
        ref = orc.csr_add(rows, 1.0, first, -1.0, second)
        assert np.array_equal(indptr, ref[0]) and np.array_equal(indices, ref[1])
        assert np.array_equal(np.asarray(data).view(np.uint64), np.asarray(ref[2]).view(np.uint64))


# rows that do and do not fit their lanes side by side (as many short entries as
# rows), and long rows on both sides of the rule
UNEVEN = [(64, 40, [5, 30], [0, 2]), (1000, 90, [3, 70, 20, 40], [0, 2, 1, 1]), (131, 90, [2, 90, 1], [1]),
          (4, 30, [3, 9], [4, 0, 0, 0]), (77, 300, [127], [1]), (77, 300, [128], [1]), (50, 400, [190, 194], [2]),
          (50, 400, [190, 193], [2]), (40, 900, [1, 800, 0, 300], [1])]


@pytest.mark.parametrize("rows,cols,long,short", UNEVEN)
def test_few_uneven(rows, cols, long, short):
    test_few(rows, cols, long, short)
