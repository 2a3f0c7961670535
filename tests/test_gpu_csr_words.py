"""CSR builds by sign words (k_csr_build_words), real and complex coefficients:
bit-exact against the oracle's rows at the edges of its layout -- groups of 1 to
past the terms held in registers, zero coefficients of both signs, one and many rows per batch,
sub-operators, more heavy groups than LDS holds, and row windows that begin
and end inside a tile."""
import ctypes

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


def _op(labels, coeffs):
    import qrusty_amd as qa
    return qa.SparsePauliOp([qa.Pauli(s) for s in labels], coeffs)


def _label(n, xm, zm):
    return "".join("IXZY"[((xm >> q) & 1) | (((zm >> q) & 1) << 1)] for q in reversed(range(n)))


def _operator(n, groups, sizes, seed, real):
    """`groups` masks of sizes[k % len(sizes)] terms each, in shuffled order,
    some coefficients 0.0 or -0.0.  `real`: every c' real (an even number of Y,
    or an odd one with an imaginary coefficient)."""
    rng = np.random.default_rng(seed)
    masks = rng.choice(1 << n, size=min(groups, 1 << n), replace=False)
    labels, coeffs = [], []
    for k, xm in enumerate(masks):
        for _ in range(sizes[k % len(sizes)]):
            zm = int(rng.integers(0, 1 << n))
            c, d = (float(rng.choice([0.0, -0.0, rng.normal()], p=[0.05, 0.05, 0.9])) for _ in range(2))
            if real:
                d = float(rng.choice([0.0, -0.0]))
                if bin(int(xm) & zm).count("1") % 2:
                    c, d = 0.0, c
            labels.append(_label(n, int(xm), zm))
            coeffs.append(complex(c, d))
    order = rng.permutation(len(labels))
    return [labels[i] for i in order], [coeffs[i] for i in order]


CASES = [(3, 1, [1]), (5, 7, [1, 2]), (9, 25, [2, 2, 2, 48]), (8, 200, [1, 2, 3, 4, 5, 6, 7, 8]),
         (11, 500, [4, 4, 6]), (11, 1024, [3]), (11, 1025, [2, 5]), (12, 2600, [4, 4, 4, 6, 9]),
         (12, 90, [40] * 60 + [2] * 30), (10, 130, [12])]


@pytest.mark.parametrize("real", [True, False])
@pytest.mark.parametrize("n,groups,sizes", CASES)
def test_whole(n, groups, sizes, real):
    labels, coeffs = _operator(n, groups, sizes, 10 * n + groups, real)
    p = orc.Params(labels, coeffs)
    assert real == bool(np.all(p.cp.view(np.float64)[1::2] == 0.0))
    print(f"[gpu] build real={real} n={n} groups={groups} T={len(labels)}", flush=True)
    ip, ind, dat = orc.build_csr(p)
    _, data, indices, indptr = _op(labels, coeffs).to_matrix_mode("RowwiseUnsafeChunked/100").export()
    assert indptr.tobytes() == ip.tobytes()
    assert indices.tobytes() == ind.tobytes()
    assert data.tobytes() == dat.tobytes()


@pytest.mark.parametrize("real", [True, False])
@pytest.mark.parametrize("n,groups,sizes", [(1, 2, [1]), (14, 1, [1]), (16, 2, [1, 3]), (17, 1, [9]), (16, 3, [2])])
def test_few_groups(n, groups, sizes, real):
    """One to three groups: the tiles of the most rows, several of them."""
    test_whole(n, groups, sizes, real)


@pytest.mark.parametrize("real", [True, False])
@pytest.mark.parametrize("n,groups,sizes", [(13, 300, [2, 4, 30]), (13, 1500, [4, 6]), (13, 20, [2, 2, 50])])
def test_row_windows(n, groups, sizes, real):
    from qrusty_amd import _lib as L
    labels, coeffs = _operator(n, groups, sizes, n + groups, real)
    p, op = orc.Params(labels, coeffs), _op(labels, coeffs)
    h = op._handle(L.QR_PHASE_ROWWISE)
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for r0, r1 in [(0, 1), (5, 9), (31, 33), (100, 4500), (4097, 8192), (8191, 8192)]:
        nnz = (r1 - r0) * h.G
        # a guard entry on both sides
        ix = torch.full((nnz + 2,), -7, dtype=torch.int64, device="cuda")
        d = torch.full((nnz + 2,), 7.0, dtype=torch.complex128, device="cuda")
        print(f"[gpu] build real={real} rows {r0}..{r1} of n={n} groups={groups}", flush=True)
        L.check(L.lib.qr_csr_build_rows(h.h, r0, r1, ctypes.c_void_p(ix.data_ptr() + 8),
                                        ctypes.c_void_p(d.data_ptr() + 16), s))
        ih, dh = ix.cpu().numpy(), d.cpu().numpy()
        assert ih[0] == ih[-1] == -7 and dh[0] == dh[-1] == 7.0
        for r in sorted({r0, (r0 + r1) // 2, r1 - 1}):
            cols, vals = orc.make_row(p, r)
            a = 1 + (r - r0) * h.G
            assert np.array_equal(ih[a:a + h.G].view(np.uint64), cols)
            assert dh[a:a + h.G].tobytes() == vals.tobytes()


@pytest.mark.parametrize("real,terms", [(True, [1]), (True, [4, 6]), (False, [1, 2]), (False, [6])])
@pytest.mark.parametrize("parts", [(488, 537), (700, 330, 20, 1), (300, 480, 10, 400), (1000, 30, 3, 200)])
def test_uneven_sub_operators(parts, real, terms):
    """Sub-operators of unlike sizes, in one launch or several."""
    rng, n = np.random.default_rng(sum(parts)), 12
    labels, coeffs = [], []
    for k, size in enumerate(parts):
        for j, m in enumerate(rng.choice(1 << 10, size, replace=False)):
            for _ in range(terms[j % len(terms)]):
                x, z = int(m) | k << 10, int(rng.integers(1 << n))
                c = complex(rng.normal(), 0.0 if real else rng.normal())
                labels.append(_label(n, x, z))
                coeffs.append(c * 1j ** bin(x & z).count("1") if real else c)
    p = orc.Params(labels, coeffs)
    print(f"[gpu] build by uneven sub-operators {parts} real={real} terms={terms}", flush=True)
    ip, ind, dat = orc.build_csr(p)
    _, data, indices, indptr = _op(labels, coeffs).to_matrix_mode("RowwiseUnsafeChunked/100").export()
    assert indptr.tobytes() == ip.tobytes()
    assert indices.tobytes() == ind.tobytes()
    assert data.tobytes() == dat.tobytes()


@pytest.mark.parametrize("n,groups,sizes", [(13, 1500, [1, 2]), (13, 40, [3]), (40, 60, [2]), (34, 2100, [1])])
def test_every_row_of_a_window(n, groups, sizes):
    """Windows of any number of tiles (the XCDs' ranges are not equal): every row
    as in the window that holds them all."""
    from qrusty_amd import _lib as L
    low = min(n, 13)
    labels, coeffs = _operator(low, groups, sizes, groups, False)
    op = _op(["Z" * (n - low) + s for s in labels], coeffs)
    h = op._handle(L.QR_PHASE_ROWWISE)
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)

    def rows(r0, r1):
        ix = torch.full(((r1 - r0) * h.G,), -7, dtype=torch.int64, device="cuda")
        d = torch.full(((r1 - r0) * h.G,), 7.0, dtype=torch.complex128, device="cuda")
        L.check(L.lib.qr_csr_build_rows(h.h, r0, r1, ctypes.c_void_p(ix.data_ptr()), ctypes.c_void_p(d.data_ptr()), s))
        return ix, d

    print(f"[gpu] build windows n={n} groups={groups}", flush=True)
    ix, d = rows(0, 4096)
    assert int((ix == -7).sum()) == 0
    for tiles in range(1, 16):
        r0, r1 = 16 * (tiles % 5), min(4096, 16 * (tiles % 5) + (16 if groups > 500 else 256) * tiles + tiles % 3)
        for got, want in zip(rows(r0, r1), (ix, d)):
            assert torch.equal(got.view(torch.uint8), want[r0 * h.G:r1 * h.G].view(torch.uint8)), (r0, r1)


@pytest.mark.parametrize("n,groups,sizes", [(9, 25, [2, 2, 2, 48]), (10, 300, [1, 3]), (12, 2600, [4, 4, 4, 6, 9])])
def test_captured_before_any_build(n, groups, sizes):
    """An operator whose first build is recorded into a graph, after an apply put
    its other tables on the device: the tile builder's entries, on every replay."""
    from qrusty_amd import _lib as L
    labels, coeffs = _operator(n, groups, sizes, 3 * n + groups, False)
    p, op = orc.Params(labels, coeffs), _op(labels, coeffs)
    h = op._handle(L.QR_PHASE_ROWWISE)
    ip, ind, dat = orc.build_csr(p)
    x = torch.ones(p.N, dtype=torch.complex128, device="cuda")
    op.apply(x)
    out = [torch.empty(p.N + 1, dtype=torch.int64, device="cuda"), torch.empty(len(ind), dtype=torch.int64, device="cuda"),
           torch.empty(len(ind), dtype=torch.complex128, device="cuda")]
    print(f"[gpu] captured first build n={n} groups={groups}", flush=True)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        L.check(L.lib.qr_csr_build(h.h, *(ctypes.c_void_p(t.data_ptr()) for t in out),
                                   ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    for _ in range(3):
        for t in out:
            t.fill_(7)
        op.apply(x)
        torch.cuda.synchronize()
        graph.replay()
        for t, want in zip(out, (ip, ind, dat)):
            assert t.cpu().numpy().tobytes() == want.tobytes()
