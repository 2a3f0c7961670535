"""Batches on both sides of the small-operator size (2^21 entries): one kernel
for the small ones, graph branches for the others.  CSR bit-exact against the
single-operator build and y within 1e-12 of the oracle, componentwise against
sum_t |c'_t||x[r ^ x_t]|, over replays with other states; indptr alone (no
CSR) is written too."""
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


def _case(specs):
    import qrusty_amd as qa
    from qrusty_amd import workloads
    ops, params = [], []
    for k, (n, t) in enumerate(specs):
        labels, coeffs = workloads.random_op(n, t, seed=0x77 + 13 * k)
        ops.append(qa.SparsePauliOp([qa.Pauli(l) for l in labels], coeffs))
        params.append(orc.Params(labels, coeffs))
    return ops, params


def _check_y(p, x, y):
    rows = np.unique(np.concatenate([[0, p.N - 1], np.random.default_rng(1).integers(0, p.N, 64)])).astype(np.uint64)
    ref = orc.apply_rows(p, x, rows)[0]
    bound = sum(abs(c) * np.abs(x[(rows ^ xm).astype(np.int64)]) for c, xm in zip(p.cp.view(np.complex128), p.x))
    assert np.all(np.abs(y[rows.astype(np.int64)] - ref) <= 1e-12 * bound + 1e-300)


# all small; one large; more large ones than branches beside small ones
@pytest.mark.parametrize("specs", [[(3, 4), (10, 900)], [(12, 700)],
                                   [(12, 600 + 40 * k) for k in range(11)] + [(5, 30), (11, 1500), (9, 100)]])
@pytest.mark.parametrize("split", [0, 1])
def test_both_sides(specs, split):
    import qrusty_amd as qa
    from qrusty_amd import workloads
    ops, params = _case(specs)
    b = qa.Batch(ops)
    single = [op.to_matrix_mode("RowwiseUnsafeChunked/100").device_arrays() for op in ops]
    for rep in range(3):
        xs = [workloads.random_states(p.N, 1, 50 * rep + k)[0] for k, p in enumerate(params)]
        b.set_states(xs)
        print(f"[gpu] batch of {len(specs)} split={split} run {rep}", flush=True)
        b.run({"tiles_per_item": 1 + rep // 2, "blocks_per_cu": 1, "order": rep % 2, "split": split})
        torch.cuda.synchronize()
        for k, p in enumerate(params):
            for got, ref in zip(b.csr(k), single[k]):
                assert torch.equal(got.reshape(-1).view(torch.uint8), ref.reshape(-1).view(torch.uint8))
            _check_y(p, xs[k], b.y[k].cpu().numpy())


@pytest.mark.parametrize("n,t", [(6, 20), (12, 800)])
def test_indptr_alone(n, t):
    import qrusty_amd as qa
    from qrusty_amd import _lib as L
    from qrusty_amd import workloads
    ops, params = _case([(n, t)])
    b = qa.Batch(ops, keep_csr=False)
    x = workloads.random_states(1 << n, 1, 3)[0]
    b.set_states([x])
    ip = torch.full(((1 << n) + 1,), -1, dtype=torch.int64, device="cuda")
    pp = (ctypes.c_void_p * 1)(ip.data_ptr())
    print(f"[gpu] batch indptr alone n={n}", flush=True)
    L.check(L.lib.qr_batch_run(b._b, pp, b._pi, b._pd, b._px, b._py, None,
                               ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    torch.cuda.synchronize()
    G = len(np.unique(params[0].x))
    assert np.array_equal(ip.cpu().numpy(), np.arange((1 << n) + 1) * G)
    _check_y(params[0], x, b.y[0].cpu().numpy())


# states of 2 to 32 tiles: every mask of the tile and a few past it (gathers), or
# masks all over (partner tiles staged); from 64 groups, shares of few, on
@pytest.mark.parametrize("form", ["1", "2"])
@pytest.mark.parametrize("n,groups,real", [(11, 1025, True), (11, 1500, False), (12, 1100, True), (13, 2049, False),
                                           (14, 150, True), (15, 70, False)])
def test_groups_in_shares(monkeypatch, n, groups, real, form):
    import qrusty_amd as qa
    from qrusty_amd import workloads
    monkeypatch.setenv("QR_APPLY_FORM", form)
    rng = np.random.default_rng(n * groups)
    low = rng.permutation(min(1 << 10, groups - 3))[:groups - 3]
    masks = list(low) + list(rng.choice(np.arange(1 << 10, 1 << n), groups - len(low), replace=False))
    labels, coeffs = [], []
    for m in masks:
        for _ in range(rng.integers(1, 4)):
            z = int(rng.integers(1 << n))
            labels.append("".join("IZXY"[2 * (int(m) >> q & 1) + (z >> q & 1)] for q in reversed(range(n))))
            ny = bin(int(m) & z).count("1")
            c = complex(rng.standard_normal(), 0 if real else rng.standard_normal())
            coeffs.append(c * 1j ** ny if real else c)
    op = qa.SparsePauliOp([qa.Pauli(s) for s in labels], coeffs)
    p = orc.Params(labels, coeffs)
    assert len(np.unique(p.x)) == groups and groups << n > 1 << 21
    for keep in (True, False):
        b = qa.Batch([op], keep_csr=keep)
        for rep in range(3):
            x = workloads.random_states(p.N, 1, 11 * rep + n)[0]
            b.set_states([x])
            print(f"[gpu] batch, groups in shares n={n} groups={groups} real={real} form={form} run {rep}", flush=True)
            b.run()
            torch.cuda.synchronize()
            _check_y(p, x, b.y[0].cpu().numpy())
