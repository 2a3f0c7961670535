"""CPU tests of which kernels the library launches and what it allocates: each
runs in a process of its own over hip_stub.c, a HIP runtime that runs nothing,
with addresses that nothing reads."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(HERE)

PRELUDE = """
import ctypes, sys
stub = ctypes.CDLL({stub!r}, mode=ctypes.RTLD_GLOBAL)
stub.stub_name.restype = ctypes.c_char_p
stub.stub_arg.restype = stub.stub_blocks.restype = ctypes.c_uint32
stub.stub_malloc_bytes.restype = ctypes.c_uint64
sys.path.insert(0, {repo!r})
from qrusty_amd import _lib as L
GB = 1 << 30

def op_of(labels, coeffs=None):
    n = len(labels)
    coeffs = coeffs or [1.0 + 0.5 * k for k in range(n)]
    c = (ctypes.c_double * (2 * n))(*[v for z in coeffs for v in (complex(z).real, complex(z).imag)])
    h = ctypes.c_void_p()
    L.check(L.lib.qr_op_create((ctypes.c_char_p * n)(*[s.encode() for s in labels]), c, n, 0, ctypes.byref(h)))
    return h

def term(n, ops):
    chars = ["I"] * n
    for q, ch in ops.items():
        chars[n - 1 - q] = ch
    return "".join(chars)

def launched(part):
    return [(stub.stub_name(i).decode(), stub.stub_arg(i), stub.stub_blocks(i))
            for i in range(stub.stub_launches()) if part in stub.stub_name(i).decode()]
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    stub = str(tmp_path_factory.mktemp("stub") / "hip_stub.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", stub, os.path.join(HERE, "hip_stub.c")], check=True)

    def go(body):
        res = subprocess.run([sys.executable, "-c", PRELUDE.format(stub=stub, repo=REPO) + body],
                             capture_output=True, text=True, timeout=120)
        assert res.returncode == 0, res.stdout + res.stderr

    return go


@pytest.mark.parametrize("split", ["", "1"])
@pytest.mark.parametrize("n,prec,kind", [(22, 0, "x17"), (23, 0, "bonds17"), (24, 0, "x17"), (28, 0, "x21"),
                                         (28, 1, "x21")])
def test_every_apply_pass_has_groups(run, n, prec, kind, split):
    """The wait for a tile's loads into LDS lies in the loop over the pass's
    chunks, so no pass may run without one: operators that window passes take
    whole."""
    run(f"""
import os
if {split!r}:
    os.environ["QR_APPLY_SPLIT"] = {split!r}
n = {n}
if {kind!r} == "bonds17":
    labels = [term(n, {{q: p, q + 1: p}}) for q in range(17, n - 1) for p in "XY"]
else:
    labels = [term(n, {{q: "X"}}) for q in range(int({kind!r}[1:]), n)]
stub.stub_watch(b"k_apply_tiled", 4)
op = op_of(labels)
L.check(L.lib.qr_pauli_apply(op, {prec}, 1, 64 * GB, 128 * GB, 192 * GB, None))
passes = launched("k_apply_tiled")
assert passes and all(nchunk > 0 for _, nchunk, _ in passes), passes
""")


@pytest.mark.parametrize("n", [24, 26, 28])
def test_complex64_apply_is_one_pass(run, n):
    """y of a complex64 state is rounded once, when it is written: its sum does
    not go through memory between passes."""
    run(f"""
n = {n}
labels = [term(n, {{q: "X", (q + 1) % n: "X"}}) for q in range(n)]
op = op_of(labels)
L.check(L.lib.qr_pauli_apply(op, L.QR_PREC_MIXED, 1, 64 * GB, 128 * GB, None, None))
assert len(launched("k_apply")) == 1, launched("k_apply")
""")


@pytest.mark.parametrize("groups,heavy", [(5, 1), (8, 1), (12, 2), (32, 6), (64, 15), (128, 30)])
def test_build_folds_every_heavy_group(run, groups, heavy):
    """A tile of the CSR build has room for the values of all heavy groups (16
    bytes a row each, after two stages of 24 bytes per entry of a batch): those
    that it does not fold it loads term by term for every row."""
    run(f"""
n, groups, heavy = 24, {groups}, {heavy}
labels = []
for g in range(groups):
    for t in range(64 if g < heavy else 1):
        xz = (g << 12, t)
        labels.append("".join("IZXY"[2 * (xz[0] >> q & 1) + (xz[1] >> q & 1)] for q in reversed(range(n))))
op = op_of(labels)
L.check(L.lib.qr_csr_build(op, 64 * GB, 128 * GB, 192 * GB, None))
(k,) = [i for i in range(stub.stub_launches()) if "k_csr_build" in stub.stub_name(i).decode()]
rows = (1 << n) // stub.stub_blocks(k)
per_batch = 1024 >> (groups - 1).bit_length()
assert stub.stub_shmem(k) >= 48 * groups * per_batch + 16 * heavy * rows, (stub.stub_shmem(k), rows)
""")


def test_apply_uploads_no_build_tables(run):
    """The sign-word builder's tables, 4 n bytes per group and more, come to the
    device with the first CSR build; one that is captured before takes the tile
    builder, which needs none, and neither allocates nor copies."""
    run("""
n = 24
labels = [term(n, {q: c for q, c in zip(range(a, a + 6), cs)}) for a in range(18)
          for cs in __import__("itertools").product("XY", "XYZ", "XI", "XZ", "IX", "XI")]
labels = list(dict.fromkeys(labels))
op, same = op_of(labels), op_of(labels)
groups = ctypes.c_uint64()
L.check(L.lib.qr_op_info(op, None, None, ctypes.byref(groups), None))
rank = 4 * n * groups.value
L.check(L.lib.qr_pauli_apply(op, 0, 1, 64 * GB, 128 * GB, None, None))
applied = stub.stub_malloc_bytes()
stub.stub_capture(1)
L.check(L.lib.qr_csr_build(op, 64 * GB, 128 * GB, 192 * GB, None))
stub.stub_capture(0)
assert stub.stub_syncs_in_capture() == 0 and stub.stub_malloc_bytes() == applied
assert launched("k_csr_build_staged") and not launched("k_csr_build_words")
L.check(L.lib.qr_csr_build(op, 64 * GB, 128 * GB, 192 * GB, None))
assert launched("k_csr_build_words") and stub.stub_malloc_bytes() >= applied + rank
built = stub.stub_malloc_bytes()
stub.stub_capture(1)
L.check(L.lib.qr_csr_build(op, 64 * GB, 128 * GB, 192 * GB, None))
stub.stub_capture(0)
assert stub.stub_syncs_in_capture() == 0 and stub.stub_malloc_bytes() == built
stub.stub_reset()
L.check(L.lib.qr_csr_build(same, 64 * GB, 128 * GB, 192 * GB, None))
assert rank <= stub.stub_malloc_bytes() and launched("k_csr_build_words")
""")


def test_batch_graph_ends_with_its_descriptors(run):
    """A tuning pass that fails part of the way has replaced the descriptors that
    the recorded graph reads: the next run records again."""
    run("""
ops = [op_of([term(8, {q: "X"}) for q in range(k)]) for k in (2, 5)]
batch = ctypes.c_void_p()
L.check(L.lib.qr_batch_create((ctypes.c_void_p * 2)(*ops), 2, ctypes.byref(batch)))

def args(at):
    return [ctypes.cast((ctypes.c_void_p * 2)((at + 2 * k) * GB, (at + 2 * k + 1) * GB), ctypes.c_void_p) for k in range(5)]

first, second = args(64), args(128)
L.check(L.lib.qr_batch_run(batch, *first, None, None))
L.check(L.lib.qr_batch_run(batch, *first, None, None))
assert stub.stub_graphs_made() == 1
stub.stub_fail_malloc_after.argtypes = [ctypes.c_long]
stub.stub_fail_malloc_after(0)  # the matvec pass's descriptors, in the split candidates
assert L.lib.qr_batch_tune(batch, *second, None, None) == -6
stub.stub_fail_malloc_after(-1)
L.check(L.lib.qr_batch_run(batch, *first, None, None))
assert stub.stub_graphs_made() == 2
""")


@pytest.mark.parametrize("n,prec,groups,form,few", [(24, 0, 100, "tiled", True), (20, 0, 90, "tiled", True),
                                                    (20, 0, 40, "staged", False), (19, 0, 100, "tiled", False),
                                                    (16, 0, 1, "staged", False), (22, 1, 100, "staged", False),
                                                    (24, 1, 100, "staged", False), (21, 1, 100, "tiled", False),
                                                    (24, 0, "ring", "tiled", False), (24, 0, "shared", "staged", False)])
def test_apply_form(run, n, prec, groups, form, few):
    """Groups on partners of their own past L2: gathers by two blocks per CU, or
    staged where they are few or the state is complex64 (past its caches); others
    as before."""
    run(f"""
import random
rng, n, groups = random.Random(5), {n}, {groups!r}
if groups == "ring":
    labels = [term(n, {{q: p, (q + 1) % n: p}}) for q in range(n) for p in "XYZ"]
elif groups == "shared":
    labels = [term(n, {{q: "X", p: "X"}}) for q in range(10, n) for p in range(10)]
else:
    labels = ["X" + "".join(rng.choice("IXYZ") for _ in range(n - 1)) for _ in range(groups)]
op = op_of(labels)
L.check(L.lib.qr_pauli_apply(op, {prec}, 1, 64 * GB, 128 * GB, None, None))
names = launched("k_apply_")
assert all("k_apply_{form}" in k[0] for k in names), names
lds = max(stub.stub_shmem(i) for i in range(stub.stub_launches()))
assert (lds >= 80 << 10) == {few}, lds
""")


@pytest.mark.parametrize("n,longer,lanes,rows", [(16, 33 << 16, 6, 16), (16, (7 << 16) + 1, 4, 16), (20, 25 << 20, 5, 64),
                                                 (20, (22 << 20) + 1, 5, 64), (20, (60 << 20) + 1, 0, 0), (18, 9 << 18, 4, 64)])
def test_lanes_of_sums(run, n, longer, lanes, rows):
    """Lanes per row of a sum with a diagonal (0: staged tiles), enough for most
    rows where these cannot be equal, and rows per wave."""
    run(f"""
n, longer = 1 << {n}, {longer}
stub.stub_watch(b"k_spadd_few", 1)
one = (ctypes.c_double * 2)(1.0, 0.0)
L.check(L.lib.qr_csr_add_fill(n, one, longer, 64 * GB, 65 * GB, 66 * GB, one, n, 67 * GB, 68 * GB, 69 * GB, 70 * GB,
                              71 * GB, 72 * GB, None))
few = launched("k_spadd_few")
assert bool(few) == bool({lanes})
if few:
    assert few[0][1] == {lanes} and few[0][2] * 4 * {rows} == n, few
""")


@pytest.mark.parametrize("qubits,candidates", [((22, 23), 6), ((22, 8), 32)])
def test_tuning_times_no_candidate_twice(run, qubits, candidates):
    """Batches without small operators: orders, forms, and the matvec pass's blocks
    per CU, without the knobs that reach no kernel of the plan."""
    run(f"""
ops = [op_of([term(q, {{0: "X"}})]) for q in {qubits}]
batch = ctypes.c_void_p()
L.check(L.lib.qr_batch_create((ctypes.c_void_p * 2)(*ops), 2, ctypes.byref(batch)))
args = [ctypes.cast((ctypes.c_void_p * 2)((64 + 4 * k) * GB, (66 + 4 * k) * GB), ctypes.c_void_p) for k in range(5)]
L.check(L.lib.qr_batch_tune(batch, *args, None, None))
large = sum(q > 20 for q in {qubits})
assert len(launched("k_csr_build")) == {candidates} * 2 * large, len(launched("k_csr_build"))
""")


@pytest.mark.parametrize("n,groups", [(11, 1500), (12, 2000), (12, 3500), (14, 300)])
def test_batch_applies_of_few_tiles_fill_more_blocks(run, n, groups):
    """y of a batch's operator whose state has few tiles: its many groups are
    shared among blocks, not walked by one per tile."""
    run(f"""
import random
rng = random.Random(7)
masks = rng.sample(range(1 << {n}), {groups})
op = op_of(["".join("IX"[m >> q & 1] for q in reversed(range({n}))) for m in masks])
batch = ctypes.c_void_p()
L.check(L.lib.qr_batch_create((ctypes.c_void_p * 1)(op), 1, ctypes.byref(batch)))
args = [ctypes.cast((ctypes.c_void_p * 1)((64 + 4 * k) * GB), ctypes.c_void_p) for k in range(5)]
L.check(L.lib.qr_batch_run(batch, *args, None, None))
applies = launched("k_apply_")
assert len(applies) == 1 and applies[0][2] >= min(64, {groups} // 64 << ({n} - 10)), applies
assert len(launched("k_sum_parts")) == 1
""")


@pytest.mark.parametrize("sizes,terms,real,launches", [((488, 537), 1, True, 1), ((1000, 520, 505), 1, False, 1),
                                                       ((880, 220), 4, False, 1), ((880, 220), 6, False, 2),
                                                       ((40, 50, 60, 1000), 1, True, 2), ((900, 700, 600), 6, False, 1)])
def test_sub_operators_of_one_launch(run, sizes, terms, real, launches):
    """A build by sub-operators writes its rows from end to end, in one launch, but
    where that idles too many threads."""
    run(f"""
import random
rng, n = random.Random(3), 22
sizes, terms, real = {sizes}, {terms}, {real}
labels = []
for k, size in enumerate(sizes):
    # prefixes 0, 10, 110, ...: each leaves the subtree of those after it
    top = ((1 << k) - 1) << (12 - k)
    for m in rng.sample(range(1 << 9), min(size, 1 << 9)) + [512 + i for i in range(size - 512)]:
        for z in rng.sample(range(1 << 10), terms):
            x = (top << 10) | m
            labels.append("".join("IZXY"[2 * (x >> q & 1) + (z >> q & 1)] for q in reversed(range(n))))
op = op_of(labels, [1.0 + 0.5 * k if real else complex(1, 1 + k) for k in range(len(labels))])
groups = ctypes.c_uint64()
L.check(L.lib.qr_op_info(op, None, None, ctypes.byref(groups), None))
assert groups.value == sum(sizes)
L.check(L.lib.qr_csr_build(op, 64 * GB, 128 * GB, 192 * GB, None))
assert len(launched("k_csr_build_words")) == {launches}, launched("k_csr_build_words")
""")


@pytest.mark.parametrize("n,groups", [(14, 3), (22, 8), (20, 30)])
def test_sums_leave_the_tile_in_place(run, n, groups):
    """The LDS of an apply by gathers holds the tile of x (2^10 complex128) beside
    the sums of its thread groups (16 bytes a row for every second of them): <x|y>
    does not read x again."""
    run(f"""
import re
op = op_of([term({n}, {{q % 4: "X", q // 4: "Y" if q // 4 != q % 4 else "X"}}) for q in range({groups})])
L.check(L.lib.qr_pauli_apply(op, 0, 1, 64 * GB, 128 * GB, 192 * GB, None))
applies = [(re.search("k_apply_tiled.*Li10ELi([24])E", stub.stub_name(i).decode()), stub.stub_shmem(i))
           for i in range(stub.stub_launches())]
applies = [(int(m[1]), lds) for m, lds in applies if m]
assert applies and all(lds >= (16 << 10) * (1 + split // 2) for split, lds in applies), applies
""")


@pytest.mark.parametrize("n,groups,far,split", [(22, 9, 0, 1), (26, 16, 0, 1), (24, 8, 0, 2), (21, 16, 0, 2), (23, 12, 1, 2),
                                                (14, 12, 0, 4)])
def test_thread_groups_inside_the_tile(run, n, groups, far, split):
    """Operators of more than 8 groups, all inside the tile, have one thread group
    per block where the tiles fill the chip many times."""
    run(f"""
import itertools
pairs = list(itertools.combinations(range(8), 2))
labels = [term({n}, {{a: "X", b: "X", 13: "Z"}}) for a, b in pairs[:{groups} - {far}]]
labels += [term({n}, {{12: "X", a: "X"}}) for a in range({far})]
op = op_of(labels)
if {far}:
    __import__("os").environ["QR_APPLY_FORM"] = "1"
L.check(L.lib.qr_pauli_apply(op, 0, 1, 64 * GB, 128 * GB, None, None))
names = [k[0] for k in launched("k_apply_")]
assert names and all("tiled" in k and "Li10ELi{split}E" in k for k in names), names
""")


@pytest.mark.parametrize("n,bonds,near,form", [(24, range(10, 22, 2), 3, "tiled"), (22, range(9, 20), 2, "tiled"),
                                               (24, range(10, 18, 2), 0, "staged"), (24, range(10, 22, 2), 7, "staged"),
                                               (21, range(10, 20, 2), 3, "tiled")])
def test_form_of_some_partners(run, n, bonds, near, form):
    """FP64, partners of their own for 5 to 12 groups, half of them or more, half
    of the partners in L2: gathers; with fewer, or more groups inside the
    tile, staged from 2^22 rows on."""
    run(f"""
labels = [term({n}, {{q: "X", q + 1: "Y"}}) for q in {list(bonds)}] + [term({n}, {{q: "X"}}) for q in range({near})]
op = op_of(labels)
L.check(L.lib.qr_pauli_apply(op, 0, 1, 64 * GB, 128 * GB, None, None))
names = [k[0] for k in launched("k_apply_")]
assert names and all("k_apply_{form}" in k for k in names), names
""")


@pytest.mark.parametrize("qubits,longer,few", [(22, 1, False), (22, 2, False), (22, 3, True), (21, 1, True)])
def test_sums_of_few_strings(run, qubits, longer, few):
    """One entry per row in one matrix and one or two in the other, many rows: the
    staged tiles."""
    run(f"""
n = 1 << {qubits}
one = (ctypes.c_double * 2)(1.0, 0.0)
L.check(L.lib.qr_csr_add_fill(n, one, {longer} * n, 64 * GB, 65 * GB, 66 * GB, one, n, 67 * GB, 68 * GB, 69 * GB, 70 * GB,
                              71 * GB, 72 * GB, None))
assert bool(launched("k_spadd_few")) == {few} and bool(launched("k_spadd_tile")) != {few}
""")
