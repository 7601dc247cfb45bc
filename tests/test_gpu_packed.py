"""Packed rows of the matrix-free operator (one vector and blocks) against the
assembled matrix of the same operator in 64-bit host arithmetic, over the
bases, operator strings, flags and scales the product takes."""

import numpy as np
import pytest
import scipy.sparse as sp

from models import chain_maps, hubbard_static, ladder_maps, xxz_static

pytestmark = pytest.mark.gpu

KW = dict(check_symm=False, check_herm=False, check_pcon=False)
EPS = {np.dtype(np.float32): 2.0 ** -24, np.dtype(np.complex64): 2.0 ** -24,
       np.dtype(np.float64): 2.0 ** -53, np.dtype(np.complex128): 2.0 ** -53}


def _all_to_all(L):
    pairs = [[0.1 * (i + 1), i, j] for i in range(L) for j in range(i + 1, L)]
    half = [[0.5 * J, i, j] for J, i, j in pairs]
    return [["+-", half], ["-+", half], ["zz", pairs]]


def _case(name):
    """(basis, static list, real elements)"""
    from quspin_amd.basis import (spin_basis_general, spinful_fermion_basis_general, spinless_fermion_basis_general)
    m = chain_maps(12)
    if name == "kpz":
        return spin_basis_general(12, Nup=6, pauli=0, kblock=(m["T"], 0), pblock=(m["P"], 0),
                                  zblock=(m["Z"], 0)), xxz_static(12), True
    if name == "momentum":
        return spin_basis_general(12, Nup=5, pauli=0, kblock=(m["T"], 5)), xxz_static(12, Delta=0.7), False
    if name == "no_nup":
        return spin_basis_general(9, pauli=0, kblock=(chain_maps(9)["T"], 2)), [
            ["xx", [[0.3, i, (i + 1) % 9] for i in range(9)]], ["xy", [[0.2, i, (i + 1) % 9] for i in range(9)]],
            ["z", [[0.4, i] for i in range(9)]]], False
    if name == "ladder":
        lm = ladder_maps(4, 2)
        bonds = [[0.5, i, (i + 1) % 4 + 4 * (i // 4)] for i in range(8)] + [[0.5, i, i + 4] for i in range(4)]
        return spin_basis_general(8, Nup=4, pauli=0, kxblock=(lm["tx"], 1), zblock=(lm["z"], 1)), [
            ["+-", bonds], ["-+", bonds], ["zz", bonds]], False
    if name == "free":
        return spin_basis_general(11, Nup=4, pauli=0), xxz_static(11, h=np.linspace(-1, 1, 11)), True
    if name == "wide_rows":  # up to 49 elements per row
        return spin_basis_general(14, Nup=7, pauli=0), _all_to_all(14), True
    if name == "words64":
        return spin_basis_general(34, Nup=3, pauli=0, kblock=(chain_maps(34)["T"], 0)), xxz_static(34), True
    if name == "spinless":
        i = np.arange(9)
        bonds = [[-1.0, j, (j + 1) % 9] for j in range(9)]
        return spinless_fermion_basis_general(9, Nf=4, kblock=((i + 1) % 9, 3)), [
            ["+-", bonds], ["-+", [[1.0, a, b] for _, a, b in bonds]], ["nn", [[1.5, a, b] for _, a, b in bonds]]], False
    i = np.arange(6)
    return spinful_fermion_basis_general(6, Nf=(3, 2), kblock=((i + 1) % 6, 1)), hubbard_static(6, U=2.0), False


def _vec(rng, n, nv, dtype):
    shape = (n,) if nv == 1 else (n, nv)
    x = rng.normal(size=shape)
    if np.dtype(dtype).kind == "c":
        x = x + 1j * rng.normal(size=shape)
    return x.astype(dtype)


def _check(y, A, x, a, diag, dtype, y0=None):
    """FP64 sums of at most m elements and one rounding of the result; the
    elements themselves are equal up to the rounding of their factors."""
    xx = x.astype(np.complex128)
    exact = a * (A @ xx)
    mag = abs(a) * (abs(A) @ np.abs(xx))
    if diag is not None:
        d = diag if x.ndim == 1 else diag[:, None]
        exact = exact + d * xx
        mag = mag + np.abs(d * xx)
    if y0 is not None:
        exact, mag = exact + y0, mag + np.abs(y0)
    m = int(np.diff(A.indptr).max())
    bound = (16 * (m + 4) * 2.0 ** -53 + 2 * EPS[np.dtype(dtype)]) * mag + 1e-300
    assert np.all(np.abs(y - exact) <= bound)


@pytest.mark.parametrize("nv", [1, 2, 3, 8, 17, 64, 70])
@pytest.mark.parametrize("name", ["kpz", "momentum", "no_nup", "ladder", "free", "wide_rows", "words64", "spinless",
                                  "spinful"])
def test_packed_product(name, nv):
    from quspin_amd import _lib as L
    from quspin_amd.operators import quantum_LinearOperator
    basis, static, real = _case(name)
    rng = np.random.default_rng(nv)
    off = [t for t in static if set(t[0]) & set("+-xy")]
    for dtype in ((np.float64, np.float32, np.complex128, np.complex64) if real else (np.complex128, np.complex64)):
        Q = quantum_LinearOperator(static, basis=basis, dtype=dtype, **KW)
        op = Q._qsx_operator()
        A = quantum_LinearOperator(off, basis=basis, dtype=np.complex128, **KW)._qsx_operator().to_csr().to_scipy()
        diag = L.to_host(op.diagonal(np.complex128))
        x = _vec(rng, basis.Ns, nv, dtype)
        a = 0.6 - (0.8j if np.dtype(dtype).kind == "c" else 0)
        y = L.empty(x.shape, dtype)
        op.apply(L.to_device(x), y, a=a, a_diag=0.5)
        assert op.config[(np.dtype(dtype), nv)]["schedule"] == "packed"
        _check(L.to_host(y), A, x, a, 0.5 * diag, dtype)
        y0 = _vec(rng, basis.Ns, nv, dtype)
        y = L.to_device(y0)
        op.apply(L.to_device(x), y, a=a, beta=1, a_diag=0.0)
        _check(L.to_host(y), A, x, a, None, dtype, y0)


@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("conjugated", [False, True])
@pytest.mark.parametrize("name", ["momentum", "spinful", "no_nup"])
def test_packed_flags(name, transposed, conjugated):
    """Transposed and conjugated operators have rows of their own."""
    from quspin_amd import _lib as L
    from quspin_amd.operators._devop import MatrixFreeOp
    basis, static, _ = _case(name)
    static = [[op, [[b[0] * (1 + 0.3j)] + list(b[1:]) for b in bonds]] for op, bonds in static
              if set(op) & set("+-xy")]
    rng = np.random.default_rng(3)
    from quspin_amd.operators._make_hamiltonian import _consolidate_static
    ol = basis._compile_oplist(_consolidate_static(static))
    A = MatrixFreeOp(basis, ol, np.complex128).to_csr().to_scipy()
    if transposed:
        A = A.T.tocsr()
    if conjugated:
        A = A.conj()
    op = MatrixFreeOp(basis, ol, np.complex128, transposed=transposed, conjugated=conjugated)
    for nv in (1, 5):
        x = _vec(rng, basis.Ns, nv, np.complex128)
        y = L.empty(x.shape, np.complex128)
        op.apply(L.to_device(x), y)
        assert op.config[(np.dtype(np.complex128), nv)]["schedule"] == "packed"
        _check(L.to_host(y), A, x, 1.0, None, np.complex128)


def _distinct_four_body(L):
    """Every four-site coupling of six strings with a value of its own."""
    from itertools import combinations
    J = 1.0
    static = []
    for opstr in ("xxxx", "xxxz", "xxzz", "zxxx", "xzzx", "zxzx"):
        bonds = []
        for sites in combinations(range(L), 4):
            J += 0.001
            bonds.append([J] + list(sites))
        static.append([opstr, bonds])
    return static


def test_packed_build_stops_when_the_dictionary_is_full():
    """More values (2,970 couplings, 5,445 with signs) than the dictionary has
    slots: the rows stop soon after the 1,023rd value, about a quarter of the
    way through the terms, and the operator is refused."""
    from quspin_amd import _lib as L
    from quspin_amd.basis import spin_basis_general
    from quspin_amd.operators import quantum_LinearOperator
    basis = spin_basis_general(12, pauli=0)
    op = quantum_LinearOperator(_distinct_four_body(12), basis=basis, dtype=np.float64, **KW)._qsx_operator()
    ctx = op._new_ctx(np.dtype(np.float64), 1)
    lib = L.load()
    nwork = lib.qsx_hv_pack_work_bytes(ctx.h)
    nsl = basis.Ns // 64
    off, work = L.empty(nsl + 1, np.int64), L.empty((nwork + 7) // 8, np.int64)
    ent, nl, bits = L._i64(), L._i32(), L._i32()
    rc = lib.qsx_hv_pack_count(ctx.h, L.ptr(off), L.ptr(work), nwork, L.C.byref(ent), L.C.byref(nl), L.C.byref(bits),
                               L.stream_handle())
    assert rc == L.QSX_ERR_UNSUPPORTED
    widths = np.diff(L.to_host(off)) // 64
    assert op.oplist.n_off == 2970 and widths.min() >= 0 and widths.max() <= 1500
    x = _vec(np.random.default_rng(0), basis.Ns, 1, np.float64)
    y = L.empty(x.shape, np.float64)
    op.apply(L.to_device(x), y)
    assert op._pk is None
    _check(L.to_host(y), op.to_csr().to_scipy(), x, 1.0, None, np.float64)


def test_packed_dictionary_overflow_takes_the_general_kernels():
    """More distinct coefficients (1,260) than the form takes (1,023): refused,
    and the product runs as it did."""
    from quspin_amd import _lib as L
    from quspin_amd.basis import spin_basis_general
    from quspin_amd.operators import quantum_LinearOperator
    basis = spin_basis_general(10, pauli=0)
    Q = quantum_LinearOperator(_distinct_four_body(10), basis=basis, dtype=np.float64, **KW)
    op = Q._qsx_operator()
    x = _vec(np.random.default_rng(0), basis.Ns, 1, np.float64)
    y = L.empty(x.shape, np.float64)
    op.apply(L.to_device(x), y)
    assert op.config[(np.dtype(np.float64), 1)]["schedule"] != "packed" and op._pk is None
    _check(L.to_host(y), op.to_csr().to_scipy(), x, 1.0, None, np.float64)


def test_packed_limit_and_replaced_diagonal(monkeypatch):
    """Rows above the byte limit are not kept; a replaced diagonal and a later
    operator on the same basis give their own products."""
    from quspin_amd import _lib as L, tuning
    from quspin_amd.operators import quantum_LinearOperator
    basis, static, _ = _case("kpz")
    x = _vec(np.random.default_rng(1), basis.Ns, 1, np.float64)
    xd = L.to_device(x)
    off = [t for t in static if set(t[0]) & set("+-")]
    A = quantum_LinearOperator(off, basis=basis, dtype=np.complex128, **KW)._qsx_operator().to_csr().to_scipy()
    Q = quantum_LinearOperator(static, basis=basis, dtype=np.float64, **KW)
    before = L.to_host(Q._qsx_operator().diagonal(np.complex128))
    _check(L.to_host(Q.dot(xd)), A, x, 1.0, before, np.float64)
    d = np.linspace(0, 1, basis.Ns)
    Q.set_diagonal(d)
    _check(L.to_host(Q.dot(xd)), A, x, 1.0, d, np.float64)
    Q2 = quantum_LinearOperator([[op, [[3 * b[0]] + b[1:] for b in bonds]] for op, bonds in static], basis=basis,
                                dtype=np.float64, **KW)
    _check(L.to_host(Q2.dot(xd)), A, x, 3.0, 3 * before, np.float64)
    monkeypatch.setattr(tuning, "packed_limit", lambda op: 4 * op.Ns)
    Q3 = quantum_LinearOperator(static, basis=basis, dtype=np.float64, **KW)
    for _ in range(tuning.PACK_AFTER + 2):
        _check(L.to_host(Q3.dot(xd)), A, x, 1.0, before, np.float64)
    assert Q3._qsx_operator()._packed_rows.tried and Q3._qsx_operator()._pk is None


@pytest.mark.parametrize("nv", [1, 4, 9])
@pytest.mark.parametrize("name", ["momentum", "spinful", "free"])
def test_packed_taylor_terms(name, nv):
    """The Taylor loop whose terms run in the packed product."""
    import scipy.linalg
    from quspin_amd import _lib as L
    from quspin_amd.operators import quantum_LinearOperator
    from quspin_amd.tools.evolution import expm_multiply_parallel
    basis, static, _ = _case(name)
    Q = quantum_LinearOperator(static, basis=basis, dtype=np.complex128, **KW)
    E = expm_multiply_parallel(Q, a=-0.9j)
    x = _vec(np.random.default_rng(nv), basis.Ns, nv, np.complex128)
    got = L.to_host(E.dot(L.to_device(x)))
    assert Q._qsx_operator().config[(np.dtype(np.complex128), nv)]["schedule"] == "packed"
    A = Q._qsx_operator().to_csr().to_scipy().toarray()
    exact = scipy.linalg.expm(-0.9j * A) @ x
    # unitary, about 30 terms, each rounded once; the largest partial sums are e^|a||A - mu| / 2
    assert np.abs(got - exact).max() <= 1e-12 * np.abs(x).max()


@pytest.mark.parametrize("L_", [19, 20])
def test_packed_elements_kept_or_evaluated_twice(monkeypatch, L_):
    """Either side of the size up to which a build keeps the evaluated
    elements (64 MiB at 24 bytes per row and term: 42 MB, 89 MB) gives the
    product of the general kernel.  Both sum at most 20 products of
    coefficients 0.5 and unit-scale elements in FP64: 2 x 22 roundings."""
    from quspin_amd import _lib as L
    from quspin_amd.basis import spin_basis_general
    from quspin_amd.operators import quantum_LinearOperator
    basis = spin_basis_general(L_, Nup=L_ // 2, pauli=0)
    x = _vec(np.random.default_rng(L_), basis.Ns, 1, np.float64)
    xd = L.to_device(x)
    y = {}
    for sched in ("packed", "rows"):
        monkeypatch.setenv("QSX_LOOKUP", "search")
        monkeypatch.setenv("QSX_SCHEDULE", sched)
        Q = quantum_LinearOperator(xxz_static(L_, Delta=0.7), basis=basis, dtype=np.float64, **KW)
        y[sched] = L.to_host(Q.dot(xd))
        op = Q._qsx_operator()
        assert next(iter(op.config.values()))["schedule"] == sched
        assert (getattr(op, "_pk", None) is not None) == (sched == "packed")
    bound = 44 * 2.0 ** -53 * (0.5 * L_ + 0.25 * L_) * np.abs(x).max()
    assert np.abs(y["packed"] - y["rows"]).max() <= bound

@pytest.mark.parametrize("nv", [1, 3, 8])
@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_packed_non_finite_vector(bad, nv):
    """An element that is not finite reaches the rows that have an element (or
    a diagonal) in its column, and no padding of its own row makes a NaN of an
    infinite one."""
    from quspin_amd import _lib as L
    from quspin_amd.operators import quantum_LinearOperator
    basis, static, _ = _case("free")
    for dtype in (np.float64, np.float32):
        op = quantum_LinearOperator(static, basis=basis, dtype=dtype, **KW)._qsx_operator()
        A = op.to_csr(np.float64).to_scipy()
        # the first row with fewer elements than another of its slice
        off = np.array([(A.indices[A.indptr[i]:A.indptr[i + 1]] != i).sum() for i in range(basis.Ns)])
        r = next(i for i in range(basis.Ns) if off[i] < off[i // 64 * 64:i // 64 * 64 + 64].max() and A[i, i] != 0)
        x = _vec(np.random.default_rng(nv), basis.Ns, nv, dtype)
        x[r] = bad
        y = L.empty(x.shape, dtype)
        op.apply(L.to_device(x), y)
        assert op.config[(np.dtype(dtype), nv)]["schedule"] == "packed"
        y = L.to_host(y)
        hit = np.flatnonzero(A[:, [r]].toarray().ravel())
        want = bad * np.sign(A[:, [r]].toarray()[hit])
        np.testing.assert_array_equal(y[hit].reshape(len(hit), -1), np.broadcast_to(want, (len(hit), nv)))
        rest = np.setdiff1d(np.arange(basis.Ns), hit)
        assert np.isfinite(y[rest]).all()


def _count_builds(monkeypatch):
    from quspin_amd import _lib as L
    lib, calls = L.load(), []
    f = lib.qsx_hv_pack_count
    monkeypatch.setattr(lib, "qsx_hv_pack_count", lambda *a: (calls.append(1), f(*a))[1])
    return calls


def test_packed_rows_shared_by_adjoints_and_copies(monkeypatch):
    """``rmatvec``, ``.H``, ``.T`` and copies evaluate the elements once per
    pair of flags; a replaced diagonal starts anew and leaves copies alone."""
    from quspin_amd import _lib as L
    from quspin_amd.operators import quantum_LinearOperator
    basis, static, _ = _case("momentum")
    calls = _count_builds(monkeypatch)
    Q = quantum_LinearOperator(static, basis=basis, dtype=np.complex128, **KW)
    A = Q._qsx_operator().to_csr().to_scipy()
    x = _vec(np.random.default_rng(8), basis.Ns, 1, np.complex128)
    xd = L.to_device(x)
    for _ in range(20):  # long enough to have built whatever it builds
        _check(L.to_host(Q.dot(xd)), A, x, 1.0, None, np.complex128)
        _check(Q.rmatvec(x), A.conj().T.tocsr(), x, 1.0, None, np.complex128)
        _check(L.to_host(Q.H.dot(xd)), A.conj().T.tocsr(), x, 1.0, None, np.complex128)
        _check(L.to_host(Q.copy().dot(xd)), A, x, 1.0, None, np.complex128)
    assert len(calls) <= 2 and Q._op_for(False, False)._pk is not None
    for _ in range(20):
        Q.T.dot(xd)
    assert len(calls) <= 3
    C = Q.copy()
    Q.set_diagonal(np.ones(basis.Ns))
    _check(L.to_host(C.dot(xd)), A, x, 1.0, None, np.complex128)
    hops = quantum_LinearOperator(static[:2], basis=basis, dtype=np.complex128, **KW)
    D = hops._qsx_operator().to_csr().to_scipy() + sp.identity(basis.Ns)
    _check(L.to_host(Q.dot(xd)), D.tocsr(), x, 1.0, None, np.complex128)


def test_packed_norm_estimates_share_the_adjoint(monkeypatch):
    """The partition of a Taylor loop estimates 1-norms of several powers: one
    build for the operator and one for its adjoint, also for a second ``a``."""
    from quspin_amd.operators import quantum_LinearOperator
    from quspin_amd.tools.evolution import expm_multiply_parallel
    basis, static, _ = _case("momentum")
    calls = _count_builds(monkeypatch)
    Q = quantum_LinearOperator(static, basis=basis, dtype=np.complex128, **KW)
    E = expm_multiply_parallel(Q, a=-20.0j)
    E.set_a(-35.0j)
    expm_multiply_parallel(Q, a=-30.0j)
    assert 1 <= len(calls) <= 2


def test_packed_rows_of_one_basis_share_a_limit(monkeypatch):
    """Operators beyond the basis' limit take the other forms; freed rows make room."""
    import gc
    from quspin_amd import _lib as L, tuning
    from quspin_amd.operators import quantum_LinearOperator
    basis, static, _ = _case("momentum")
    x = _vec(np.random.default_rng(9), basis.Ns, 1, np.complex128)

    def made(scale):
        op = quantum_LinearOperator([[o, [[scale * b[0]] + b[1:] for b in bb]] for o, bb in static], basis=basis,
                                    dtype=np.complex128, **KW)._qsx_operator()
        y = L.empty(x.shape, np.complex128)
        op.apply(L.to_device(x), y)
        _check(L.to_host(y), op.to_csr().to_scipy(), x, 1.0, None, np.complex128)
        return op
    first = made(1.0)
    one = 4 * int(first._pk[1].numel())
    monkeypatch.setattr(tuning, "PACKED_TOTAL", 2 * one)
    second, third = made(2.0), made(3.0)
    assert second._pk is not None and third._pk is None
    del first
    gc.collect()
    assert made(4.0)._pk is not None


def test_packed_rows_without_memory(monkeypatch):
    """No memory for the build: the product takes another form."""
    import torch
    from quspin_amd import _lib as L
    from quspin_amd.operators import quantum_LinearOperator
    basis, static, _ = _case("momentum")
    op = quantum_LinearOperator(static, basis=basis, dtype=np.complex128, **KW)._qsx_operator()
    x = _vec(np.random.default_rng(10), basis.Ns, 1, np.complex128)
    y = L.empty(x.shape, np.complex128)
    real = L.empty

    def empty(shape, dtype):
        if np.dtype(dtype) == np.int64:
            raise torch.OutOfMemoryError("no memory")
        return real(shape, dtype)
    monkeypatch.setattr(L, "empty", empty)
    op.apply(L.to_device(x), y)
    monkeypatch.undo()
    assert op._pk is None
    _check(L.to_host(y), op.to_csr().to_scipy(), x, 1.0, None, np.complex128)


@pytest.mark.parametrize("nv", [1, 5])
@pytest.mark.parametrize("name", ["free", "momentum"])
def test_rows_are_built_after_single_products(name, nv, monkeypatch):
    """An operator asked for one product at a time makes ``PACK_AFTER`` vectors
    without packed rows (the first one on a symmetry-reduced basis builds them
    at once, the others go through the sector table); every product is the
    operator's, before and after."""
    from quspin_amd import _lib as L, tuning
    from quspin_amd.operators import quantum_LinearOperator
    basis, static, _ = _case(name)
    calls = _count_builds(monkeypatch)
    x = _vec(np.random.default_rng(nv), basis.Ns, nv, np.complex128)
    xd = L.to_device(x)
    for i in range(3):
        Q = quantum_LinearOperator([[o, [[(1 + i) * b[0]] + b[1:] for b in bb]] for o, bb in static], basis=basis,
                                   dtype=np.complex128, **KW)
        A = Q._qsx_operator().to_csr().to_scipy()
        calls.clear()
        first = name == "momentum" and i == 0
        for k in range(20):
            _check(L.to_host(Q.dot(xd)), A, x, 1.0, None, np.complex128)
            assert len(calls) == (1 if first or (k + 1) * nv > tuning.PACK_AFTER else 0)
        assert Q._qsx_operator().config[(np.dtype(np.complex128), nv)]["schedule"] == "packed"
    assert basis.has_lookup_table() == (name == "momentum")


def test_a_captured_product_builds_nothing(monkeypatch):
    """Products of one operator, one of them captured: the capture holds the
    form without rows and replays its product after the rows are built."""
    import torch
    from quspin_amd import _lib as L, tuning
    from quspin_amd.operators import quantum_LinearOperator
    basis, static, _ = _case("free")
    calls = _count_builds(monkeypatch)
    Q = quantum_LinearOperator(static, basis=basis, dtype=np.float64, **KW)
    A = Q._qsx_operator().to_csr().to_scipy()
    x = _vec(np.random.default_rng(3), basis.Ns, 1, np.float64)
    xd = L.to_device(x)
    y = torch.empty_like(xd)
    op = Q._qsx_operator()
    for _ in range(3):
        op.apply(xd, y, products=1)
    monkeypatch.setattr(tuning, "PACK_AFTER", 2)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        op.apply(xd, y, products=1)
    assert not calls and op._pk is None
    for _ in range(3):
        y.zero_()
        graph.replay()
        _check(L.to_host(y), A, x, 1.0, None, np.float64)
        y.zero_()
        op.apply(xd, y, products=1)
        _check(L.to_host(y), A, x, 1.0, None, np.float64)
    assert len(calls) == 1 and op._pk is not None
