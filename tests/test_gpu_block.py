"""Products with several vectors at once: the assembled matrix and the
matrix-free operator against the same product in 64-bit host arithmetic."""

import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu

EPS = {np.dtype(np.float32): 2.0 ** -24, np.dtype(np.complex64): 2.0 ** -24,
       np.dtype(np.float64): 2.0 ** -53, np.dtype(np.complex128): 2.0 ** -53}


def _random_csr(rng, n, lengths, cplx):
    rows = np.repeat(np.arange(n), lengths)
    cols = np.concatenate([rng.choice(n, size=m, replace=False) for m in lengths]) if rows.size else rows
    vals = rng.normal(size=rows.size)
    if cplx:
        vals = vals + 1j * rng.normal(size=rows.size)
    return sp.csr_matrix((vals, (rows, cols)), shape=(n, n))


def _vectors(rng, n, nv, dtype):
    x = rng.normal(size=(n, nv))
    if np.dtype(dtype).kind == "c":
        x = x + 1j * rng.normal(size=(n, nv))
    return x.astype(dtype)


def _bound(A, x, dtype):
    """|computed - exact| <= (entries + 4) eps_64 |A| |x| from the FP64 sums,
    plus one rounding of the stored result."""
    m = int(np.diff(A.indptr).max()) if A.nnz else 0
    mag = abs(A) @ np.abs(x.astype(np.complex128))
    return 4 * (m + 4) * 2.0 ** -53 * mag + 2 * EPS[np.dtype(dtype)] * mag


@pytest.mark.parametrize("mdt,vdt", [(np.float32, np.float32), (np.float64, np.float64), (np.float32, np.complex64),
                                     (np.complex64, np.complex64), (np.float64, np.complex128),
                                     (np.complex128, np.complex128)])
@pytest.mark.parametrize("n,nv", [(1, 2), (31, 3), (129, 2), (257, 8), (300, 12), (64, 33), (70, 64), (65, 130)])
def test_csr_block_product(mdt, vdt, n, nv):
    from quspin_amd import _lib as L
    from quspin_amd.operators._devop import DeviceCSR
    rng = np.random.default_rng(n * 1000 + nv)
    # empty rows, short rows and one full row
    lengths = rng.integers(0, min(n, 20) + 1, size=n)
    lengths[rng.integers(n)] = n
    A = _random_csr(rng, n, lengths, np.dtype(mdt).kind == "c").astype(mdt)
    A.sort_indices()
    D = DeviceCSR.from_scipy(A, mdt)
    x = _vectors(rng, n, nv, vdt)
    y0 = _vectors(rng, n, nv, vdt)
    a = 0.75 - (0.5j if np.dtype(vdt).kind == "c" else 0)
    exact = a * (A.astype(np.complex128) @ x.astype(np.complex128))
    bound = abs(a) * 4 * _bound(A, x, vdt) + 2 * EPS[np.dtype(vdt)] * np.abs(y0)
    xd, yd = L.to_device(x), L.empty((n, nv), vdt)
    D.apply(xd, yd, a=a)
    assert np.all(np.abs(L.to_host(yd) - exact) <= bound)
    yd = L.to_device(y0)
    D.apply(xd, yd, a=a, beta=1)
    assert np.all(np.abs(L.to_host(yd) - exact - y0) <= bound)


@pytest.mark.parametrize("vdt", [np.float32, np.float64, np.complex64, np.complex128])
@pytest.mark.parametrize("n,k,nv", [(30011, 10, 2), (30011, 10, 3), (60000, 24, 2), (1000, 200, 2), (1000, 200, 8),
                                    (1000, 200, 64), (30000, 60, 3), (30000, 60, 5)])
def test_csr_block_product_either_side_of_the_rule(vdt, n, k, nv):
    """Few vectors on short rows of a large matrix (a block's entries in one
    staged round and in three), and few and many vectors on long rows."""
    from quspin_amd import _lib as L
    from quspin_amd.operators._devop import DeviceCSR
    rng = np.random.default_rng(n + nv)
    mdt = np.float32 if vdt in (np.float32, np.complex64) else np.float64
    r = np.repeat(np.arange(n), k)
    A = sp.csr_matrix((rng.normal(size=n * k).astype(mdt), (r, rng.integers(0, n, n * k))), shape=(n, n))
    D = DeviceCSR.from_scipy(A, mdt)
    A = D.to_scipy()  # duplicates summed
    x = _vectors(rng, n, nv, vdt)
    y = L.empty((n, nv), vdt)
    D.apply(L.to_device(x), y)
    exact = A.astype(np.float64) @ x.astype(np.complex128)
    assert np.all(np.abs(L.to_host(y) - exact) <= _bound(A, x, vdt))


def test_csr_block_long_rows_and_unaligned_vectors():
    """Rows longer than one staged round, and vectors off the 16-byte boundary."""
    from quspin_amd import _lib as L
    from quspin_amd.operators._devop import DeviceCSR
    rng = np.random.default_rng(5)
    n, nv = 2600, 6
    lengths = rng.integers(0, 4, size=n)
    lengths[[3, 4, 1000, n - 1]] = [1024, 1025, 2600, 2049]
    A = _random_csr(rng, n, lengths, False)
    A.sort_indices()
    D = DeviceCSR.from_scipy(A, np.float64)
    x = _vectors(rng, n, nv, np.float64)
    buf = L.empty(n * nv + 1, np.float64)
    for off in (0, 1):
        xd = buf[off:off + n * nv].view(n, nv)
        xd.copy_(L.to_device(x))
        yd = L.empty((n, nv), np.float64)
        D.apply(xd, yd)
        assert np.all(np.abs(L.to_host(yd) - A @ x) <= _bound(A, x, np.float64))


@pytest.mark.parametrize("nv", [2, 5, 16])
@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
def test_expm_block_equals_single_columns(nv, dtype):
    """The Taylor loop on a block equals the loop on each column to rounding
    (the block's truncation test takes row sums, so it may run longer)."""
    from models import xxz_static
    from quspin_amd import _lib as L
    from quspin_amd.basis import spin_basis_general
    from quspin_amd.operators import hamiltonian
    from quspin_amd.tools.evolution import expm_multiply_parallel
    size = 9
    rng = np.random.default_rng(nv)
    B = spin_basis_general(size, Nup=4, pauli=0)
    real = np.float32 if np.dtype(dtype) == np.complex64 else np.float64
    H = hamiltonian(xxz_static(size, h=rng.uniform(-1, 1, size)), [], basis=B, dtype=real, check_symm=False,
                    check_herm=False, check_pcon=False)
    E = expm_multiply_parallel(H, a=-0.7j, dtype=dtype)
    X = _vectors(rng, B.Ns, nv, dtype)
    got = L.to_host(E.dot(L.to_device(X)))
    import scipy.linalg
    exact = scipy.linalg.expm(-0.7j * H.toarray().astype(np.float64)) @ X.astype(np.complex128)
    # the loop's truncation tolerance and one rounding per term, with a margin
    tol = 40 * EPS[np.dtype(dtype)] * 2
    assert np.abs(got - exact).max() <= tol * np.abs(X).max() * 4


@pytest.mark.parametrize("nv", [1, 2, 8, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
def test_sector_batch_long_rows(nv, dtype):
    """Few rows of more than 40 entries (53 on average): the forms that the
    choice by row length takes, products and a Taylor loop."""
    from models import chain_maps
    from quspin_amd import _lib as L
    from quspin_amd.basis import spin_basis_general
    from quspin_amd.operators import quantum_LinearOperator
    from quspin_amd.operators._devop import SectorBatch
    from quspin_amd.tools.evolution import expm_multiply_sectors
    size = 14
    bonds = [[0.5 / d, i, (i + d) % size] for d in range(1, 8) for i in range(size)]
    static = [["+-", bonds], ["-+", bonds], ["zz", bonds]]
    kw = dict(check_symm=False, check_herm=False, check_pcon=False)
    ops = [quantum_LinearOperator(static, basis=spin_basis_general(size, Nup=7, pauli=0,
                                                                   kblock=(chain_maps(size)["T"], k)), dtype=dtype,
                                  **kw) for k in (0, 5)]
    mf = [op._qsx_operator() for op in ops]
    mats = [op.to_csr(dtype).to_scipy() for op in mf]
    assert sum(A.nnz for A in mats) > 40 * sum(A.shape[0] for A in mats)
    rng = np.random.default_rng(nv)
    x = [_vectors(rng, op.Ns, nv, dtype) for op in ops]
    batch = SectorBatch(mf, dtype, nv, form="csr", chunk_rows=16)
    Y = batch.empty()
    batch.apply(batch.stack(x), Y)
    for y, A, xs in zip(batch.unstack(Y), mats, x):
        exact = A.astype(np.complex128) @ xs.astype(np.complex128)
        assert np.all(np.abs(L.to_host(y) - exact) <= _bound(A, xs, dtype))
    from scipy.sparse.linalg import expm_multiply
    E = expm_multiply_sectors(ops, a=-0.2j, dtype=dtype, nvec=nv, form="csr", chunk_rows=16)
    at = 0
    F = L.to_host(E.dot(x))
    for A, xs in zip(mats, x):
        exact = expm_multiply(-0.2j * A.astype(np.complex128), xs.astype(np.complex128))
        assert np.abs(F[at:at + len(xs)] - exact).max() <= 100 * EPS[np.dtype(dtype)] * np.abs(xs).max() * 4
        at += len(xs)


@pytest.mark.parametrize("nv", [1, 2, 3, 8, 9, 16, 17, 31, 32, 33, 34, 63, 64, 70])
@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
def test_sector_batch_csr_rows_side_by_side(nv, dtype):
    """The CSR form of a sector batch at the edges of its column groups:
    products against each sector's own matrix, and a Taylor step against the
    per-sector path.  The long-range couplings give passes of more staged
    entries than one round holds."""
    from models import chain_maps
    from quspin_amd import _lib as L
    from quspin_amd.basis import spin_basis_general
    from quspin_amd.operators import quantum_LinearOperator
    from quspin_amd.operators._devop import SectorBatch
    from quspin_amd.tools.evolution import expm_multiply_parallel, expm_multiply_sectors
    size = 10
    pairs = [[1.0 / min((j - i) % size, (i - j) % size), i, j] for i in range(size) for j in range(i + 1, size)]
    half = [[0.5 * J, i, j] for J, i, j in pairs]
    static = [["+-", half], ["-+", half], ["zz", pairs]]
    kw = dict(check_symm=False, check_herm=False, check_pcon=False)
    ops = [quantum_LinearOperator(static, basis=spin_basis_general(size, Nup=4 + (k % 2), pauli=0,
                                                                   kblock=(chain_maps(size)["T"], k)), dtype=dtype,
                                  **kw) for k in (0, 3, 7)]
    mf = [op._qsx_operator() for op in ops]
    rng = np.random.default_rng(nv)
    for chunk in (1, 5, 16):
        batch = SectorBatch(mf, dtype, nv, form="csr", chunk_rows=chunk)
        x = [_vectors(rng, op.Ns, nv, dtype) for op in ops]
        X = batch.stack(x)
        Y = batch.empty()
        batch.apply(X, Y, a=0.5 - 0.25j)
        y0 = L.to_host(Y).copy()
        batch.apply(X, Y, a=0.5 - 0.25j, beta=1)
        y1 = L.to_host(Y)
        at = 0
        for op, xs in zip(mf, x):
            A = op.to_csr(dtype).to_scipy()
            exact = (0.5 - 0.25j) * (A.astype(np.complex128) @ xs.astype(np.complex128))
            rows = slice(at, at + op.Ns)
            bound = _bound(A, xs, dtype)
            assert np.all(np.abs(y0[rows] - exact) <= bound)
            assert np.all(np.abs(y1[rows] - 2 * exact) <= 4 * bound)
            at += op.Ns
    if nv > 64:
        return
    E = expm_multiply_sectors(ops, a=-0.4j, dtype=dtype, nvec=nv, form="csr", chunk_rows=5)
    x = [_vectors(rng, op.Ns, nv, dtype) for op in ops]
    F = L.to_host(E.dot(x))
    at = 0
    for op, xs in zip(ops, x):
        one = L.to_host(expm_multiply_parallel(op, a=-0.4j, dtype=dtype).dot(L.to_device(xs)))
        assert np.abs(F[at:at + op.Ns] - one.reshape(F[at:at + op.Ns].shape)).max() <= \
            100 * EPS[np.dtype(dtype)] * np.abs(xs).max() * 4
        at += op.Ns


@pytest.mark.parametrize("nv", [1, 2])
@pytest.mark.parametrize("blocks", [448, 449, 8192])
def test_expm_norms_by_grid(blocks, nv):
    """Taylor loops either side of the number of blocks up to which the norms
    go straight into their slots, and on a large grid: the truncation that the
    norms decide gives the exponential of a tridiagonal matrix.  Error: one
    rounding per term of partial sums of at most e^|a A|, |a A| <= 2."""
    from scipy.sparse.linalg import expm_multiply
    from quspin_amd import _lib as L
    from quspin_amd.operators._devop import DeviceCSR
    from quspin_amd.tools.evolution import expm_multiply_parallel
    n = 128 * blocks  # two lanes per row
    rng = np.random.default_rng(blocks)
    A = sp.diags([rng.uniform(-1, 1, n), np.full(n - 1, 0.5), np.full(n - 1, 0.5)], [0, 1, -1]).tocsr()
    E = expm_multiply_parallel(DeviceCSR.from_scipy(A, np.float64), a=-1.0j)
    x = rng.normal(size=(n,) if nv == 1 else (n, nv)) + 0j
    got = L.to_host(E.dot(L.to_device(x)))
    exact = expm_multiply(-1.0j * A, x, traceA=-1.0j * A.diagonal().sum())
    assert np.abs(got - exact).max() <= 40 * 2.0 ** -53 * np.exp(2.0) * np.abs(x).max()
