"""The one-workgroup Taylor loop and Lanczos recurrence of small operators,
at the edges of their row ranges, against 64-bit host arithmetic."""

import numpy as np
import pytest
import scipy.sparse as sp

from models import chain_maps, xxz_static

pytestmark = pytest.mark.gpu

EPS = {np.dtype(np.float32): 2.0 ** -24, np.dtype(np.complex64): 2.0 ** -24,
       np.dtype(np.float64): 2.0 ** -53, np.dtype(np.complex128): 2.0 ** -53}
KW = dict(check_symm=False, check_herm=False, check_pcon=False)


def _hermitian(rng, n, cplx, bands=(0, 1, 7)):
    """Banded Hermitian matrix with some empty rows and norm of order one."""
    A = sp.lil_matrix((n, n), dtype=np.complex128 if cplx else np.float64)
    for b in bands:
        for i in range(n - b):
            if rng.random() < 0.8:
                z = rng.normal() * 0.3 + (1j * rng.normal() * 0.3 if cplx and b else 0)
                A[i, i + b] = z
                A[i + b, i] = np.conj(z)
    return A.tocsr()


def _vec(rng, n, dtype):
    x = rng.normal(size=n)
    if np.dtype(dtype).kind == "c":
        x = x + 1j * rng.normal(size=n)
    return (x / np.linalg.norm(x)).astype(dtype)


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1023, 1024, 1025, 2048, 2049, 4095, 4096, 4097])
@pytest.mark.parametrize("mdt,vdt,a", [(np.float64, np.complex128, -3.0j), (np.complex128, np.complex128, -0.4j),
                                       (np.float64, np.float64, -0.7), (np.float32, np.complex64, -1.1j),
                                       (np.complex64, np.complex64, -0.3j), (np.float32, np.float32, -0.5)])
def test_small_expm(n, mdt, vdt, a):
    from scipy.sparse.linalg import expm_multiply
    from quspin_amd import _lib as L
    from quspin_amd.operators._devop import DeviceCSR
    from quspin_amd.tools.evolution import expm_multiply_parallel
    rng = np.random.default_rng(n)
    A = _hermitian(rng, n, np.dtype(mdt).kind == "c").astype(mdt)
    E = expm_multiply_parallel(DeviceCSR.from_scipy(A, mdt), a=a, dtype=vdt)
    x = _vec(rng, n, vdt)
    got = L.to_host(E.dot(L.to_device(x)))
    wide = A.astype(np.complex128 if np.iscomplexobj(A) else np.float64)
    exact = expm_multiply(a * wide, x.astype(np.complex128))
    # each stage: the truncation tolerance and one rounding per term of partial sums of at most e^|a A|
    radius = abs(a) * float(abs(wide).sum(axis=0).max()) / E.partition[1]
    bound = E.partition[1] * (E.partition[0] + 2) * EPS[np.dtype(vdt)] * min(np.exp(radius), 1e4)
    assert np.linalg.norm(got - exact) <= bound * max(np.linalg.norm(exact), np.linalg.norm(x))


@pytest.mark.parametrize("n,m", [(2, 1), (40, 9), (64, 20), (65, 20), (1024, 12), (1025, 12), (2049, 12), (4096, 12),
                                 (4097, 12)])
@pytest.mark.parametrize("dtype", [np.float64, np.complex128, np.complex64])
def test_small_lanczos(n, m, dtype):
    from quspin_amd import _lib as L
    from quspin_amd.operators._devop import DeviceCSR
    from quspin_amd.tools.lanczos import _host_loop, lanczos_full, lanczos_iter
    rng = np.random.default_rng(n + m)
    A = _hermitian(rng, n, np.dtype(dtype).kind == "c").astype(dtype)
    x = 2.5 * _vec(rng, n, dtype)  # not normalised
    E, V, Q = lanczos_full(DeviceCSR.from_scipy(A, dtype), L.to_device(x), m)
    wide = A.astype(np.complex128)
    a, b, mm, Qh = _host_loop(wide, x.astype(np.complex128), m, np.complex128, 0.0)
    Eh = np.linalg.eigvalsh(np.diag(a) + np.diag(b[:-1], 1) + np.diag(b[:-1], -1))
    # the first vectors to rounding grown by at most a factor of 8 per step here
    tol = 64 * EPS[np.dtype(dtype)]
    k = min(m, 5)
    assert np.abs(L.to_host(Q)[:k] - Qh[:k]).max() <= tol * 8 ** k
    assert np.abs(E - Eh).max() <= 200 * EPS[np.dtype(dtype)] * max(1.0, np.abs(Eh).max()) * m
    E2, V2 = lanczos_iter(DeviceCSR.from_scipy(A, dtype), L.to_device(x), m, return_vec_iter=False)
    assert np.array_equal(E, E2)
    out = L.empty((m, 2 * n), dtype)[:, :n]  # rows apart
    E3, _, Q3 = lanczos_full(DeviceCSR.from_scipy(A, dtype), L.to_device(x), m, out=out)
    assert np.array_equal(E, E3) and np.array_equal(L.to_host(Q3), L.to_host(Q))


@pytest.mark.parametrize("dtype", [np.float64, np.float32, np.complex128])
def test_small_packed_rows_match_the_large_path(dtype, monkeypatch):
    """A matrix-free sector: the one-launch forms against the launch-per-step
    forms of the same operator (a forced schedule has no packed rows)."""
    from quspin_amd import _lib as L
    from quspin_amd.basis import spin_basis_general
    from quspin_amd.operators import quantum_LinearOperator
    from quspin_amd.tools.evolution import expm_multiply_parallel
    from quspin_amd.tools.lanczos import lanczos_full
    m = chain_maps(12)
    basis = spin_basis_general(12, Nup=6, pauli=0, kblock=(m["T"], 0 if np.dtype(dtype).kind == "f" else 5))
    x = _vec(np.random.default_rng(2), basis.Ns, dtype)
    got = []
    for forced in (None, "rows"):
        if forced:
            monkeypatch.setenv("QSX_SCHEDULE", forced)
        Q = quantum_LinearOperator(xxz_static(12, Delta=0.8), basis=basis, dtype=dtype, **KW)
        F = expm_multiply_parallel(Q, a=-0.6, dtype=dtype).dot(L.to_device(x))
        E, V, _ = lanczos_full(Q, L.to_device(x), 20)
        sched = Q._qsx_operator().config[(np.dtype(dtype), 1)]["schedule"]
        assert (sched == "packed") == (forced is None)
        got.append((L.to_host(F), E))
    assert np.abs(got[0][0] - got[1][0]).max() <= 200 * EPS[np.dtype(dtype)]
    assert np.abs(got[0][1] - got[1][1]).max() <= 4000 * EPS[np.dtype(dtype)]


def _small_codes(monkeypatch):
    """Return codes of the one-launch recurrence from here on."""
    from quspin_amd import _lib as L
    lib, codes = L.load(), []
    f = lib.qsx_lanczos_small

    def call(*args):
        codes.append(f(*args))
        return codes[-1]
    monkeypatch.setattr(lib, "qsx_lanczos_small", call)
    return codes


@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.complex64, np.complex128])
@pytest.mark.parametrize("L_,Nup", [(13, 6), (28, 3)])
def test_small_lanczos_packed_rows_per_thread(dtype, L_, Nup, monkeypatch):
    """One launch on packed rows with two (1,716) and four (3,276) rows per
    thread; complex128 takes 69 KB of LDS at the larger.  Against the host
    recurrence in 64 bits."""
    from quspin_amd import _lib as L
    from quspin_amd.basis import spin_basis_general
    from quspin_amd.operators import quantum_LinearOperator
    from quspin_amd.tools.lanczos import _host_loop, lanczos_full
    basis = spin_basis_general(L_, Nup=Nup, pauli=0)
    Q = quantum_LinearOperator(xxz_static(L_, h=np.linspace(-1, 1, L_)), basis=basis, dtype=dtype, **KW)
    A = Q._qsx_operator().to_csr(np.complex128).to_scipy()
    x = (1.7 * _vec(np.random.default_rng(L_), basis.Ns, dtype)).astype(dtype)
    codes, m = _small_codes(monkeypatch), 12
    E, V, K = lanczos_full(Q, L.to_device(x), m)
    assert codes == [L.QSX_OK]
    a, b, _, Kh = _host_loop(A, x.astype(np.complex128), m, np.complex128, 0.0)
    Eh = np.linalg.eigvalsh(np.diag(a) + np.diag(b[:-1], 1) + np.diag(b[:-1], -1))
    # rounding of a step grows by at most a factor of 8 per step here
    assert np.abs(L.to_host(K)[:5] - Kh[:5]).max() <= 64 * EPS[np.dtype(dtype)] * 8 ** 5
    assert np.abs(E - Eh).max() <= 200 * EPS[np.dtype(dtype)] * np.abs(Eh).max() * m


@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.complex64, np.complex128])
def test_small_expm_packed_two_rows_per_thread(dtype):
    """The Taylor loop in one workgroup on packed rows, 1,716 of them."""
    from scipy.sparse.linalg import expm_multiply
    from quspin_amd import _lib as L
    from quspin_amd.basis import spin_basis_general
    from quspin_amd.operators import quantum_LinearOperator
    from quspin_amd.tools.evolution import expm_multiply_parallel
    basis = spin_basis_general(13, Nup=6, pauli=0)
    Q = quantum_LinearOperator(xxz_static(13, h=np.linspace(-1, 1, 13)), basis=basis, dtype=dtype, **KW)
    A = Q._qsx_operator().to_csr(np.complex128).to_scipy()
    x = _vec(np.random.default_rng(13), basis.Ns, dtype)
    a = -0.4j if np.dtype(dtype).kind == "c" else -0.4
    E = expm_multiply_parallel(Q, a=a, dtype=dtype)
    got = L.to_host(E.dot(L.to_device(x)))
    assert Q._qsx_operator().config[(np.dtype(dtype), 1)]["schedule"] == "packed"
    exact = expm_multiply(a * A, x.astype(np.complex128))
    # one rounding per term of partial sums of at most e^|a A|, |a A| <= 0.4 x 11
    terms = E.partition[0] * E.partition[1]
    assert np.linalg.norm(got - exact) <= (terms + 2) * EPS[np.dtype(dtype)] * np.exp(4.4)


@pytest.mark.parametrize("dtype,small", [(np.float64, True), (np.float32, True), (np.complex128, False),
                                         (np.complex64, False)])
def test_small_lanczos_limit_by_type(dtype, small, monkeypatch):
    """3,876 rows of at most 8 elements (30,592 in slices): one launch in real
    types, two per step in complex ones, and the same tridiagonal matrix."""
    from quspin_amd import _lib as L
    from quspin_amd.basis import spin_basis_general
    from quspin_amd.operators import quantum_LinearOperator
    from quspin_amd.tools.lanczos import _host_loop, lanczos_iter
    basis = spin_basis_general(19, Nup=4, pauli=0)
    Q = quantum_LinearOperator(xxz_static(19), basis=basis, dtype=dtype, **KW)
    A = Q._qsx_operator().to_csr(np.complex128).to_scipy()
    x = _vec(np.random.default_rng(5), basis.Ns, dtype)
    codes, m = _small_codes(monkeypatch), 10
    E, V = lanczos_iter(Q, L.to_device(x), m, return_vec_iter=False)
    assert codes == [L.QSX_OK if small else L.QSX_ERR_UNSUPPORTED]
    a, b, _, _ = _host_loop(A, x.astype(np.complex128), m, np.complex128, 0.0)
    Eh = np.linalg.eigvalsh(np.diag(a) + np.diag(b[:-1], 1) + np.diag(b[:-1], -1))
    assert np.abs(E - Eh).max() <= 400 * EPS[np.dtype(dtype)] * np.abs(Eh).max() * m


@pytest.mark.parametrize("dtype", [np.float64, np.complex128, np.complex64])
@pytest.mark.parametrize("blocks,Nup,L_", [(None, 8, 16), ("k", 9, 19), (None, 6, 15), (None, 11, 22)])
def test_packed_lanczos_two_launches_per_step(dtype, blocks, Nup, L_, monkeypatch):
    """Sectors above the one-launch sizes (4,862 to 705,432 states; more rows
    than one round of the capped grid at the largest): a and b, the vectors
    and lanczos_iter against the host recurrence in 64 bits, and a start
    vector that is a row of ``out``."""
    from quspin_amd import _lib as L
    from quspin_amd.basis import spin_basis_general
    from quspin_amd.operators import quantum_LinearOperator
    from quspin_amd.tools.lanczos import _host_loop, lanczos_full, lanczos_iter
    kw = {"kblock": (chain_maps(L_)["T"], 3)} if blocks else {}
    if blocks and np.dtype(dtype).kind != "c":
        pytest.skip("complex characters")
    basis = spin_basis_general(L_, Nup=Nup, pauli=0, **kw)
    h = None if blocks else np.linspace(-1, 1, L_)
    monkeypatch.setattr("quspin_amd.tuning.time_candidates",
                        lambda op, ctx, vdt, nvec, reps=5: {"lookup": "search", "schedule": "packed"})
    monkeypatch.setenv("QSX_TUNE_CACHE", "/nonexistent/tune.json")
    monkeypatch.setattr("quspin_amd.tuning._mem", {})
    Q = quantum_LinearOperator(xxz_static(L_, h=h), basis=basis, dtype=dtype, **KW)
    rng = np.random.default_rng(4)
    m = 12
    A = Q._qsx_operator().to_csr(np.complex128).to_scipy()
    codes = _small_codes(monkeypatch)
    for scale in (1.0, 3.0):
        x = (scale * _vec(rng, basis.Ns, dtype)).astype(dtype)
        xd = L.to_device(x)
        E, V, K = lanczos_full(Q, xd, m)
        assert Q._qsx_operator().config[(np.dtype(dtype), 1)]["schedule"] == "packed"
        assert np.array_equal(L.to_host(xd), x)
        a, b, _, Kh = _host_loop(A, x.astype(np.complex128), m, np.complex128, 0.0)
        Eh = np.linalg.eigvalsh(np.diag(a) + np.diag(b[:-1], 1) + np.diag(b[:-1], -1))
        # rounding of a step grows by at most a factor of 8 per step here; two more roundings of q and H q
        assert np.abs(L.to_host(K)[:5] - Kh[:5]).max() <= 128 * EPS[np.dtype(dtype)] * 8 ** 5
        assert np.abs(E - Eh).max() <= 400 * EPS[np.dtype(dtype)] * np.abs(Eh).max() * m
        E2, _ = lanczos_iter(Q, xd, m, return_vec_iter=False)
        assert np.array_equal(E, E2)
        out = L.empty((m, basis.Ns), dtype)
        out[0].copy_(xd)
        E3, _, K3 = lanczos_full(Q, out[0], m, out=out)
        assert np.array_equal(E, E3) and np.array_equal(L.to_host(K3), L.to_host(K))
    assert L.QSX_OK not in codes


def test_lanczos_memory_of_the_captured_sequence():
    """An operator with neither form holds the result and the workspace's
    vectors, not a third basis."""
    import torch
    from quspin_amd import _lib as L
    from quspin_amd.operators._devop import DeviceCSR
    from quspin_amd.tools.lanczos import lanczos_full
    n, m = 200_000, 40
    d = sp.diags([np.linspace(-1, 1, n), np.full(n - 1, 0.5), np.full(n - 1, 0.5)], [0, 1, -1]).tocsr()
    A = DeviceCSR.from_scipy(d, np.float64)
    x = L.to_device(_vec(np.random.default_rng(0), n, np.float64))
    torch.cuda.empty_cache()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    lanczos_full(A, x, m)
    # two bases of m vectors and a few vectors
    assert torch.cuda.max_memory_allocated() - before <= (2 * m + 8) * n * 8


@pytest.mark.parametrize("n,k,small", [(200, 100, False), (500, 48, False), (500, 14, True), (64, 32, True),
                                       (1900, 20, False)])
@pytest.mark.parametrize("dtype", [np.float64, np.complex64])
def test_small_csr_by_row_length(n, k, small, dtype, monkeypatch):
    """Assembled matrices with long rows keep a launch per term and step; both
    sides of the rule give the exponential and the recurrence."""
    from scipy.sparse.linalg import expm_multiply
    from quspin_amd import _lib as L
    from quspin_amd.operators._devop import DeviceCSR
    from quspin_amd.tools.evolution import expm_multiply_parallel
    from quspin_amd.tools.lanczos import _host_loop, lanczos_full
    rng = np.random.default_rng(n)
    offs = np.unique(np.concatenate([[0], rng.permutation(n - 1)[:k // 2] + 1]))
    A = sum((sp.diags([np.full(n - d, 0.5 / k)], [d], shape=(n, n)) for d in offs), sp.csr_matrix((n, n)))
    # circulant bands: every row has about k entries
    A = (A + sum((sp.diags([np.full(d, 0.5 / k)], [d - n], shape=(n, n)) for d in offs if d), sp.csr_matrix((n, n))))
    A = (A + A.T).tocsr().astype(np.float32 if dtype == np.complex64 else np.float64)
    D = DeviceCSR.from_scipy(A)
    x = _vec(rng, n, dtype)
    codes, m = _small_codes(monkeypatch), 10
    E, V, K = lanczos_full(D, L.to_device(x), m)
    assert codes == [L.QSX_OK if small else L.QSX_ERR_UNSUPPORTED]
    a, b, _, Kh = _host_loop(A.astype(np.complex128), x.astype(np.complex128), m, np.complex128, 0.0)
    Eh = np.linalg.eigvalsh(np.diag(a) + np.diag(b[:-1], 1) + np.diag(b[:-1], -1))
    assert np.abs(E - Eh).max() <= 400 * EPS[np.dtype(dtype)] * max(1.0, np.abs(Eh).max()) * m
    got = L.to_host(expm_multiply_parallel(D, a=-1.0, dtype=dtype).dot(L.to_device(x)))
    exact = expm_multiply(-A.astype(np.float64), x.astype(np.complex128))
    # |A| <= 1.1: partial sums of at most e^1.1, one rounding per term
    assert np.abs(got - exact).max() <= 40 * EPS[np.dtype(dtype)] * np.exp(1.1) * np.abs(x).max()
