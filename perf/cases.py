"""What programs on this framework spend their time in, as measurable cases.

A case is one of six kinds of work, each through the public entry points:

  hv       ``quantum_LinearOperator.dot``: the matrix-free product of a ground
           state search or a spectral method, one vector or a block of them
  csr      ``hamiltonian.dot``: the product with the assembled matrix
  expm     ``expm_multiply_parallel(...).dot``: one time (or imaginary time)
           step of an evolution, on the assembled matrix or matrix-free
  lanczos  ``lanczos_full`` and ``expm_lanczos``: a Krylov basis from a random
           vector and e^{tau H} v combined from it
  sectors  ``expm_multiply_sectors``: many vectors in every momentum sector
  driven   ``DrivenEvolution.run``: steps of a driven Hubbard chain

on the chains the tests and ``bench.py`` use: the XXZ chain with random fields
in one magnetisation sector (``xxz``), the Heisenberg chain with translation,
parity and spin inversion (``heis``) or in one momentum sector (``mom``), and
the spinful Hubbard chain without (``hubbard``) or with (``hubbard_k``)
translation.  Sizes go from sectors of a few dozen states, where a call is all
latency, to the 40 million states of the L = 28 chain.
"""

import math

import numpy as np
import torch

from quspin_amd.basis import spin_basis_general, spinful_fermion_basis_general
from quspin_amd.operators import hamiltonian, quantum_LinearOperator
from quspin_amd.tools.evolution import expm_multiply_parallel, expm_multiply_sectors
from quspin_amd.tools.lanczos import expm_lanczos, lanczos_full
from quspin_amd.tools.learned_step import DrivenEvolution

NO_CHECKS = dict(check_symm=False, check_herm=False, check_pcon=False)
COMPLEX = {"float32": "complex64", "float64": "complex128"}


def listed():
    return [
        # a product on a small chain, as in a loop over parameters or time: all call latency
        {"name": "hv_xxz_12", "kind": "hv", "model": "xxz", "L": 12, "k": 0, "dtype": "complex128", "nvec": 1},
        # the product of a ground-state search in the fully symmetric sector (bench.py's headline size)
        {"name": "hv_heis_28", "kind": "hv", "model": "heis", "L": 28, "k": 0, "dtype": "float64", "nvec": 1},
        # the largest single sector without symmetries that bench.py evolves, in single precision
        {"name": "hv_xxz_28", "kind": "hv", "model": "xxz", "L": 28, "k": 0, "dtype": "complex64", "nvec": 1},
        # a block of random vectors in one momentum sector (block methods, typicality averages)
        {"name": "hv_mom_24_block", "kind": "hv", "model": "mom", "L": 24, "k": 3, "dtype": "complex128", "nvec": 16},
        # the assembled Hubbard matrix on one vector (what eigsh and ODE right-hand sides call)
        {"name": "csr_hubbard_12", "kind": "csr", "model": "hubbard", "L": 12, "k": 0, "dtype": "float64", "nvec": 1},
        # a time step on a small assembled matrix: launches and latency
        {"name": "expm_xxz_12", "kind": "expm", "form": "csr", "model": "xxz", "L": 12, "k": 0,
         "dtype": "float64", "nvec": 1, "t": 1.0, "imag": False},
        # a time step on the assembled matrix for an ensemble of states
        {"name": "expm_xxz_18_block", "kind": "expm", "form": "csr", "model": "xxz", "L": 18, "k": 0,
         "dtype": "float64", "nvec": 12, "t": 0.5, "imag": False},
        # a matrix-free time step of a large disordered chain in double precision
        {"name": "expm_xxz_26", "kind": "expm", "form": "mf", "model": "xxz", "L": 26, "k": 0,
         "dtype": "float64", "nvec": 1, "t": 0.1, "imag": False},
        # a Krylov basis in the fully symmetric sector and a thermal state from it
        {"name": "lanczos_heis_28", "kind": "lanczos", "model": "heis", "L": 28, "k": 0, "dtype": "float64",
         "m": 40, "tau": 0.5},
        # the same on a small sector, as in a scan over sectors and seeds
        {"name": "lanczos_mom_16", "kind": "lanczos", "model": "mom", "L": 16, "k": 5, "dtype": "complex128",
         "m": 40, "tau": 0.5},
        # every momentum sector of a chain, many states each, in single precision
        {"name": "sectors_20", "kind": "sectors", "L": 20, "dtype": "complex64", "nvec": 32, "t": 2.0},
        # steps of the driven Hubbard chain in its factorised form, FP32 terms with FP64 accumulation
        {"name": "driven_hubbard_14", "kind": "driven", "L": 14, "form": "kron", "dtype": "complex64",
         "nsteps": 20, "dt": 0.02},
    ]


def _loguniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["hv", "hv", "hv", "csr", "csr", "expm", "expm", "lanczos", "sectors", "driven"])
    real = rng.choice(["float64", "float64", "float32"])
    dtype = rng.choice([real, COMPLEX[real]])
    nvec = rng.choice([1, 1, _loguniform(rng, 2, 40)])
    models = {"xxz": (6, 26), "heis": (10, 28), "mom": (9, 25), "hubbard": (4, 12), "hubbard_k": (5, 11)}
    if kind == "sectors":
        return {"kind": kind, "L": rng.randint(8, 18), "dtype": COMPLEX[real], "nvec": _loguniform(rng, 3, 64),
                "t": round(rng.uniform(0.2, 2.0), 3)}
    if kind == "driven":
        return {"kind": kind, "L": rng.randint(5, 12), "form": rng.choice(["kron", "kron", "csr"]),
                "dtype": COMPLEX[real], "nsteps": rng.randint(3, 25), "dt": round(rng.uniform(0.01, 0.04), 4)}
    model = rng.choice(["xxz", "heis", "mom", "hubbard", "hubbard_k"])
    lo, hi = models[model]
    if kind != "hv":
        # the assembled matrices, Krylov bases and Taylor loops stay below the largest listed case
        hi = min(hi, {"xxz": 22, "heis": 26, "mom": 24, "hubbard": 11, "hubbard_k": 11}[model])
    size = rng.randint(lo, hi)
    if model == "heis":
        size += size % 2  # parity and spin inversion at half filling: even lengths
    k = rng.randrange(size) if model in ("mom", "hubbard_k") else 0
    if k and 2 * k != size:
        dtype = COMPLEX[real]  # complex characters
    case = {"kind": kind, "model": model, "L": size, "k": k, "dtype": dtype}
    if kind == "lanczos":
        while states({"model": model, "L": size}) < 800:
            size += 2
        case.update(L=size, dtype=dtype.replace("float32", "float64").replace("complex64", "complex128"),
                    m=rng.randint(12, 36), tau=round(rng.uniform(0.1, 1.0), 3))
        return case
    while states(case) * nvec > 12e6 and nvec > 1:
        nvec = max(1, nvec // 2)
    case["nvec"] = nvec
    if kind == "expm":
        imag = rng.random() < 0.3
        cplx = bool(k and 2 * k != size)
        case.update(form=rng.choice(["csr", "mf"]), dtype=COMPLEX[real] if cplx else real, imag=imag,
                    t=round(rng.uniform(0.05, 1.0), 3))
    return case


def states(case):
    """Number of states of a case's sector (to within the rounding of the orbit count)."""
    size = case["L"]
    if case.get("model") == "heis":
        return max(1, math.comb(size, size // 2) // (4 * size))
    if case.get("model") == "mom":
        return max(1, math.comb(size, size // 2) // size)
    if case.get("model") in ("hubbard", "hubbard_k"):
        n = math.comb(size, size // 2) ** 2
        return max(1, n // size) if case["model"] == "hubbard_k" else n
    return math.comb(size, size // 2)


# ------------------------------------------------------------------ models
def _fields(size, seed):
    return np.random.default_rng(seed).uniform(-3, 3, size)


def _model(case, seed):
    """(basis, static list) of the case's operator."""
    size, model = case["L"], case["model"]
    i = np.arange(size)
    ring = [[i_, (i_ + 1) % size] for i_ in range(size)]
    shift = (i + 1) % size
    if model in ("hubbard", "hubbard_k"):
        blocks = {"kblock": (shift, case["k"])} if model == "hubbard_k" else {}
        basis = spinful_fermion_basis_general(size, Nf=(size // 2, size // 2), **blocks)
        right, left = [[-1.0] + b for b in ring], [[1.0] + b for b in ring]
        return basis, [["+-|", right], ["-+|", left], ["|+-", right], ["|-+", left],
                       ["n|n", [[4.0, j, j] for j in range(size)]]]
    blocks = {}
    if model == "heis":
        blocks = {"kblock": (shift, 0), "pblock": (i[::-1].copy(), 0), "zblock": (-(i + 1), 0)}
    elif model == "mom":
        blocks = {"kblock": (shift, case["k"])}
    static = [["+-", [[0.5] + b for b in ring]], ["-+", [[0.5] + b for b in ring]], ["zz", [[1.0] + b for b in ring]]]
    if model == "xxz":
        static.append(["z", [[float(h), j] for j, h in enumerate(_fields(size, seed))]])
    return spin_basis_general(size, Nup=size // 2, pauli=0, **blocks), static


def _vectors(rows, nvec, dtype, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    x = torch.randn((rows,) if nvec == 1 else (rows, nvec), dtype=getattr(torch, dtype), device="cuda", generator=gen)
    return x / x.norm()


def _evolved_dtype(case):
    """dtype of an expm case's vectors: real only for real operators in imaginary time."""
    return case["dtype"] if case["imag"] and not case["dtype"].startswith("complex") \
        else COMPLEX.get(case["dtype"], case["dtype"])


def _drive(t):
    return 4.0 + 2.0 * math.cos(3.0 * t)


# --------------------------------------------------------------- prepare / run
def prepare(case, seed):
    kind = case["kind"]
    if kind == "sectors":
        size = case["L"]
        ops = []
        for k in range(size):
            basis, static = _model({"model": "mom", "L": size, "k": k}, seed)
            ops.append(quantum_LinearOperator(static, basis=basis, dtype=case["dtype"], **NO_CHECKS))
        evolve = expm_multiply_sectors(ops, a=-1j * case["t"], dtype=case["dtype"], nvec=case["nvec"])
        rows = sum(op.Ns for op in ops)
        x = _vectors(rows, case["nvec"], case["dtype"], seed).reshape(rows, case["nvec"])
        return {"case": case, "evolve": evolve, "x": x}
    if kind == "driven":
        size = case["L"]
        basis, static = _model({"model": "hubbard", "L": size, "k": 0}, seed)
        hop = quantum_LinearOperator(static[:4], basis=basis, dtype=case["dtype"], **NO_CHECKS)
        pair = quantum_LinearOperator([["n|n", [[1.0, j, j] for j in range(size)]]], basis=basis, dtype=np.float64,
                                      **NO_CHECKS)
        drive = DrivenEvolution(hop, pair, _drive, case["dt"], dtype=case["dtype"], state_dtype=np.complex128,
                                form=case["form"])
        x = _vectors(basis.Ns, 1, "complex128", seed)
        return {"case": case, "drive": drive, "x": x, "psi": torch.empty_like(x)}
    basis, static = _model(case, seed)
    if kind == "csr" or (kind == "expm" and case["form"] == "csr"):
        op = hamiltonian(static, [], basis=basis, dtype=case["dtype"], **NO_CHECKS)
    else:
        op = quantum_LinearOperator(static, basis=basis, dtype=case["dtype"], **NO_CHECKS)
    if kind == "expm":
        dtype = _evolved_dtype(case)
        evolve = expm_multiply_parallel(op, a=(-1.0 if case["imag"] else -1j) * case["t"], dtype=dtype)
        x = _vectors(basis.Ns, case["nvec"], dtype, seed)
        work = torch.empty((2 * basis.Ns,) + tuple(x.shape[1:]), dtype=x.dtype, device="cuda")
        return {"case": case, "evolve": evolve, "x": x, "work": work}
    return {"case": case, "op": op, "x": _vectors(basis.Ns, case.get("nvec", 1), case["dtype"], seed)}


def run(state):
    case, x = state["case"], state["x"]
    kind = case["kind"]
    if kind in ("hv", "csr"):
        return state["op"].dot(x)
    if kind == "expm":
        return state["evolve"].dot(x, work_array=state["work"])
    if kind == "lanczos":
        E, V, Q = lanczos_full(state["op"], x, case["m"])
        return {"E": E, "Q": Q, "psi": expm_lanczos(E, V, Q, a=-case["tau"])}
    if kind == "sectors":
        return state["evolve"].dot(x)
    psi = state["psi"]
    psi.copy_(x)
    return state["drive"].run(psi, 0.0, case["nsteps"], learned=False, block=case["nsteps"], exact="device")


# ------------------------------------------------------------------------ work
def _entries(case):
    """Off-diagonal elements of a row, on average."""
    size = case["L"]
    n = size // 2
    one = 2.0 * size * n * (size - n) / (size * (size - 1)) if size > 1 else 0.0
    return 2 * one if case.get("model", "hubbard") in ("hubbard", "hubbard_k") else one


def _terms(radius, dtype):
    """Products a Taylor series of e^{A}, ||A|| <= radius, takes to the dtype's precision."""
    m, term, eps = 0, 1.0, 6e-8 if dtype in ("float32", "complex64") else 1e-16
    while term > eps and m < 2000:
        m += 1
        term *= radius / m
    return m


def work(case):
    kind = case["kind"]
    esz = {"float32": 4, "float64": 8, "complex64": 8, "complex128": 16}
    if kind == "sectors":
        rows, nv = math.comb(case["L"], case["L"] // 2), case["nvec"]
        e, m = esz[case["dtype"]], _terms(case["t"] * 0.45 * case["L"], case["dtype"])
        per = _entries({"model": "mom", "L": case["L"]})
        return {"bytes": m * (5 * rows + 6 * rows * nv * e), "flops": m * rows * nv * 8 * (per + 1)}
    if kind == "driven":
        rows, e = states({"model": "hubbard", "L": case["L"]}), esz[case["dtype"]]
        m = case["nsteps"] * _terms(case["dt"] * 2.0 * case["L"], case["dtype"])
        return {"bytes": m * rows * (2 * e + 32 + 8), "flops": m * rows * 4 * (_entries({"L": case["L"]}) + 2)}
    rows, e, per = states(case), esz[case["dtype"]], _entries(case)
    nv = case.get("nvec", 1)
    mul = 2 if case["dtype"].startswith("float") else 8
    free = (8 if case["L"] * (2 if "hubbard" in case["model"] else 1) > 32 else 4) + 1
    if kind == "hv":
        return {"bytes": rows * (free + 2 * nv * e), "flops": rows * nv * mul * (per + 1)}
    nnz = rows * (per + 1)
    if kind == "csr":
        return {"bytes": 4 * rows + nnz * (4 + e) + 2 * rows * nv * e, "flops": nnz * nv * mul}
    if kind == "lanczos":
        m = case["m"]
        return {"bytes": m * rows * (free + 7 * e) + m * rows * e, "flops": m * rows * mul * (per + 6)}
    v = esz[_evolved_dtype(case)]
    m = _terms(case["t"] * (0.45 + (0.75 if case["model"] == "xxz" else 0.5)) * case["L"], case["dtype"])
    matrix = rows * free if case["form"] == "mf" else 4 * rows + nnz * (4 + e)
    return {"bytes": m * (matrix + 4 * rows * nv * v), "flops": m * nnz * nv * 4}


def tolerance(case):
    """About four times the largest error against ``exact`` seen over the drawn ranges."""
    kind = case["kind"]
    single = case["dtype"] in ("float32", "complex64")
    if kind in ("hv", "csr"):
        return {"rel": 4e-7 if single else 1e-14}
    if kind == "lanczos":
        return {"rel": 5e-11}  # the Krylov vectors amplify rounding from step to step
    if kind == "driven":
        return {"rel": 1e-7 if single else 1e-14}
    return {"rel": 2e-6 if single else 1.5e-14}


# ------------------------------------------------- the same in plain torch, 64 bits
def _popcount(x):
    x = x - ((x >> 1) & 0x5555555555555555)
    x = (x & 0x3333333333333333) + ((x >> 2) & 0x3333333333333333)
    x = (x + (x >> 4)) & 0x0F0F0F0F0F0F0F0F
    for s in (8, 16, 32):
        x = x + (x >> s)
    return x & 0x7F


def _sector_words(size, n, device):
    words = torch.arange((1 << size) - 1, -1, -1, dtype=torch.int64, device=device)
    return words[_popcount(words) == n]


def _orbit(words, model, size, k):
    """Orbit maximum, character and stabiliser character sum of every word.
    Site j is bit size - 1 - j; a translation moves every bit up by one."""
    full = (1 << size) - 1
    best = words.clone()
    chi = torch.ones(words.shape, dtype=torch.complex128, device=words.device)
    norm = torch.zeros(words.shape, dtype=torch.complex128, device=words.device)
    flips = [(p, z) for p in (0, 1) for z in (0, 1)] if model == "heis" else [(0, 0)]
    for p, z in flips:
        w = words
        if p:
            w = torch.zeros_like(words)
            for b in range(size):
                w |= ((words >> b) & 1) << (size - 1 - b)
        if z:
            w = w ^ full
        for step in range(size):
            c = complex(math.cos(2 * math.pi * k * step / size), math.sin(2 * math.pi * k * step / size))
            up = w > best
            best = torch.where(up, w, best)
            chi[up] = c
            norm[w == words] += c
            w = ((w << 1) & full) | (w >> (size - 1))
    return best, chi, norm.real


class _Reference:
    """Off-diagonal elements as gathers (index, coefficient) and the diagonal
    of a case's operator, in complex128 (float64 where real)."""

    def __init__(self, case, seed, device):
        size, model = case["L"], case["model"]
        self.gathers = []
        if model == "hubbard":
            n = size // 2
            words = _sector_words(size, n, device)
            self.shape = (len(words), len(words))
            both = _popcount(words[:, None] & words[None, :])
            self.pairs = both.to(torch.float64).reshape(-1)
            self.diag = 4.0 * self.pairs
            asc = words.flip(0)
            self.hops = []
            for j in range(size):
                a, b = size - 1 - j, size - 1 - (j + 1) % size
                src = ((words >> a) & 1) != ((words >> b) & 1)
                other = words ^ ((1 << a) | (1 << b))
                at = len(words) - 1 - torch.searchsorted(asc, other).clamp_(max=len(words) - 1)
                lo, hi = min(a, b), max(a, b)
                between = _popcount(words & (((1 << hi) - 1) ^ ((1 << (lo + 1)) - 1)))
                amp = torch.where(src, -1.0 + 2.0 * (between & 1).to(torch.float64), torch.zeros((), device=device, dtype=torch.float64))
                self.hops.append((torch.where(src, at, torch.zeros_like(at)), amp))
            return
        words = _sector_words(size, size // 2, device)
        norm = None
        if model != "xxz":
            best, _, norm = _orbit(words, model, size, case["k"])
            keep = (best == words) & (norm > 0.5)
            words, norm = words[keep], norm[keep]
        asc = words.flip(0)
        spins = [((words >> (size - 1 - j)) & 1).to(torch.float64) - 0.5 for j in range(size)]
        self.diag = sum(spins[j] * spins[(j + 1) % size] for j in range(size))
        if model == "xxz":
            self.diag = self.diag + sum(float(h) * s for h, s in zip(_fields(size, seed), spins))
        for j in range(size):
            a, b = size - 1 - j, size - 1 - (j + 1) % size
            src = ((words >> a) & 1) != ((words >> b) & 1)
            other = words ^ ((1 << a) | (1 << b))
            amp = 0.5 * src.to(torch.float64)
            if norm is not None:
                other, chi, _ = _orbit(other, model, size, case["k"])
            at = torch.searchsorted(asc, other).clamp_(max=max(len(words) - 1, 0))
            hit = src & (asc[at] == other)
            at = torch.where(hit, len(words) - 1 - at, torch.zeros_like(at))
            if norm is not None:
                amp = amp * chi.conj() * torch.sqrt(norm[at] / norm)
                if case["k"] == 0 or 2 * case["k"] == size:
                    amp = amp.real.contiguous()
            self.gathers.append((at, torch.where(hit, amp, torch.zeros_like(amp))))

    def dot(self, x, pairs=None):
        """H x (Hubbard with ``pairs``: hopping + pairs * double occupancies)."""
        wide = x.dim() > 1
        if hasattr(self, "hops"):
            diag = self.diag if pairs is None else pairs * self.pairs
            y = diag[:, None] * x if wide else diag * x
            shape = self.shape + tuple(x.shape[1:])
            grid, out = x.reshape(shape), y.view(shape)
            tail = (1,) * (len(shape) - 2)
            for at, amp in self.hops:
                out += amp.reshape((-1, 1) + tail) * grid[at]
                out += amp.reshape((1, -1) + tail) * grid[:, at]
            return y
        y = self.diag[:, None] * x if wide else self.diag * x
        for at, amp in self.gathers:
            y = y + (amp[:, None] * x[at] if wide else amp * x[at])
        return y

    def radius(self, pairs=None):
        if hasattr(self, "hops"):
            return (4.0 if pairs is None else abs(pairs)) * float(self.pairs.max()) + 2.0 * len(self.hops)
        return float(self.diag.abs().max()) + 0.5 * len(self.gathers)

    def expm(self, x, a, pairs=None):
        parts = max(1, math.ceil(abs(a) * self.radius(pairs) / 4.0))
        for _ in range(parts):
            term, total, m = x, x, 0
            while m < 80:
                m += 1
                term = self.dot(term, pairs) * (a / parts / m)
                total = total + term
                if float(term.abs().max()) <= 1e-18 * float(total.abs().max()):
                    break
            x = total
        return x


def exact(case, seed):
    kind, device = case["kind"], "cuda"
    if case.get("model") == "hubbard_k":
        return None
    wide = {torch.float32: torch.float64, torch.complex64: torch.complex128}
    if kind == "sectors":
        size, nv, out, at = case["L"], case["nvec"], [], 0
        refs = [_Reference({"model": "mom", "L": size, "k": k}, seed, device) for k in range(size)]
        x = _vectors(sum(len(r.diag) for r in refs), nv, case["dtype"], seed).to(torch.complex128)
        x = x.reshape(-1, nv)
        for ref in refs:
            out.append(ref.expm(x[at:at + len(ref.diag)], -1j * case["t"]))
            at += len(ref.diag)
        return torch.cat(out)
    if kind == "driven":
        ref = _Reference({"model": "hubbard", "L": case["L"]}, seed, device)
        x = _vectors(len(ref.diag), 1, "complex128", seed)
        for s in range(case["nsteps"]):
            x = ref.expm(x, -1j * case["dt"], _drive((s + 0.5) * case["dt"]))
        return x
    ref = _Reference(case, seed, device)
    rows = len(ref.diag)
    dtype = _evolved_dtype(case) if kind == "expm" else case["dtype"]
    x = _vectors(rows, case.get("nvec", 1), dtype, seed)
    x = x.to(wide.get(x.dtype, x.dtype))
    if kind in ("hv", "csr"):
        return ref.dot(x)
    if kind == "expm":
        return ref.expm(x, (-1.0 if case["imag"] else -1j) * case["t"])
    m = case["m"]
    Q = torch.empty((m, rows), dtype=x.dtype, device=device)
    alpha, beta = np.zeros(m), np.zeros(m)
    Q[0] = x / x.norm()
    for j in range(m):
        r = ref.dot(Q[j])
        if j:
            r = r - beta[j - 1] * Q[j - 1]
        alpha[j] = float(torch.vdot(Q[j], r).real)
        r = r - alpha[j] * Q[j]
        beta[j] = float(r.norm())
        if j + 1 < m:
            Q[j + 1] = r / beta[j]
    E, V = np.linalg.eigh(np.diag(alpha) + np.diag(beta[:-1], 1) + np.diag(beta[:-1], -1))
    c = torch.from_numpy(V @ (np.exp(-case["tau"] * E) * V[0])).to(device)
    return {"E": E, "Q": Q, "psi": (c[:, None] * Q).sum(0)}
