"""Launch-configuration autotuner for the fused H.v kernel.

For a matrix-free operator the tuner chooses the representative lookup
("search": orbit search + prefix-block binary search; "table": sector lookup
table in HBM) and the schedule ("rows": one lane per row; "rows2/4/8": that
many lanes per row with shuffle reduction; "queue": compacted LDS work queue;
"batch4/8": terms in batches with all lookups of a batch in flight, for
rank-based lookups; "batch14": the same with 14 terms per batch, for the
table; "batch14x": batch14 with the workgroups of each XCD on one contiguous
run of rows; "split": blocks of the split-chain layout of one hard-core-boson
sector without symmetry maps; "split2": the same layout in two passes, lower
half-chain terms per block, then upper-half and crossing terms over column
strips; "chunk4/8": direct-rank rows with the terms in chunks and predicated
gathers; all but "rows" for one vector only; "packed": the elements evaluated
once, four bytes each, and streamed, for one vector or several).  A
symmetry-reduced operator, and one on fewer than 4,096 states, takes its packed
rows where they are no larger than its sector table would be
(``packed_limit``); the others' candidates are timed on the operator's own
basis with HIP events (a few launches each) and the winner is cached per
(basis signature, dtype, nvec) in memory and in a JSON file
(``QSX_TUNE_CACHE``, default ``~/.cache/quspin_amd/tune.json``).
``QSX_TUNE=off`` disables timing and uses the static rule below;
``QSX_LOOKUP``/``QSX_SCHEDULE`` force a choice.
"""

import json
import os

import numpy as np

from . import _lib as L

_mem = {}

# schedule name -> launch code of qsx_hv_ctx_set_schedule
SCHEDULES = {"rows": 0, "queue": 1, "rows2": 2, "rows4": 3, "rows8": 4, "batch4": 5, "batch8": 6, "split": 7,
             "chunk4": 8, "chunk8": 9, "batch14": 10, "split2": 11, "batch14x": 12, "packed": 13}

# packed rows of sectors without symmetry maps, and of small sectors: of one
# operator, and of all operators on a basis together
PACKED_BYTES, PACKED_TOTAL = 64 << 20, 1 << 30
# Vectors an operator multiplies one product at a time before its packed rows
# are built, about what a build costs: 924 states 95 us against 6 us gained per
# product, 63,504 Hubbard states 250 against 15, Heisenberg L = 28 through the
# sector table 600 against 14.  Without the wait the first product of each
# further operator on a basis took 250 us in place of 155, 430 in place of 180,
# and (built by orbit search) 4,950 in place of 1,580.
PACK_AFTER = 16


def packed_limit(op):
    """Bytes the packed rows of ``op`` may take: what the sector table they
    stand in for takes, 64 MiB where that is less or there is none."""
    b = op.basis
    if not len(b._pers) or 4 * op.oplist.n_off * b.Ns <= PACKED_BYTES:
        return PACKED_BYTES
    return max(PACKED_BYTES, b.lookup_table_bytes())


def packed_fits(basis, nbytes):
    """Whether the packed rows of all operators on a basis may take ``nbytes``
    together: 1 GiB, or what its sector table, of which there is one, would."""
    return nbytes <= PACKED_TOTAL or nbytes <= basis.lookup_table_bytes()


def _cache_path():
    return os.environ.get("QSX_TUNE_CACHE", os.path.join(os.path.expanduser("~"), ".cache", "quspin_amd",
                                                         "tune.json"))


_file = (None, {})  # (path, time and size) of the file read last, and its contents


def _load_file():
    global _file
    path = _cache_path()
    try:
        st = os.stat(path)
        seen = (path, st.st_mtime_ns, st.st_size)
        if _file[0] != seen:
            with open(path) as f:
                _file = (seen, json.load(f))
        return dict(_file[1])
    except Exception:
        return {}


def _save_file(d):
    try:
        p = _cache_path()
        os.makedirs(os.path.dirname(p), exist_ok=True)
        with open(p, "w") as f:
            json.dump(d, f, indent=1, sort_keys=True)
    except Exception:
        pass


def signature(op, vdt, nvec):
    b = op.basis
    # (the number of schedules: a file written with fewer is timed again)
    return "S{}_N{}_Ns{}_G{}_maps{}_q{}_off{}_diag{}_{}_nv{}_T{}C{}".format(
        len(SCHEDULES),
        b.N, b.Ns, int(np.prod(b._pers)) if len(b._pers) else 1, len(b._pers), tuple(int(q) for q in b._qs),
        op.oplist.n_off, op.oplist.n_diag, np.dtype(vdt).name, nvec, int(op.transposed), int(op.conjugated))


def static_rule(op, vdt, nvec):
    b = op.basis
    G = int(np.prod(b._pers)) if len(b._pers) else 1
    lookup = "table" if G > 1 else "search"
    if nvec != 1:
        schedule = "rows"
    elif lookup == "table":
        schedule = "batch8"
    elif _rank_lookup(op):
        # spin / hard-core-boson sectors: "rows" launches the fast one-term-at-
        # a-time kernel when every term is bit-parallel, which outruns the
        # branch-free batches on the direct rank; other sectors keep batches
        from .basis.base_general import hcb_basis_general
        schedule = "rows" if isinstance(op.basis, hcb_basis_general) else "batch8"
    else:
        schedule = "queue" if op.oplist.n_off >= 4 else "rows"
    return {"lookup": lookup, "schedule": schedule}


def candidates(op, vdt, nvec):
    b = op.basis
    lookups = ["search"]
    if len(b._pers):
        lookups.append("table")
    out = [] if len(b._pers) else [{"lookup": "search", "schedule": "packed"}]
    for lk in lookups:
        if nvec != 1:
            out.append({"lookup": lk, "schedule": "rows"})
            continue
        scheds = ["rows", "rows2", "rows4", "queue"]
        if lk == "table" or _rank_lookup(op):
            scheds += ["batch4", "batch8"]
        if lk == "table":
            scheds += ["batch14", "batch14x"]
        if lk == "search" and _split_layout(op):
            scheds += ["split", "split2"]
        if lk == "search" and _rank_lookup(op) and not len(b._pers):
            scheds += ["chunk4", "chunk8"]
        out += [{"lookup": lk, "schedule": sc} for sc in scheds]
    return out


def _split_layout(op):
    """One hard-core-boson particle sector without symmetry maps on at most
    32 bits (the library also needs every term in the bit-parallel form and
    falls back to "rows" otherwise)."""
    from .basis.base_general import hcb_basis_general
    b = op.basis
    return (isinstance(b, hcb_basis_general) and not len(b._pers) and b.N <= 32 and b._Np is not None
            and not isinstance(b._Np, (list, tuple)))


def _rank_lookup(op):
    """No-symmetry single-sector bases index states by rank (no search)."""
    b = op.basis
    return not len(b._pers) and b._Np is not None and not isinstance(b._Np, (list, tuple)) or \
        (not len(b._pers) and getattr(b, "_spinful", False) and b._Np is not None and len(b._Np) == 1)


def choose(op, ctx, vdt, nvec, now=True):
    """Lookup and schedule of an operator.  ``now`` False: packed rows that are
    not there yet are not built; the best other choice known without timing
    anything for them is given, marked "later"."""
    forced_l, forced_s = os.environ.get("QSX_LOOKUP"), os.environ.get("QSX_SCHEDULE")
    if forced_l or forced_s:
        cfg = static_rule(op, vdt, nvec)
        if forced_l:
            cfg["lookup"] = forced_l
        if forced_s:
            cfg["schedule"] = forced_s
        return cfg
    if os.environ.get("QSX_TUNE", "on") == "off":
        return static_rule(op, vdt, nvec)
    tuned = op.basis.Ns >= 4096
    if len(op.basis._pers) or not tuned:
        if not now:
            cfg = None
            if tuned:
                key = signature(op, vdt, nvec)
                cfg = _cached(key) or _cached(key + "_unpacked")
            cfg = dict(cfg or static_rule(op, vdt, nvec), later=True)
            if cfg["lookup"] != "table" or _make_table(op.basis):
                return cfg
        # through the sector table where the basis holds it, or has to: a
        # second operator's build by orbit search takes longer than the table's
        lookup = "search"
        if op.basis.has_lookup_table() or (op._later_on_basis() and not op._packed_rows.tried and _make_table(op.basis)):
            lookup = "table"
            ctx.configure({"lookup": lookup, "schedule": "rows"}, op.basis)
        if op._packed(ctx) is not None:
            return {"lookup": lookup, "schedule": "packed"}
    if not tuned:
        return static_rule(op, vdt, nvec)
    key = signature(op, vdt, nvec)
    known = _cached(key)
    if known is not None and known["schedule"] != "packed":
        return known
    if not now:
        others = [t for t in (known or {}).get("timings", ()) if t[1] != "packed"]
        if others:
            lookup, schedule, _ = min(others, key=lambda t: t[2])
            return {"lookup": lookup, "schedule": schedule, "later": True}
        if known is None and _cached(key + "_unpacked") is not None:
            return dict(_cached(key + "_unpacked"), later=True)
    # whether there are packed rows depends on the coefficients, which the key
    # does not hold: operators refused them for that have a choice of their own
    if op._packed(ctx) is None and not op._packed_rows.too_large:
        key += "_unpacked"
        known = _cached(key)
    if known is not None:
        return known
    best = time_candidates(op, ctx, vdt, nvec)
    _mem[key] = best
    disk = _load_file()
    disk[key] = best
    _save_file(disk)
    return best


def _make_table(basis):
    """Whether the basis has its sector table, built where it can be."""
    try:
        return basis.lookup_table() is not None
    except L.torch().OutOfMemoryError:
        return False


def _cached(key):
    """The choice kept under ``key``, in memory or in the file, or None."""
    if key not in _mem:
        disk = _load_file()
        if key not in disk:
            return None
        _mem[key] = disk[key]
    return _mem[key]


def time_candidates(op, ctx, vdt, nvec, reps=5):
    t = L.torch()
    shape = (op.Ns,) if nvec == 1 else (op.Ns, nvec)
    x = t.ones(shape, dtype=L.torch_dtype(vdt), device="cuda")
    y = t.empty_like(x)
    lib = L.load()
    st = t.cuda.current_stream()

    def timed(cfg, n):
        op._configure(ctx, cfg)
        if ctx.cfg["lookup"] != cfg["lookup"] or ctx.cfg["schedule"] != cfg["schedule"]:
            return None
        for _ in range(2):
            lib.qsx_hv_ctx_apply(ctx.h, L.ptr(x), L.ptr(y), 1.0, 0.0, 1.0, 0.0, 0, L.stream_handle())
        e0, e1 = t.cuda.Event(enable_timing=True), t.cuda.Event(enable_timing=True)
        e0.record(st)
        for _ in range(n):
            lib.qsx_hv_ctx_apply(ctx.h, L.ptr(x), L.ptr(y), 1.0, 0.0, 1.0, 0.0, 0, L.stream_handle())
        e1.record(st)
        t.cuda.synchronize()
        return e0.elapsed_time(e1) / n

    results = []
    for cfg in candidates(op, vdt, nvec):
        ms = timed(cfg, reps)
        if ms is not None:
            results.append((cfg, ms))
    # candidates within 15 % of the best are timed again, longer and in
    # alternation, so that launch-to-launch noise does not pick the winner
    first = min(ms for _, ms in results)
    close = [i for i, (_, ms) in enumerate(results) if ms <= 1.15 * first]
    if len(close) > 1:
        refined = {i: float("inf") for i in close}
        for _ in range(2):
            for i in close:
                refined[i] = min(refined[i], timed(results[i][0], 8 * reps))
        for i in close:
            results[i] = (results[i][0], refined[i])
    bi = min(range(len(results)), key=lambda i: results[i][1])
    best, best_ms = dict(results[bi][0]), results[bi][1]
    best["ms"] = round(best_ms, 5)
    best["timings"] = [[c["lookup"], c["schedule"], round(ms, 5)] for c, ms in results]
    return best


# (rows per wavefront chunk, XCD slices) candidates of the batched sector kernel
BATCH_SCHEDULES = tuple((c, x) for x in (0, 1) for c in (4, 8, 16, 32))


def _batch_work(batch, terms):
    """What a sector batch is timed on: four Taylor terms (up to 64 vectors,
    what the loop takes), or one product."""
    t = L.torch()
    x = t.ones((batch.rows, batch.nvec), dtype=L.torch_dtype(batch.vdt), device="cuda")
    n = len(batch.ops)
    if terms and batch.nvec <= 64:
        work = t.empty(2 * x.numel(), dtype=x.dtype, device="cuda")
        # a tiny step: tol 0 runs all four
        return lambda: batch.expm_inplace(x, work, [(4, 1)] * n, [0.0] * n, [0.0] * n, 1e-6, graph=False)
    y = t.empty_like(x)
    return lambda: batch.apply(x, y)


def choose_batch_schedule(batch, reps=3):
    """Chunk size and chunk order for a sector batch: timed on the batch's own
    sectors, cached like the single-operator choices.  The CSR form is timed
    on Taylor terms, whose norms cost an atomic pair per chunk that the plain
    product does not have (26 sectors of L = 26 x 64 complex64 vectors: chunks
    of 4 rows give the fastest product, 7.6 ms, and a step of 1.79 s; chunks of
    16 a step of 1.15 s).  ``QSX_BATCH_CHUNK`` / ``QSX_BATCH_XCD`` force values."""
    fc, fx = os.environ.get("QSX_BATCH_CHUNK"), os.environ.get("QSX_BATCH_XCD")
    if fc or fx:
        return int(fc or 16), int(fx or 0)
    if os.environ.get("QSX_TUNE", "on") == "off" or batch.rows < 65536:
        return 16, 0
    key = _batch_key(batch.ops, batch.vdt, batch.nvec) + "_" + batch.form + "_terms"
    if key in _mem:
        return tuple(_mem[key]["schedule"])
    disk = _load_file()
    if key in disk:
        _mem[key] = disk[key]
        return tuple(disk[key]["schedule"])
    t = L.torch()
    once = _batch_work(batch, batch.form == "csr")
    st = t.cuda.current_stream()
    res = []

    for ch, xs in BATCH_SCHEDULES:
        if batch.form == "csr" and ch > 63:
            continue
        batch.set_schedule(ch, xs)
        once()
        e0, e1 = t.cuda.Event(enable_timing=True), t.cuda.Event(enable_timing=True)
        e0.record(st)
        for _ in range(reps):
            once()
        e1.record(st)
        t.cuda.synchronize()
        res.append((e0.elapsed_time(e1) / reps, (ch, xs)))
    ms, best = min(res)
    entry = {"schedule": list(best), "ms": round(ms, 5), "timings": [[list(c), round(m_, 5)] for m_, c in res]}
    _mem[key] = entry
    disk[key] = entry
    _save_file(disk)
    return best


def _batch_key(ops, vdt, nvec):
    rows = sum(op.Ns for op in ops)
    return "batch_rows{}_nsec{}_nv{}_{}_N{}".format(rows, len(ops), int(nvec), np.dtype(vdt).name, ops[0].basis.N)


def choose_batch_form(cls, ops, vdt, nvec):
    """'mf' or 'csr' for a sector batch: both forms are built and timed on the
    same work (Taylor terms) with their own tuned schedules (cached;
    ``QSX_BATCH_FORM`` forces one)."""
    forced = os.environ.get("QSX_BATCH_FORM")
    if forced:
        return forced
    rows = sum(op.Ns for op in ops)
    if os.environ.get("QSX_TUNE", "on") == "off" or rows < 65536:
        return "csr" if nvec >= 8 else "mf"
    key = _batch_key(ops, vdt, nvec) + "_form_terms"
    if key in _mem:
        return _mem[key]["form"]
    disk = _load_file()
    if key in disk:
        _mem[key] = disk[key]
        return disk[key]["form"]
    t = L.torch()
    res = []
    for form in ("mf", "csr"):
        b = cls(ops, vdt, nvec, form=form)
        once = _batch_work(b, True)
        once()
        st = t.cuda.current_stream()
        e0, e1 = t.cuda.Event(enable_timing=True), t.cuda.Event(enable_timing=True)
        e0.record(st)
        for _ in range(3):
            once()
        e1.record(st)
        t.cuda.synchronize()
        res.append((round(e0.elapsed_time(e1) / 3, 5), form))
        del b, once
    ms, best = min(res)
    entry = {"form": best, "timings": [[f, m_] for m_, f in res]}
    _mem[key] = entry
    disk[key] = entry
    _save_file(disk)
    return best
