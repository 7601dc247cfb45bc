"""Which form an operator is given (host logic; the timing is replaced)."""

import types

import numpy as np
import pytest

from quspin_amd import tuning

F64 = np.dtype(np.float64)


class Op:
    """An operator on a sector of 5,000 states without symmetry maps, with or
    without packed rows."""

    transposed = conjugated = False
    Ns = 5000

    def __init__(self, packable):
        self.packable = packable
        self.builds = 0
        self.basis = types.SimpleNamespace(N=20, Ns=5000, _pers=[], _qs=[], _Np=None)
        self.oplist = types.SimpleNamespace(n_off=20, n_diag=0)
        self._packed_rows = types.SimpleNamespace(too_large=False)

    def _packed(self, ctx):
        self.builds += 1
        return ("rows",) if self.packable else None


@pytest.fixture
def timed(monkeypatch, tmp_path):
    """Operators timed; packed rows win where there are some."""
    monkeypatch.setenv("QSX_TUNE_CACHE", str(tmp_path / "tune.json"))
    for v in ("QSX_LOOKUP", "QSX_SCHEDULE", "QSX_TUNE"):
        monkeypatch.delenv(v, raising=False)
    monkeypatch.setattr(tuning, "_mem", {})
    ops = []

    def time_candidates(op, ctx, vdt, nvec, reps=5):
        ops.append(op)
        return {"lookup": "search", "schedule": "packed" if op.packable else "split2"}
    monkeypatch.setattr(tuning, "time_candidates", time_candidates)
    return ops


@pytest.mark.parametrize("order", [(True, False), (False, True)])
def test_refused_operators_have_a_choice_of_their_own(timed, order):
    """Two operators of one shape, one with too many distinct coefficients for
    packed rows: each gets the form timed for its kind, in either order, and
    once per kind, also through the file."""
    for _ in range(2):
        for packable in order:
            cfg = tuning.choose(Op(packable), None, F64, 1)
            assert cfg["schedule"] == ("packed" if packable else "split2")
        tuning._mem.clear()
    assert [op.packable for op in timed] == list(order)


def test_no_rows_are_built_where_another_form_won(timed, monkeypatch):
    """Once another form won for operators with packed rows, the next ones do
    not evaluate theirs."""
    monkeypatch.setattr(tuning, "time_candidates",
                        lambda op, ctx, vdt, nvec, reps=5: {"lookup": "search", "schedule": "split2"})
    tuning.choose(Op(True), None, F64, 1)
    op = Op(True)
    assert tuning.choose(op, None, F64, 1)["schedule"] == "split2" and op.builds == 0


def test_an_operator_too_large_for_rows_is_not_tried_again(timed):
    """A refusal for the size holds for every operator of the shape: the choice
    is kept under the common key and the next operator builds nothing."""
    op = Op(False)
    op._packed_rows.too_large = True
    assert tuning.choose(op, None, F64, 1)["schedule"] == "split2"
    op = Op(False)
    assert tuning.choose(op, None, F64, 1)["schedule"] == "split2" and op.builds == 0


def test_rows_not_built_yet_take_the_best_other_choice(timed, monkeypatch):
    """``now`` False: the fastest form besides packed rows, marked to be
    replaced, and nothing is built or timed; with ``now`` the rows."""
    timings = [["search", "packed", 1.0], ["search", "rows", 3.0], ["search", "split2", 2.0]]
    monkeypatch.setattr(tuning, "time_candidates", lambda op, ctx, vdt, nvec, reps=5: {
        "lookup": "search", "schedule": "packed", "timings": timings})
    tuning.choose(Op(True), None, F64, 1)
    op = Op(True)
    assert tuning.choose(op, None, F64, 1, now=False) == {"lookup": "search", "schedule": "split2", "later": True}
    assert op.builds == 0
    assert tuning.choose(op, None, F64, 1)["schedule"] == "packed" and op.builds == 1


def test_small_sector_waits_with_the_static_rule(timed):
    op = Op(True)
    op.Ns = op.basis.Ns = 900
    op.basis.has_lookup_table = lambda: False
    op._later_on_basis = lambda: False
    cfg = tuning.choose(op, None, F64, 1, now=False)
    assert cfg == dict(tuning.static_rule(op, F64, 1), later=True) and op.builds == 0
    assert tuning.choose(op, None, F64, 1)["schedule"] == "packed"
