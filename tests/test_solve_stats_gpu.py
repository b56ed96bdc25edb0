"""What a solve reports: factorizations and phase times mean the same whichever
kernels ran it (the row solver: the default here; the tile kernels: G2G_ROWS=0)."""
import sys

import numpy as np
import pytest

from gpusim2grid_amd import _capi
from gpusim2grid_amd import synthetic as syn

pytestmark = pytest.mark.gpu


def _stats(g, S, prec, rows_on, monkeypatch, edits=None, max_iter=10):
    print(f"solve stats n={g.n_bus} rows={S.shape[0]} prec={prec} rows_on={rows_on}", flush=True)
    sys.stdout.flush()
    if rows_on is None:
        monkeypatch.delenv("G2G_ROWS", raising=False)
    else:
        monkeypatch.setenv("G2G_ROWS", rows_on)
    B = _capi.Batch(_capi.Plan.from_grid(g.Ybus, g.pv, g.pq, g.slack), S.shape[0], precision=prec,
                    per_row_ybus=edits is not None)
    B.set_sbus(S)
    if edits is not None:
        B.set_ybus_edits(*edits)
    for _ in range(2):  # (the phases' clocks are the first solve's)
        B.set_v(g.flat_start())
        s = B.solve(max_iter=max_iter, tol=1e-8)
        _check_phases(s)
    return s, B.results()


def _check_phases(s):
    ph = [s["ms_mismatch"], s["ms_factor"], s["ms_backward"]]
    assert min(ph) > 0.0 and sum(ph) <= 1.0001 * s["ms_total"]


@pytest.mark.parametrize("n,rows,prec,hard", [(118, 1, _capi.FP64, 0), (118, 300, _capi.FP64, 1),
                                              (2000, 1, _capi.MIXED, 0), (2000, 200, _capi.FP64, 0),
                                              (118, 40, _capi.MIXED, 40)])
def test_factorizations_and_phases(n, rows, prec, hard, monkeypatch):
    g = {118: syn.grid_118, 2000: syn.grid_c1}[n]()
    p, q = syn.injection_scenarios(g, rows, seed=61)
    S = (p + 1j * q) / g.sn_mva
    S[:hard] *= 12.0  # no solution: every update of the budget
    s, (st, it, _) = _stats(g, S, prec, None, monkeypatch)
    t, (stt, itt, _) = _stats(g, S, prec, "0", monkeypatch)
    np.testing.assert_array_equal(st, stt)
    # one factorization per Newton update of the slowest row
    assert t["n_factor_launches"] == itt.max() and s["n_factor_launches"] == it.max()
    assert s["rows_factored"] == it.sum()


def test_a_tail_on_the_row_solver_counts_on(monkeypatch):
    """More rows than the row solver is taken for at the start: the tile kernels
    begin, the row solver ends the last rows, and the counts are theirs together."""
    g = syn.grid_c2()
    rows = 3 * 256 + 40
    p, q = syn.injection_scenarios(g, rows, seed=62)
    S = (p + 1j * q) / g.sn_mva
    edits = syn.outage_edits(g, syn.random_outages(g, rows, max_k=2, seed=63))
    s, (st, it, _) = _stats(g, S, _capi.FP64, None, monkeypatch, edits)
    t, (stt, itt, _) = _stats(g, S, _capi.FP64, "0", monkeypatch, edits)
    np.testing.assert_array_equal(st, stt)
    np.testing.assert_array_equal(it, itt)
    assert s["iterations"] == t["iterations"] and s["n_factor_launches"] == t["n_factor_launches"] == it.max()


@pytest.mark.parametrize("n", [118, 2000])
def test_single_power_flow_timings(n):
    """``AcPfGPU``'s timings: refactorizations are Newton updates, and each phase has its time."""
    from gpusim2grid_amd.facades import AcPfGPU
    g = {118: syn.grid_118, 2000: syn.grid_c1}[n]()
    pf = AcPfGPU((g.Ybus, g.flat_start(), g.Sbus, np.array([g.slack]), np.array([1.0]), g.pv, g.pq),
                 init_from_n_powerflow=False)
    pf.resolve(g.flat_start(), g.Sbus)
    t = pf.timings
    assert t.converged and t.nb_iter >= 3
    assert t.n_refactorize == t.nb_iter
    for e in (t.t_mismatch, t.t_refactorize, t.t_solve):
        assert e.gpu_ms > 0.0
    assert t.t_mismatch.gpu_ms + t.t_refactorize.gpu_ms + t.t_solve.gpu_ms <= 1.0001 * t.t_total_ms
