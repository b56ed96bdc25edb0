"""The row solver (one workgroup per power flow) against the tile kernels
(G2G_ROWS=0) and the CPU oracle, at the edges of its shapes: the smallest
grids (one bus with unknowns, one elimination level), fixed buses, every block
and V in LDS, the blocks alone, part of the blocks; one row, partial tiles,
more rows than workgroups; edited Ybus rows, learned starts with restarts,
refinement, both schedules; and rows that do not converge, which it leaves to
the tile kernels."""
import sys

import numpy as np
import pytest

from gpusim2grid_amd import _capi
from gpusim2grid_amd import synthetic as syn
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _grid(n):
    if n in (2, 3):
        return syn.make_grid(n, n - 1, n_pv=n - 2, accept=False)
    named = {14: syn.grid_c0, 118: syn.grid_118, 2000: syn.grid_c1, 6500: syn.grid_c2}
    return named[n]() if n in named else syn.make_grid(n, (3 * n) // 2, pv_frac=0.15)


def _solve(g, S, prec, monkeypatch, rows_on, pv=None, pq=None, edits=None, ir=0, sched=_capi.CONTINUOUS, max_iter=10):
    print(f"row solver n={g.n_bus} rows={S.shape[0]} prec={prec} rows_on={rows_on} ir={ir}", flush=True)
    sys.stdout.flush()
    monkeypatch.setenv("G2G_ROWS", str(rows_on))
    P = _capi.Plan.from_grid(g.Ybus, g.pv if pv is None else pv, g.pq if pq is None else pq, g.slack)
    B = _capi.Batch(P, S.shape[0], precision=prec, per_row_ybus=edits is not None)
    if ir:
        B.set_step_control(ir_steps=ir)
        B.set_refinement_residual(True)
    B.set_sbus(S)
    B.set_v(g.flat_start())
    if edits is not None:
        B.set_ybus_edits(*edits)
    stats = B.solve(max_iter=max_iter, tol=1e-8, scheduling=sched)
    st, it, res = B.results()
    return B.get_v(), st, it, res, stats


def _S(g, rows, seed):
    p, q = syn.injection_scenarios(g, rows, seed=seed)
    return (p + 1j * q) / g.sn_mva


# FP64 answers of two solvers differ by rounding (1e-12 of |V| = 1 after the
# condition number of a 6,500-bus Jacobian); a mixed answer is within the
# tolerance's distance of the root: 1e-8 pu of residual through the inverse
# Jacobian's few tens of pu, the bound the other mixed tests use
ATOL = {_capi.FP64: 1e-10, _capi.MIXED: 1e-7}


@pytest.mark.parametrize("n,rows,prec", [
    (2, 1, _capi.FP64), (3, 65, _capi.MIXED), (14, 63, _capi.FP64), (14, 130, _capi.MIXED),
    (37, 5000, _capi.FP64), (118, 64, _capi.MIXED), (301, 700, _capi.FP64), (997, 300, _capi.FP64),
    (2000, 1, _capi.MIXED), (2000, 300, _capi.MIXED), (2000, 70, _capi.FP64), (2000, 600, _capi.FP64),
    (6500, 1, _capi.FP64), (6500, 300, _capi.MIXED),
    # V and blocks in the scratch, V an odd number of 16-byte values before the 32-byte blocks
    (3001, 40, _capi.FP64),
    # two workgroups a CU share the LDS (more rows than CUs), with blocks in the scratch
    (601, 257, _capi.FP64), (997, 257, _capi.MIXED), (1501, 513, _capi.FP64), (1501, 513, _capi.MIXED),
])
def test_row_solver_matches_oracle_and_tile_kernels(n, rows, prec, monkeypatch):
    g = _grid(n)
    S = _S(g, rows, 41)
    V, st, it, res, stats = _solve(g, S, prec, monkeypatch, 1)
    Vt, stt, itt, _, stats_t = _solve(g, S, prec, monkeypatch, 0)
    np.testing.assert_array_equal(st, stt)
    k = min(rows, 128)
    Vo, sto, ito, _ = orc.nr_batch(g.Ybus, g.flat_start(), S[:k], g.pv, g.pq, 10, 1e-8, n_threads=16)
    np.testing.assert_array_equal(st[:k], sto)
    if prec == _capi.FP64:
        np.testing.assert_array_equal(it, itt)
        np.testing.assert_array_equal(it[:k], ito)
        assert stats["iterations"] == stats_t["iterations"]
        assert stats["rows_factored"] == int(it.sum())
    assert (st == 0).all() and (res < 1e-8).all()
    assert np.abs(V - Vt).max() < ATOL[prec]
    assert np.abs(V[:k] - Vo).max() < ATOL[prec]


@pytest.mark.parametrize("prec", [_capi.FP64, _capi.MIXED])
def test_fixed_buses(prec, monkeypatch):
    g = _grid(118)
    S = _S(g, 70, 42)
    pv, pq = g.pv[3:], g.pq[5:]  # eight more buses held at their start
    V, st, it, _, _ = _solve(g, S, prec, monkeypatch, 1, pv=pv, pq=pq)
    Vt, stt, itt, _, _ = _solve(g, S, prec, monkeypatch, 0, pv=pv, pq=pq)
    np.testing.assert_array_equal(st, stt)
    assert (st == 0).all()
    assert np.abs(V - Vt).max() < ATOL[prec]
    held = np.concatenate([g.pv[:3], g.pq[:5], g.slack])
    np.testing.assert_array_equal(V[:, held], np.broadcast_to(g.flat_start()[held], (70, held.size)))


@pytest.mark.parametrize("n,prec,ir", [(118, _capi.FP64, 0), (2000, _capi.MIXED, 0), (2000, _capi.FP64, 0),
                                       (2000, _capi.MIXED, 2), (118, _capi.MIXED, 1)])
def test_edited_rows_and_refinement(n, prec, ir, monkeypatch):
    g = _grid(n)
    rows = 130
    S = _S(g, rows, 43)
    edits = syn.outage_edits(g, syn.random_outages(g, rows, max_k=2, seed=44))
    V, st, it, _, _ = _solve(g, S, prec, monkeypatch, 1, edits=edits, ir=ir)
    Vt, stt, itt, _, _ = _solve(g, S, prec, monkeypatch, 0, edits=edits, ir=ir)
    np.testing.assert_array_equal(st, stt)
    ok = st == 0
    assert ok.mean() > 0.9
    assert np.abs(V[ok] - Vt[ok]).max() < ATOL[prec]
    if prec == _capi.FP64:
        np.testing.assert_array_equal(it, itt)


def test_chunked_schedule_runs_its_count(monkeypatch):
    g = _grid(118)
    S = _S(g, 40, 45)
    for k in (0, 3, 6):
        V, st, it, _, _ = _solve(g, S, _capi.FP64, monkeypatch, 1, sched=_capi.CHUNKED, max_iter=k)
        Vt, stt, itt, _, _ = _solve(g, S, _capi.FP64, monkeypatch, 0, sched=_capi.CHUNKED, max_iter=k)
        np.testing.assert_array_equal(st, stt)
        np.testing.assert_array_equal(it, itt)
        assert (it == k).all()
        assert np.abs(V - Vt).max() < 1e-12


@pytest.mark.parametrize("prec", [_capi.FP64, _capi.MIXED])
def test_rows_that_do_not_converge_are_the_tile_kernels(prec, monkeypatch):
    """Overloaded rows (no solution) among sound ones: statuses, counts, residuals
    and voltages of the tile kernels, bit for bit."""
    g = _grid(118)
    S = _S(g, 150, 46)
    hard = [3, 64, 149]
    S[hard] *= 12.0
    V, st, it, res, _ = _solve(g, S, prec, monkeypatch, 1)
    Vt, stt, itt, rest, _ = _solve(g, S, prec, monkeypatch, 0)
    np.testing.assert_array_equal(st, stt)
    assert (st[hard] != 0).all() and (np.delete(st, hard) == 0).all()
    np.testing.assert_array_equal(it[hard], itt[hard])
    np.testing.assert_array_equal(res[hard], rest[hard])
    np.testing.assert_array_equal(V[hard], Vt[hard])


def test_learned_start_restarts(monkeypatch):
    """A network of no use (its outputs are the flat angles plus noise) makes rows
    restart from the fallback: restarts, statuses and voltages as the tile kernels'."""
    from gpusim2grid_amd.warmstart import WarmStart
    g = _grid(118)
    rows = 200
    S = _S(g, rows, 47)
    rng = np.random.default_rng(7)
    ws = WarmStart(g.n_bus, g.pv, g.pq, g.slack, np.abs(g.flat_start()), n_hidden=64, seed=3)
    mu = np.zeros(ws.n_out, np.float32)
    mu[1::2] = 1.0
    ws.mlp.set_normalization(np.zeros(ws.n_in, np.float32), np.ones(ws.n_in, np.float32), mu,
                             np.full(ws.n_out, 0.6, np.float32))
    ws.mlp.set_params({k: rng.normal(0, 0.3, v.shape).astype(np.float32) for k, v in ws.mlp.get_params().items()})
    out = []
    for on in ("1", "0"):
        monkeypatch.setenv("G2G_ROWS", on)
        P = _capi.Plan.from_grid(g.Ybus, g.pv, g.pq, g.slack)
        B = _capi.Batch(P, rows, precision=_capi.FP64)
        B.set_sbus(S)
        B.set_v(g.flat_start())
        stats = B.solve_warm(ws.mlp, k_warm=4, growth=1.0, max_iter=10, tol=1e-8)
        out.append((B.get_v(), *B.results(), stats))
    (V, st, it, _, s1), (Vt, stt, itt, _, s0) = out
    assert s1["n_requeued"] == s0["n_requeued"] > 0
    np.testing.assert_array_equal(st, stt)
    np.testing.assert_array_equal(it, itt)
    assert (st == 0).all()
    assert np.abs(V - Vt).max() < 1e-9


@pytest.mark.parametrize("n,prec", [(118, _capi.FP64), (2000, _capi.MIXED)])
def test_streamed_rounds(n, prec, monkeypatch):
    """Slots filled in two goes, rounds of one and three updates (graph replays
    among them), a scratch and an edit-list capacity that grow between rounds:
    the same answers as a plain solve of the tile kernels."""
    g = _grid(n)
    rows = 150
    S = _S(g, rows, 48)
    outs = syn.random_outages(g, rows, max_k=2, seed=49)
    edits = syn.outage_edits(g, outs)
    Vt, stt, itt, _, _ = _solve(g, S, prec, monkeypatch, 0, edits=edits)
    monkeypatch.setenv("G2G_ROWS", "1")
    P = _capi.Plan.from_grid(g.Ybus, g.pv, g.pq, g.slack)
    B = _capi.Batch(P, rows, precision=prec, per_row_ybus=True)

    def part(r0, r1):
        rp, en, de = edits
        return rp[r0:r1 + 1] - rp[r0], en[rp[r0]:rp[r1]], de[rp[r0]:rp[r1]]

    for go in range(2):
        B.stream_begin()
        B.stream_fill(np.arange(100), S[:100], g.flat_start()[None], edits=part(0, 100))
        for _ in range(3):
            B.stream_round(k=1, max_iter=10, tol=1e-8)
        if go == 1:  # twenty edits on one row (entries repeated and undone): the lists grow
            rp, en, de = part(100, 101)
            k = np.arange(20) % g.Ybus.nnz
            z = (np.array([0, en.size + 20], np.int32), np.concatenate([en, k]), np.concatenate([de, np.zeros(20)]))
            B.stream_fill([100], S[100:101], g.flat_start()[None], edits=z)
            B.stream_fill(np.arange(101, rows), S[101:], g.flat_start()[None], edits=part(101, rows))
        else:
            B.stream_fill(np.arange(100, rows), S[100:], g.flat_start()[None], edits=part(100, rows))
        for _ in range(12):
            B.stream_round(k=1 if go else 3, max_iter=10, tol=1e-8)
            st, it, _ = B.results()
            if not (st == -1).any():
                break
        np.testing.assert_array_equal(st, stt)
        if prec == _capi.FP64:
            np.testing.assert_array_equal(it, itt)
        V = B.stream_take(np.arange(rows))
        ok = st == 0
        assert np.abs(V[ok] - Vt[ok]).max() < ATOL[prec]


def _solve_from(g, S, V0, prec, monkeypatch, env, **kw):
    if env is None:
        monkeypatch.delenv("G2G_ROWS", raising=False)
    else:
        monkeypatch.setenv("G2G_ROWS", env)
    print(f"row solver rule n={g.n_bus} rows={S.shape[0]} prec={prec} env={env} {kw}", flush=True)
    P = _capi.Plan.from_grid(g.Ybus, g.pv, g.pq, g.slack)
    B = _capi.Batch(P, S.shape[0], precision=prec)
    B.set_sbus(S)
    B.set_v(V0)
    B.solve(tol=1e-8, **kw)
    return (B.get_v(), *B.results())


@pytest.mark.parametrize("n,max_iter,tiles", [(118, 0, True), (118, 2, True), (118, 3, False), (601, 3, True),
                                              (601, 4, False), (2000, 3, True), (2000, 4, False), (6500, 5, True),
                                              (6500, 6, False)])
def test_short_budgets_stay_on_the_tile_kernels(n, max_iter, tiles, monkeypatch):
    """With too few updates for the usual start the row solver would hand every row
    back unconverged, so the rule leaves such a solve to the tile kernels whatever
    its start.  Which solver ran shows in the last bits of rows that converge
    (here from next to their solution)."""
    g = _grid(n)
    S = _S(g, 20, 52)
    V, st, _, _ = _solve_from(g, S, g.flat_start(), _capi.FP64, monkeypatch, "0", max_iter=10)
    assert (st == 0).all()
    rng = np.random.default_rng(5)
    free = np.concatenate([g.pv, g.pq])
    V0 = V.copy()
    V0[:, free] *= np.exp(1e-4j * rng.standard_normal((20, free.size)))
    a = _solve_from(g, S, V0, _capi.FP64, monkeypatch, None, max_iter=max_iter)
    b = _solve_from(g, S, V0, _capi.FP64, monkeypatch, "0", max_iter=max_iter)
    np.testing.assert_array_equal(a[1], b[1])
    np.testing.assert_array_equal(a[2], b[2])
    if tiles:
        np.testing.assert_array_equal(a[0], b[0])
    else:
        assert (a[1] == 0).all() and 0.0 < np.abs(a[0] - b[0]).max() < ATOL[_capi.FP64]


@pytest.mark.parametrize("where", [[5], [4990], [5, 4990], list(range(0, 5000, 7))])
@pytest.mark.parametrize("prec", [_capi.FP64, _capi.MIXED])
def test_hard_rows_among_many(prec, where, monkeypatch):
    """Rows with no solution among more rows than two rounds of workgroups: found in
    the first round they send the rows after it to the tile kernels; found later
    they alone go there.  Either way every answer is the tile kernels', those of
    the hard rows and of the rows sent along with them bit for bit."""
    g = _grid(118)
    S = _S(g, 5000, 53)
    S[where] *= 12.0
    V, st, it, res = _solve_from(g, S, g.flat_start(), prec, monkeypatch, None, max_iter=10)
    Vt, stt, itt, rest = _solve_from(g, S, g.flat_start(), prec, monkeypatch, "0", max_iter=10)
    np.testing.assert_array_equal(st, stt)
    assert (st[where] != 0).all() and (np.delete(st, where) == 0).all()
    exact = np.arange(4200, 5000) if where[0] < 10 else np.array(where)
    exact = np.union1d(exact, where)
    for a, b in ((V, Vt), (it, itt), (res, rest)):
        np.testing.assert_array_equal(a[exact], b[exact])
    ok = st == 0
    assert np.abs(V[ok] - Vt[ok]).max() < ATOL[prec]
    if prec == _capi.FP64:
        np.testing.assert_array_equal(it, itt)


@pytest.mark.parametrize("n,rows,tiles", [(13001, 512, False), (13001, 513, True)])
def test_large_grids_change_over_at_few_rows(n, rows, tiles, monkeypatch):
    """Past the sizes whose blocks the caches hold, mixed precision: two rows a CU on
    the row solver, more on the tile kernels (which ran shows in the last bits)."""
    g = _grid(n)
    S = 0.8 * _S(g, 8, 54)[np.arange(rows) % 8]
    a = _solve_from(g, S, g.flat_start(), _capi.MIXED, monkeypatch, None, max_iter=10)
    b = _solve_from(g, S, g.flat_start(), _capi.MIXED, monkeypatch, "0", max_iter=10)
    assert (a[1] == 0).all() and (b[1] == 0).all()
    assert np.abs(a[0] - b[0]).max() < ATOL[_capi.MIXED]
    assert np.array_equal(a[0], b[0]) == tiles


def _net(n, edges, y=1.0 / (0.01 + 0.1j), drop=(), zeros=()):
    """Ybus of branches with a little charging; `drop`: entries taken out of the
    pattern one way only; `zeros`: stored entries of value zero."""
    import scipy.sparse as sp
    e = np.asarray(edges)
    f, t = e[:, 0], e[:, 1]
    Y = sp.coo_matrix((np.concatenate([np.full(2 * len(e), -y), np.full(2 * len(e), y + 0.01j), np.full(n, 1e-3j)]),
                       (np.concatenate([f, t, f, t, np.arange(n)]), np.concatenate([t, f, f, t, np.arange(n)]))),
                      shape=(n, n)).tocsr()
    Y = Y.tolil()
    for i, j in drop:
        Y[i, j] = 0
    Y = Y.tocsr()
    Y.eliminate_zeros()
    if zeros:
        i, j = np.asarray(zeros).T
        Y = Y + sp.coo_matrix((np.full(len(i), 1e-300), (i, j)), shape=(n, n)).tocsr()
        Y.data[np.abs(Y.data) < 1e-200] = 0.0
    Y.sort_indices()
    return Y


FORMS = {
    "chain": (300, [(i, i + 1) for i in range(299)], dict(y=1.0 / (1e-4 + 1e-3j))),
    "star": (90, [(0, i) for i in range(1, 90)], {}),
    "star past a record's terms": (200, [(0, i) for i in range(1, 200)], {}),
    "complete": (8, [(i, j) for i in range(8) for j in range(i)], {}),
    "entries one way only": (60, [(i, (i + 1) % 60) for i in range(60)] + [(i, i + 2) for i in range(0, 58, 2)],
                             dict(drop=[(3, 4), (10, 12), (58, 59), (0, 2)])),
    "stored zeros": (60, [(i, (i + 1) % 60) for i in range(60)],
                     dict(zeros=[(2, 40), (40, 2), (5, 30), (33, 11)])),
}


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("prec", [_capi.FP64, _capi.MIXED])
def test_forms_of_the_bus_graph(form, prec, monkeypatch):
    """Graphs at and past the record format's bounds (which the tile kernels solve;
    denser ones no plan takes), patterns that are not symmetric, stored zeros, fixed buses off the graph."""
    n, edges, kw = FORMS[form]
    Y = _net(n, edges, **kw)
    rng = np.random.default_rng(8)
    slack, pv, rest = 1, np.array([0, n // 2]), np.setdiff1d(np.arange(n), [0, 1, n // 2])
    pq = rest[:-2]  # (the last two buses are fixed)
    scale = 0.3 / n
    S = -scale * (rng.uniform(0.5, 1.5, (70, n)) + 0.3j * rng.uniform(0.5, 1.5, (70, n)))
    V0 = np.ones(n, np.complex128)
    out = []
    for env in ("1", "0"):
        monkeypatch.setenv("G2G_ROWS", env)
        print(f"form {form} prec={prec} rows_on={env}", flush=True)
        B = _capi.Batch(_capi.Plan.from_grid(Y, pv, pq, np.array([slack])), 70, precision=prec)
        B.set_sbus(S)
        B.set_v(V0)
        B.solve(max_iter=10, tol=1e-8)
        out.append((B.get_v(), *B.results()))
    (V, st, it, _), (Vt, stt, itt, _) = out
    Vo, sto, ito, _ = orc.nr_batch(Y, V0, S, pv, pq, 10, 1e-8, n_threads=16)
    assert (sto == 0).all()
    np.testing.assert_array_equal(st, sto)
    np.testing.assert_array_equal(stt, sto)
    assert np.abs(V - Vt).max() < ATOL[prec] and np.abs(V - Vo).max() < ATOL[prec]
    if prec == _capi.FP64:
        np.testing.assert_array_equal(it, ito)


@pytest.mark.parametrize("where", [[5, 900], [4990]])
def test_hard_rows_among_learned_starts(where, monkeypatch):
    """The same from learned starts, some of which fail and restart in the first round
    before the rest is sent on: statuses, counts and restarts are the tile kernels'."""
    from gpusim2grid_amd.warmstart import WarmStart
    g = _grid(118)
    rows = 5000
    S = _S(g, rows, 55)
    S[where] *= 12.0
    rng = np.random.default_rng(9)
    ws = WarmStart(g.n_bus, g.pv, g.pq, g.slack, np.abs(g.flat_start()), n_hidden=64, seed=3)
    mu = np.zeros(ws.n_out, np.float32)
    mu[1::2] = 1.0
    ws.mlp.set_normalization(np.zeros(ws.n_in, np.float32), np.ones(ws.n_in, np.float32), mu,
                             np.full(ws.n_out, 0.6, np.float32))
    ws.mlp.set_params({k: rng.normal(0, 0.3, v.shape).astype(np.float32) for k, v in ws.mlp.get_params().items()})
    out = []
    for env in (None, "0"):
        if env is None:
            monkeypatch.delenv("G2G_ROWS", raising=False)
        else:
            monkeypatch.setenv("G2G_ROWS", env)
        print(f"hard rows among learned starts {where} env={env}", flush=True)
        B = _capi.Batch(_capi.Plan.from_grid(g.Ybus, g.pv, g.pq, g.slack), rows, precision=_capi.FP64)
        B.set_sbus(S)
        B.set_v(g.flat_start())
        stats = B.solve_warm(ws.mlp, k_warm=4, growth=1.0, max_iter=10, tol=1e-8)
        out.append((B.get_v(), *B.results(), stats))
    (V, st, it, res, s1), (Vt, stt, itt, rest, s0) = out
    np.testing.assert_array_equal(st, stt)
    np.testing.assert_array_equal(it, itt)
    assert s1["n_requeued"] == s0["n_requeued"] > 0
    assert (st[where] != 0).all() and (np.delete(st, where) == 0).all()
    np.testing.assert_array_equal(V[where], Vt[where])
    np.testing.assert_array_equal(res[where], rest[where])
    ok = st == 0
    assert np.abs(V[ok] - Vt[ok]).max() < 1e-9
