"""The tile kernels on the paths that the default rule gives to the row solver at
these sizes (G2G_ROWS=0): streamed rounds, eager and captured, the serving loop's
slot refill, learned starts, a compacted tail on the split walk, and FP64-residual
refinement that changes from the main to the split walk midway."""
import sys

import numpy as np
import pytest

import test_refine_fp64_gpu
import test_serving_gpu
import test_split_walk_gpu
import test_stream_graph_gpu
import test_warm_gpu
from gpusim2grid_amd import _capi
from gpusim2grid_amd import synthetic as syn

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def tiles(monkeypatch):
    monkeypatch.setenv("G2G_ROWS", "0")


@pytest.mark.parametrize("prec,refine", [(_capi.FP64, False), (_capi.MIXED, False), (_capi.MIXED, True)])
def test_graph_rounds_equal_eager_rounds(prec, refine):
    test_stream_graph_gpu.test_graph_rounds_equal_eager_rounds(prec, refine)


@pytest.mark.parametrize("prec,outages", [(_capi.FP64, True), (_capi.MIXED, True)])
def test_streamed_rows_match_oracle(prec, outages):
    test_serving_gpu.test_streamed_rows_match_oracle(prec, outages)


@pytest.mark.parametrize("start", ["flat", "per_row"])
def test_bad_learned_starts_restart(start, monkeypatch):
    test_warm_gpu.test_untrained_mlp_falls_back_to_flat_start(start, None, monkeypatch)


def test_contraction_rule():
    test_warm_gpu.test_contraction_rule_restarts_rows_at_their_second_update()


def test_refined_mixed_solves_match_the_oracle():
    test_refine_fp64_gpu.test_refined_mixed_solves_match_the_oracle()


def test_split_walk_on_outage_rows_and_compaction(monkeypatch):
    test_split_walk_gpu.test_split_walk_on_outage_rows_and_compaction(monkeypatch)


@pytest.mark.parametrize("ir", [1, 2])
def test_refinement_across_a_change_of_walk(ir, monkeypatch):
    """Rows of every kind of progress: the batch starts on the main walk (more tiles
    than the split walk is taken for), the rows that need more updates go on, packed,
    on the split walk, over the same multiplier stream in the other layout; then a
    second solve starts on the main walk again.  Bitwise the answers of second
    factorizations."""
    g = syn.grid_c1()
    rows = 129 * 64
    print(f"refinement across a change of walk ir={ir}", flush=True)
    sys.stdout.flush()
    p, q = syn.injection_scenarios(g, rows, seed=64)
    S = (p + 1j * q) / g.sn_mva
    S[::97] *= 2.5  # (stressed rows: more updates than the others)
    plan = _capi.Plan.from_grid(g.Ybus, g.pv, g.pq, g.slack)
    assert plan.info()["n_split"] > 0
    got = {}
    for refactor in ("0", "1"):
        monkeypatch.setenv("G2G_IR_REFACTOR", refactor)
        B = _capi.Batch(plan, rows, precision=_capi.MIXED)
        B.set_step_control(ir_steps=ir)
        B.set_refinement_residual(True)
        B.set_sbus(S)
        out = []
        for _ in range(2):
            B.set_v(g.flat_start())
            s = B.solve(max_iter=10, tol=1e-8)
            assert 0 < s["n_factor_main"] < s["n_factor_launches"]  # both walks ran
            out += [B.get_v(), *B.results()]
        got[refactor] = out
        del B
    for a, b in zip(got["0"], got["1"]):
        np.testing.assert_array_equal(a, b)
    assert (got["0"][1] == 0).mean() > 0.9


@pytest.mark.parametrize("prec", [_capi.FP64, _capi.MIXED])
def test_rounds_change_over_midway(prec, monkeypatch):
    """A row with more edits than the row solver holds arrives between rounds: the
    rounds go on on the tile kernels, rows under way included (captured rounds are
    captured again), with the answers of a plain solve."""
    monkeypatch.delenv("G2G_ROWS")
    g = syn.grid_118()
    rows = 150
    p, q = syn.injection_scenarios(g, rows, seed=65)
    S = (p + 1j * q) / g.sn_mva
    rp, en, de = syn.outage_edits(g, syn.random_outages(g, rows, max_k=2, seed=66))
    plan = _capi.Plan.from_grid(g.Ybus, g.pv, g.pq, g.slack)
    B = _capi.Batch(plan, rows, precision=prec, per_row_ybus=True)
    B.set_sbus(S)
    B.set_v(g.flat_start())
    B.set_ybus_edits(rp, en, de)
    B.solve(max_iter=10, tol=1e-8)
    V, st, it = B.get_v(), *B.results()[:2]
    part = lambda a, b: (rp[a:b + 1] - rp[a], en[rp[a]:rp[b]], de[rp[a]:rp[b]])  # noqa: E731
    B = _capi.Batch(plan, rows, precision=prec, per_row_ybus=True)
    B.stream_begin()
    B.stream_fill(np.arange(60), S[:60], g.flat_start()[None], edits=part(0, 60))
    for _ in range(2):
        B.stream_round(k=1, max_iter=10, tol=1e-8)
    e, d = part(60, 61)[1:]
    many = np.setdiff1d(np.arange(100), e)[:80]  # eighty edits that change nothing
    B.stream_fill([60], S[60:61], g.flat_start()[None],
                  edits=(np.array([0, e.size + 80]), np.concatenate([e, many]), np.concatenate([d, np.zeros(80)])))
    B.stream_fill(np.arange(61, rows), S[61:], g.flat_start()[None], edits=part(61, rows))
    for _ in range(14):
        B.stream_round(k=1, max_iter=10, tol=1e-8)
        if not (B.results()[0] == -1).any():
            break
    sts, its, _ = B.results()
    np.testing.assert_array_equal(sts, st)
    if prec == _capi.FP64:
        np.testing.assert_array_equal(its, it)
    ok = st == 0
    assert ok.mean() > 0.9
    Vs = B.stream_take(np.arange(rows))
    assert np.abs(Vs[ok] - V[ok]).max() < (1e-10 if prec == _capi.FP64 else 1e-7)
