"""Branch currents at the edges of the flow kernel's tiles (64 rows x 32
branches): ragged rows and branch counts, missing terminals, tripped branches,
host and device outputs, against the closed form."""
import ctypes

import numpy as np
import pytest

from gpusim2grid_amd import _capi
from gpusim2grid_amd import synthetic as syn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m,rows", [(14, 1, 1), (14, 20, 64), (118, 33, 65), (118, 180, 130), (118, 32, 63)])
def test_flows_match_the_closed_form(n, m, rows):
    import torch
    g = {14: syn.grid_c0, 118: syn.grid_118}[n]()
    rng = np.random.default_rng(n + m + rows)
    V = (1.0 + 0.05 * rng.standard_normal((rows, n))) * np.exp(0.3j * rng.standard_normal((rows, n)))
    B = _capi.Batch(_capi.Plan.from_grid(g.Ybus, g.pv, g.pq, g.slack), rows)
    B.set_v(V)
    f, t = g.branch_from[:m].copy(), g.branch_to[:m].copy()
    if m > 2:
        f[1], t[2] = -1, -1  # missing terminals
    y = [a[:m] for a in (g.yff, g.yft, g.ytf, g.ytt)]
    bo, be = rng.uniform(1, 2, m), rng.uniform(1, 2, m)
    trips = [sorted(rng.choice(m, size=min(m, r % 3), replace=False).tolist()) for r in range(rows)]
    orr, ex = B.branch_flows(f, t, *y, bo, be, trips=trips)
    z = np.zeros((rows, 1))
    Vx = np.concatenate([V, z], axis=1)  # bus -1 reads 0
    ro = np.where(f >= 0, np.abs(y[0] * Vx[:, f] + y[1] * Vx[:, t]) * bo, 0.0)
    re = np.where(t >= 0, np.abs(y[2] * Vx[:, f] + y[3] * Vx[:, t]) * be, 0.0)
    for r, tr in enumerate(trips):
        ro[r, tr] = re[r, tr] = 0.0
    # a few FP64 roundings of terms of this size
    scale = 1e-14 * (np.abs(y[0]).max() + np.abs(y[1]).max()) * 4
    assert np.abs(orr - ro).max() < scale and np.abs(ex - re).max() < scale
    # the same into device arrays
    do, de = (torch.full((rows, m), -1.0, dtype=torch.float64, device="cuda") for _ in range(2))
    torch.cuda.synchronize()
    y4 = np.ascontiguousarray(np.stack(y, axis=1), dtype=np.complex128)
    tp = np.concatenate([[0], np.cumsum([len(x) for x in trips])]).astype(np.int32)
    tb = np.array([b for x in trips for b in x] + [0], np.int32)
    f, t = f.astype(np.int32), t.astype(np.int32)
    P = lambda a: a.ctypes.data_as(ctypes.c_void_p)  # noqa: E731
    assert _capi.lib().g2g_batch_branch_flows(B._h, m, P(f), P(t), P(y4), P(bo), P(be), P(tp), P(tb),
                                              ctypes.c_void_p(do.data_ptr()), ctypes.c_void_p(de.data_ptr())) == 0
    np.testing.assert_array_equal(do.cpu().numpy(), orr)
    np.testing.assert_array_equal(de.cpu().numpy(), ex)
    bad = np.array([m] * tb.size, np.int32)  # a branch out of range is still refused
    if tp[-1] > 0:
        assert _capi.lib().g2g_batch_branch_flows(B._h, m, P(f), P(t), P(y4), P(bo), P(be), P(tp), P(bad),
                                                  ctypes.c_void_p(do.data_ptr()),
                                                  ctypes.c_void_p(de.data_ptr())) == _capi.G2G_ERR_INVALID


@pytest.mark.parametrize("rows_then", [40, 3])
def test_flows_outlive_a_run_that_fails(rows_then):
    """The currents of one run stay readable, as they were computed, after a later
    run (of as many rows or of fewer) that raised before it solved anything."""
    from gpusim2grid_amd.facades import InjectionSweepGPU
    from gpusim2grid_amd.warmstart import WarmStart
    g, other = syn.grid_118(), syn.grid_c0()
    f = InjectionSweepGPU((g.Ybus, g.flat_start(), g.Sbus, np.array([g.slack]), np.array([1.0]), g.pv, g.pq),
                          init_from_n_powerflow=False, nb_iter=8)
    f.set_branch_data(*g.branch_data(), bus_vn_kv=np.full(g.n_bus, 225.0), sn_mva=g.sn_mva)
    p, q = syn.injection_scenarios(g, 40, seed=51)
    f.set_injections(p, q, g.sn_mva)
    f.compute(batch_size=16)
    f.compute_flows()
    orr, ex = f.or_amps, f.ex_amps
    assert np.isfinite(orr).all() and orr.shape == (40, g.n_branch)
    f.set_injections(p[:rows_then], q[:rows_then], g.sn_mva)
    f.set_warm_start(WarmStart(other.n_bus, other.pv, other.pq, other.slack, np.abs(other.flat_start()), n_hidden=16))
    with pytest.raises(Exception, match="MLP"):  # another grid's network
        f.compute(batch_size=16)
    np.testing.assert_array_equal(f.or_amps, orr)
    np.testing.assert_array_equal(f.ex_amps, ex)


def test_trip_lists_that_step_back_are_empty():
    """A row whose trip_ptr steps back has no tripped branch (the C call reads
    ranges, it has never asked for them in order), and entries that no row's
    range covers are not looked at."""
    g = syn.grid_c0()
    rows, m = 4, g.n_branch
    B = _capi.Batch(_capi.Plan.from_grid(g.Ybus, g.pv, g.pq, g.slack), rows)
    B.set_v(np.tile(g.flat_start() * np.exp(0.1j * np.arange(g.n_bus)), (rows, 1)))
    f, t = g.branch_from.astype(np.int32), g.branch_to.astype(np.int32)
    y4 = np.ascontiguousarray(np.stack([g.yff, g.yft, g.ytf, g.ytt], axis=1), dtype=np.complex128)
    one = np.ones(m)
    tp = np.array([1, 4, 2, 3, 1], np.int32)  # rows: [1, 4), none, [2, 3), none
    tb = np.array([m + 7, 5, 0, 9], np.int32)  # the first entry is no row's
    P = lambda a: a.ctypes.data_as(ctypes.c_void_p)  # noqa: E731

    def flows(*trips):
        o, e = np.full((rows, m), -1.0), np.full((rows, m), -1.0)
        rc = _capi.lib().g2g_batch_branch_flows(B._h, m, P(f), P(t), P(y4), P(one), P(one), *trips, P(o), P(e))
        assert rc == 0
        return o, e

    plain, tripped = flows(None, None), flows(P(tp), P(tb))
    for a, b in zip(plain, tripped):
        a = a.copy()
        a[0, [5, 0, 9]] = 0.0
        a[2, 0] = 0.0
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("batch", [7, 64])
def test_flows_in_host_memory_equal_those_on_the_device(batch):
    """A screen's currents past the bound of what the device keeps: the same, row
    by row (trips, rows not simulated, chunks whose rows are not consecutive)."""
    from gpusim2grid_amd.facades import ContingencyAnalysisGPU
    g = syn.grid_118()
    f = ContingencyAnalysisGPU((g.Ybus, g.flat_start(), g.Sbus, np.array([g.slack]), np.array([1.0]), g.pv, g.pq),
                               init_from_n_powerflow=False, nb_iter=10)
    f.set_branch_data(*g.branch_data(), bus_vn_kv=np.full(g.n_bus, 225.0), sn_mva=g.sn_mva)
    cand = syn.bridges(g.n_bus, g.branch_from, g.branch_to)  # (a bridge's outage splits the grid: not simulated)
    assert cand.any() and not cand.all()
    f.add_contingencies_by_branch_id([[int(b)] for b in range(0, 60)])
    f.compute(batch_size=batch)
    f.compute_flows()
    orr, ex = f.or_amps, f.ex_amps
    f.solver._flow_device_bytes = 2 * orr.nbytes - 1
    f.compute_flows()
    np.testing.assert_array_equal(f.or_amps, orr)
    np.testing.assert_array_equal(f.ex_amps, ex)
    skipped = np.isnan(orr).all(axis=1)
    np.testing.assert_array_equal(skipped, cand[:60])
    f.solver._flow_device_bytes = 2 * orr.nbytes  # (and back)
    f.compute_flows()
    np.testing.assert_array_equal(f.or_amps, orr)
