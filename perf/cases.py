"""The work that users of this framework have it do, as timed cases.

A case is a dict of plain values.  Its ``kind`` names the call:

``pf``     one AC power flow through ``AcPfGPU.resolve`` (host arrays in and
           out): what an operator's or an environment's step calls in a loop.
``sweep``  rows of injections on one grid through ``Batch`` (device arrays in
           and out), plain FP64 or mixed precision, optionally with an
           FP64-residual refinement round per Newton step or with 0-2 branch
           outages per row.
``n1``     a branch-outage screen through ``ContingencyAnalysisGPU.compute``,
           optionally followed by the branch currents.
``warm``   ``sweep`` from the learned warm start (``Batch.solve_warm``).
``serve``  continuous batching through the streamed-row calls: pinned host
           payloads fill the slots, rounds run until every row has ended, the
           voltages come back to a pinned buffer.
``train``  optimiser steps of the warm start's MLP over device minibatches,
           and the trained weights read back.
``adjoint`` the batched J^T solve at solved voltages (host arrays).

Grids are the seeded synthetic ones of ``gpusim2grid_amd.synthetic``: 14, 118,
2,000 and 6,500 buses as its constructors name them, and three odd sizes
between from the same generator.  Injections follow its scenario recipe
(per-row lognormal(0, 0.1) times per-bus lognormal(0, 0.05), generation
redispatched in proportion), drawn on the device from the case's seed.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from gpusim2grid_amd import _capi
from gpusim2grid_amd import synthetic as syn
from gpusim2grid_amd.facades import AcPfGPU, ContingencyAnalysisGPU
from gpusim2grid_amd.warmstart import WarmStart, torch_angle

TOL, MAX_ITER = 1e-8, 10
DEVICE = "cuda" if torch.cuda.is_available() else "cpu"
# Newton updates from the usual start (flat; a trained network or the base case for the others)
FLAT_ITERS = {14: 4, 37: 4, 118: 4, 301: 4, 997: 5, 2000: 5, 6500: 6}


def listed():
    return [
        # one power flow of a small grid: a simulation step, all latency
        dict(name="pf_118", kind="pf", n=118, precision="fp64"),
        # one power flow of a national-size grid
        dict(name="pf_6500", kind="pf", n=6500, precision="fp64"),
        # many scenarios of a small grid, plain FP64 from the flat start
        dict(name="sweep_118_fp64", kind="sweep", n=118, rows=16384, precision="fp64", outages=False, ir=0),
        # a ragged handful of tiles: a planner's few hundred what-ifs of a mid-size grid, mixed precision
        dict(name="sweep_2000_mixed_777", kind="sweep", n=2000, rows=777, precision="mixed", outages=False, ir=0),
        # the N-1 screen: every single-branch outage of the 2,000-bus grid that does not island it, with currents
        dict(name="n1_2000", kind="n1", n=2000, rows=0, precision="fp64", scheduling="continuous", flows=True),
        # the sweep of 2,000 buses with 0-2 outages per row from the learned warm start
        dict(name="warm_2000_outages", kind="warm", n=2000, rows=16384, hidden=1024, outages=True),
        # the 6,500-bus injection sweep: plain FP64, mixed precision, warm start
        dict(name="sweep_6500_fp64", kind="sweep", n=6500, rows=16384, precision="fp64", outages=False, ir=0),
        dict(name="sweep_6500_mixed", kind="sweep", n=6500, rows=16384, precision="mixed", outages=False, ir=0),
        dict(name="warm_6500", kind="warm", n=6500, rows=16384, hidden=1024, outages=False),
        # a quarter of it with FP64-residual refinement of every Newton step, a ragged row count
        dict(name="sweep_6500_ir_4001", kind="sweep", n=6500, rows=4001, precision="mixed", outages=False, ir=1),
        # a serving node's burst: 1,000 requests of the 2,000-bus grid, each with its outages
        dict(name="serve_2000", kind="serve", n=2000, rows=1000, precision="mixed"),
        # the warm start's training at the 6,500-bus widths
        dict(name="train_6500", kind="train", n=6500, batch=512, hidden=1024, steps=24, mask=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["pf", "sweep", "sweep", "sweep", "n1", "warm", "serve", "train", "adjoint"])
    n = rng.choice([14, 37, 118, 301, 997, 2000, 2000, 6500])
    precision = rng.choice(["fp64", "mixed"])
    if kind == "pf":
        return dict(kind=kind, n=n, precision=precision)
    if kind == "sweep":
        ir = rng.choice([0, 0, 0, 1]) if precision == "mixed" else 0
        return dict(kind=kind, n=n, rows=_log_int(rng, 1, 8192 if ir else 16384), precision=precision,
                    outages=rng.random() < 0.4 and n >= 118, ir=ir)
    if kind == "n1":
        n = rng.choice([118, 301, 997, 2000])
        return dict(kind=kind, n=n, rows=_log_int(rng, 20, 4000), precision=precision,
                    scheduling=rng.choice(["continuous", "chunked"]), flows=rng.random() < 0.5)
    if kind == "warm":
        n = rng.choice([118, 301, 997, 2000, 6500])
        return dict(kind=kind, n=n, rows=_log_int(rng, 64, 16384), hidden=rng.choice([256, 512, 1024]),
                    outages=rng.random() < 0.5 and n <= 2000)
    if kind == "serve":
        n = rng.choice([118, 301, 997, 2000, 6500])
        return dict(kind=kind, n=n, rows=_log_int(rng, 32, 2048), precision=precision)
    if kind == "train":
        n = rng.choice([118, 301, 997, 2000, 6500])
        return dict(kind=kind, n=n, batch=_log_int(rng, 64, 1024), hidden=rng.choice([256, 512, 1000, 1024]),
                    steps=rng.randint(8, 24), mask=rng.random() < 0.5)
    n = rng.choice([118, 301, 997, 2000])
    return dict(kind=kind, n=n, rows=_log_int(rng, 1, 256), precision="fp64")


# ---------------------------------------------------------------------------
# Grids, injections, outages
# ---------------------------------------------------------------------------

@functools.lru_cache(maxsize=None)
def _grid(n):
    named = {14: syn.grid_c0, 118: syn.grid_118, 2000: syn.grid_c1, 6500: syn.grid_c2}
    if n in named:
        return named[n]()
    return syn.make_grid(n, (3 * n) // 2, pv_frac=0.15)


@functools.lru_cache(maxsize=None)
def _outage_candidates(n):
    g = _grid(n)
    return np.flatnonzero(~syn.bridges(g.n_bus, g.branch_from, g.branch_to))


def _injections(n, rows, seed):
    """Sbus [rows, n] complex128 on the device, per unit."""
    g = _grid(n)
    gen = torch.Generator(device=DEVICE).manual_seed(int(seed))
    t = lambda a: torch.as_tensor(np.asarray(a, np.float64), device=DEVICE)  # noqa: E731
    a = torch.exp(0.1 * torch.randn((rows, 1), generator=gen, device=DEVICE, dtype=torch.float64))
    c = torch.exp(0.05 * torch.randn((rows, n), generator=gen, device=DEVICE, dtype=torch.float64))
    c *= a
    ratio = (c @ t(g.p_load))[:, None] / float(g.p_load.sum())
    return torch.complex(t(g.p_gen)[None] * ratio - t(g.p_load)[None] * c, -t(g.q_load)[None] * c)


def _outages(case, seed):
    if not case.get("outages", case["kind"] == "serve"):
        return None
    return syn.random_outages(_grid(case["n"]), case["rows"], max_k=2, seed=seed + 3)


def _n1_trips(case, seed):
    """Every single non-islanding outage (rows 0), or that many random sets of one or two."""
    if case["rows"] == 0:
        return [[int(b)] for b in _outage_candidates(case["n"])]
    sets = syn.random_outages(_grid(case["n"]), 2 * case["rows"], max_k=2, seed=seed + 3)
    sets = [s for s in sets if s] or [[int(_outage_candidates(case["n"])[0])]]
    return (sets * (1 + case["rows"] // len(sets)))[:case["rows"]]


def _precision(case):
    return _capi.FP64 if case["precision"] == "fp64" else _capi.MIXED


def _bases(g):
    """Amperes per unit current of each branch end (a 225 kV grid)."""
    b = g.sn_mva * 1e6 / (math.sqrt(3.0) * 225e3)
    return np.full(g.n_branch, b)


# ---------------------------------------------------------------------------
# prepare / run
# ---------------------------------------------------------------------------

def prepare(case, seed):
    return _PREPARE[case["kind"]](case, int(seed))


def run(state):
    return _RUN[state["kind"]](state)


def _prepare_pf(case, seed):
    g = _grid(case["n"])
    S = _injections(case["n"], 1, seed)[0].cpu().numpy()
    pf = AcPfGPU(g.as_tuple(), precision=case["precision"], max_iter=MAX_ITER, tol=TOL, init_from_n_powerflow=False)
    return dict(kind="pf", pf=pf, V0=g.flat_start(), S=S)


def _run_pf(s):
    s["pf"].resolve(s["V0"], s["S"])
    return s["pf"].solve()


def _prepare_sweep(case, seed):
    g, rows = _grid(case["n"]), case["rows"]
    S = _injections(case["n"], rows, seed)
    outs = _outages(case, seed)
    plan = _capi.Plan.from_grid(g.Ybus, g.pv, g.pq, g.slack)
    B = _capi.Batch(plan, rows, precision=_precision(case), per_row_ybus=outs is not None)
    if outs is not None:
        B.set_ybus_edits(*syn.outage_edits(g, outs))
    if case["ir"]:
        B.set_step_control(ir_steps=case["ir"])
        B.set_refinement_residual(True)
    V0 = torch.as_tensor(g.flat_start(), device=DEVICE)
    V = torch.empty((rows, g.n_bus), dtype=torch.complex128, device=DEVICE)
    torch.cuda.synchronize()
    return dict(kind="sweep", B=B, S=S, V0=V0, V=V, n=g.n_bus, rows=rows)


def _run_sweep(s):
    B, n, rows = s["B"], s["n"], s["rows"]
    B.set_sbus_device(s["S"].data_ptr(), n, rows)
    B.set_v_device(s["V0"].data_ptr(), 0, rows)
    B.solve(max_iter=MAX_ITER, tol=TOL, scheduling=_capi.CONTINUOUS)
    B.get_v_device(s["V"].data_ptr(), n)
    return dict(V=s["V"], status=B.results()[0])


def _prepare_n1(case, seed):
    g = _grid(case["n"])
    S = _injections(case["n"], 1, seed)[0].cpu().numpy()
    grid = (g.Ybus, g.flat_start(), S, g.slack, g.slack_weights, g.pv, g.pq)
    f = ContingencyAnalysisGPU(grid, init_from_n_powerflow=False, precision=case["precision"], tol=TOL,
                               nb_iter=MAX_ITER if case["scheduling"] == "continuous" else 5,
                               scheduling=case["scheduling"])
    f.set_branch_data(*g.branch_data(), bus_vn_kv=np.full(g.n_bus, 225.0), sn_mva=g.sn_mva)
    trips = _n1_trips(case, seed)
    f.add_contingencies_by_branch_id(trips)
    return dict(kind="n1", f=f, rows=len(trips), flows=case["flows"])


def _run_n1(s):
    f = s["f"]
    out = dict(V=torch.from_dlpack(f.compute(batch_size=s["rows"])), status=np.asarray(f.get_row_status()))
    if s["flows"]:
        f.compute_flows()
        out["or_amps"], out["ex_amps"] = f.or_amps, f.ex_amps
    return out


def _warm_network(case, seed):
    """A network that predicts voltages: random hidden layers, and an output layer
    fitted by ridge regression to 2,048 solved rows (a stand-in for a training run
    that is the same wherever it is made)."""
    n, g = case["n"], _grid(case["n"])
    rows = 2048
    fit = dict(case, rows=rows)
    S = _injections(n, rows, seed + 77)
    outs = _outages(fit, seed + 77)
    plan = _capi.Plan.from_grid(g.Ybus, g.pv, g.pq, g.slack)
    B = _capi.Batch(plan, rows, precision=_capi.FP64, per_row_ybus=outs is not None)
    V = torch.empty((rows, n), dtype=torch.complex128, device=DEVICE)
    V0 = torch.as_tensor(g.flat_start(), device=DEVICE)
    torch.cuda.synchronize()
    if outs is not None:
        B.set_ybus_edits(*syn.outage_edits(g, outs))
    B.set_sbus_device(S.data_ptr(), n, rows)
    B.set_v_device(V0.data_ptr(), 0, rows)
    B.solve(max_iter=MAX_ITER, tol=TOL)
    B.get_v_device(V.data_ptr(), n)
    ok = torch.as_tensor(B.results()[0] == 0, device=DEVICE)
    S, V = S[ok].contiguous(), V[ok].contiguous()
    mask = None
    if outs is not None:
        mask = torch.as_tensor(syn.outage_mask(g, outs), device=DEVICE)[ok].contiguous()
    ws = WarmStart(n, g.pv, g.pq, g.slack, np.abs(g.flat_start()), n_hidden=case["hidden"],
                   n_mask=g.n_branch if outs is not None else 0, seed=5)
    ws.fit_normalization(S, V, mask)
    X, T = ws._normalised(S, V, mask)
    p = {k: torch.as_tensor(v, device=DEVICE) for k, v in ws.mlp.get_params().items()}
    gelu = torch.nn.functional.gelu
    H = gelu(gelu(X @ p["W1"] + p["b1"]) @ p["W2"] + p["b2"]).double()
    H = torch.cat([H, H.new_ones((H.shape[0], 1))], dim=1)
    G = H.T @ H
    G += torch.eye(G.shape[0], device=DEVICE, dtype=torch.float64) * (1e-4 * torch.trace(G) / G.shape[0])
    W = torch.linalg.solve(G, H.T @ T.double()).float()
    p["W3"], p["b3"] = W[:-1], W[-1]
    ws.mlp.set_params({k: v.cpu().numpy() for k, v in p.items()})
    return ws


def _prepare_warm(case, seed):
    g, rows, n = _grid(case["n"]), case["rows"], case["n"]
    ws = _warm_network(case, seed)
    S = _injections(n, rows, seed)
    outs = _outages(case, seed)
    plan = _capi.Plan.from_grid(g.Ybus, g.pv, g.pq, g.slack)
    B = _capi.Batch(plan, rows, precision=_capi.MIXED, per_row_ybus=outs is not None)
    if outs is not None:
        B.set_ybus_edits(*syn.outage_edits(g, outs))
        B.set_warm_mask(syn.outage_mask(g, outs))
    one = _capi.Batch(plan, 1)
    one.set_sbus(g.Sbus)
    one.set_v(g.flat_start())
    one.solve(max_iter=MAX_ITER, tol=TOL)
    V0 = torch.as_tensor(one.get_v()[0], device=DEVICE)  # the fallback start: the base case
    V = torch.empty((rows, n), dtype=torch.complex128, device=DEVICE)
    torch.cuda.synchronize()
    return dict(kind="warm", B=B, ws=ws, S=S, V0=V0, V=V, n=n, rows=rows)


def _run_warm(s):
    B, n, rows = s["B"], s["n"], s["rows"]
    B.set_sbus_device(s["S"].data_ptr(), n, rows)
    B.set_v_device(s["V0"].data_ptr(), 0, rows)
    B.solve_warm(s["ws"].mlp, k_warm=6, growth=1.0, max_iter=MAX_ITER, tol=TOL)
    B.get_v_device(s["V"].data_ptr(), n)
    return dict(V=s["V"], status=B.results()[0])


def _prepare_serve(case, seed):
    g, rows, n = _grid(case["n"]), case["rows"], case["n"]
    pin = lambda: torch.empty((rows, n), dtype=torch.complex128, pin_memory=True).numpy()  # noqa: E731
    S, V = pin(), pin()
    S[...] = _injections(n, rows, seed).cpu().numpy()
    plan = _capi.Plan.from_grid(g.Ybus, g.pv, g.pq, g.slack)
    B = _capi.Batch(plan, rows, precision=_precision(case), per_row_ybus=True)
    B.stream_begin()
    edits = syn.outage_edits(g, _outages(case, seed))
    return dict(kind="serve", B=B, S=S, V=V, V0=g.flat_start(), edits=edits, slots=np.arange(rows, dtype=np.int32))


def _run_serve(s):
    B = s["B"]
    B.stream_fill(s["slots"], s["S"], s["V0"][None], edits=s["edits"])
    for _ in range(MAX_ITER + 2):
        B.stream_round(k=1, max_iter=MAX_ITER, tol=TOL)
        status = B.results()[0]
        if not (status == -1).any():
            break
    return dict(V=B.stream_take(s["slots"], out=s["V"]), status=status)


def _train_data(case, seed):
    """Network widths, the starting parameters and the minibatches' (X, T):
    normalised injections (and a 0/1 mask), and targets that depend on them."""
    g = _grid(case["n"])
    n_mask = g.n_branch if case["mask"] else 0
    n_in, H, n_out = 2 * g.n_bus + n_mask, case["hidden"], 2 * g.n_bus
    rows = case["batch"] * case["steps"]
    gen = torch.Generator(device=DEVICE).manual_seed(int(seed))
    rnd = lambda *s: torch.randn(s, generator=gen, device=DEVICE, dtype=torch.float32)  # noqa: E731
    load = rnd(rows, 1)
    X = torch.empty((rows, n_in), device=DEVICE, dtype=torch.float32)
    X[:, :n_out] = 0.9 * load + 0.45 * rnd(rows, n_out)
    if n_mask:
        X[:, n_out:] = (torch.rand((rows, n_mask), generator=gen, device=DEVICE) < 1.0 / n_mask).float()
    T = -0.8 * load + 0.1 * load * load + 0.3 * X[:, :n_out] + 0.2 * rnd(rows, n_out)
    glorot = lambda i, o: (2.0 * torch.rand((i, o), generator=gen, device=DEVICE) - 1.0) * math.sqrt(6.0 / (i + o))  # noqa: E731
    p = dict(W1=glorot(n_in, H), b1=0.05 * rnd(H), W2=glorot(H, H), b2=0.05 * rnd(H), W3=glorot(H, n_out),
             b3=0.05 * rnd(n_out))
    return n_in, H, n_out, p, X, T.contiguous()


def _rate(k):
    return 1e-3 * (k + 1) / 390  # the step size's rise over the first 5 % of a run


CLIP = 0.3


def _prepare_train(case, seed):
    n_in, H, n_out, p, X, T = _train_data(case, seed)
    mlp = _capi.Mlp(n_in, H, n_out, seed=0)
    mlp.set_params({k: v.cpu().numpy() for k, v in p.items()})
    mlp.set_grad_clip(CLIP)
    torch.cuda.synchronize()
    return dict(kind="train", mlp=mlp, X=X, T=T, batch=case["batch"], steps=case["steps"], n_in=n_in, n_out=n_out)


def _run_train(s):
    mlp, b = s["mlp"], s["batch"]
    x, t = s["X"].data_ptr(), s["T"].data_ptr()
    losses = [mlp.train_step_device(x + 4 * k * b * s["n_in"], t + 4 * k * b * s["n_out"], b, _rate(k))
              for k in range(s["steps"])]
    return dict(losses=torch.tensor(losses), **mlp.get_params())


def _prepare_adjoint(case, seed):
    g, rows, n = _grid(case["n"]), case["rows"], case["n"]
    S = _injections(n, rows, seed)
    plan = _capi.Plan.from_grid(g.Ybus, g.pv, g.pq, g.slack)
    B = _capi.Batch(plan, rows, precision=_precision(case))
    torch.cuda.synchronize()
    B.set_sbus_device(S.data_ptr(), n, rows)
    B.set_v(g.flat_start())
    B.solve(max_iter=MAX_ITER, tol=1e-10)
    return dict(kind="adjoint", B=B, rhs=_adjoint_rhs(case, seed))


def _adjoint_rhs(case, seed):
    g = _grid(case["n"])
    return np.random.default_rng(seed).standard_normal((case["rows"], 2 * g.pq.size + g.pv.size))


def _run_adjoint(s):
    return s["B"].solve_adjoint(s["rhs"])


_PREPARE = dict(pf=_prepare_pf, sweep=_prepare_sweep, n1=_prepare_n1, warm=_prepare_warm, serve=_prepare_serve,
                train=_prepare_train, adjoint=_prepare_adjoint)
_RUN = dict(pf=_run_pf, sweep=_run_sweep, n1=_run_n1, warm=_run_warm, serve=_run_serve, train=_run_train,
            adjoint=_run_adjoint)


# ---------------------------------------------------------------------------
# work
# ---------------------------------------------------------------------------

@functools.lru_cache(maxsize=None)
def _plan_info(n):
    g = _grid(n)
    return _capi.Plan.from_grid(g.Ybus, g.pv, g.pq, g.slack).info()


def work(case):
    """Inputs read once, outputs written once; the operations of the Newton updates
    (factorization, both substitutions, mismatch and Jacobian) or of the products."""
    n, g = case["n"], _grid(case["n"])
    if case["kind"] == "train":
        n_in, H, n_out = 2 * n + (g.n_branch if case["mask"] else 0), case["hidden"], 2 * n
        weights = n_in * H + H * H + H * n_out
        rows = case["batch"] * case["steps"]
        # X and T in; weights and both moments read and written by every step; the weights out
        return dict(bytes=4.0 * rows * (n_in + n_out) + case["steps"] * 24.0 * weights + 4.0 * weights,
                    flops=rows * (6.0 * weights - 2.0 * n_in * H) + case["steps"] * 12.0 * weights)
    rows = 1 if case["kind"] == "pf" else case["rows"]
    if case["kind"] == "n1" and rows == 0:
        rows = _outage_candidates(n).size
    inf = _plan_info(n)
    per_row = 2.0 * inf["n_updates"] + 4.0 * inf["nLU"] + 30.0 * inf["nY"]
    if case["kind"] == "adjoint":
        return dict(bytes=16.0 * rows * (inf["d"] + n), flops=rows * per_row)
    iters = 3 if case["kind"] in ("n1", "warm") else FLAT_ITERS[n]
    w = dict(bytes=32.0 * rows * n, flops=rows * iters * per_row)
    if case["kind"] == "n1":
        w["bytes"] = 16.0 * rows * n + (16.0 * rows * g.n_branch if case["flows"] else 0.0)
    if case["kind"] == "warm":
        n_in = 2 * n + (g.n_branch if case["outages"] else 0)
        weights = case["hidden"] * (n_in + case["hidden"] + 2 * n)
        w["bytes"] += 4.0 * weights + (rows * g.n_branch if case["outages"] else 0)
        w["flops"] += 2.0 * rows * weights
    return w


# ---------------------------------------------------------------------------
# exact: plain torch / scipy in 64 bits
# ---------------------------------------------------------------------------

def _jacobian(g, V):
    """The polar power-flow Jacobian at one V (scipy, [P of pvpq | Q of pq])."""
    import scipy.sparse as sp
    Y, pvpq, pq = g.Ybus, np.sort(np.concatenate([g.pv, g.pq])), g.pq
    I = Y @ V
    D, N = sp.diags(V), sp.diags(V / np.abs(V))
    dA = (1j * D @ (sp.diags(I) - Y @ D).conj()).tocsr()
    dM = (D @ (Y @ N).conj() + sp.diags(np.conj(I)) @ N).tocsr()
    return sp.bmat([[dA[pvpq][:, pvpq].real, dM[pvpq][:, pq].real],
                    [dA[pq][:, pvpq].imag, dM[pq][:, pq].imag]], format="csc")


@functools.lru_cache(maxsize=2)
def _base(n):
    """The base case's V (scipy Newton) and the dense inverse of its Jacobian on the device."""
    import scipy.sparse.linalg as spl
    g = _grid(n)
    pvpq, pq = np.sort(np.concatenate([g.pv, g.pq])), g.pq
    V = g.flat_start()
    for _ in range(20):
        mis = V * np.conj(g.Ybus @ V) - g.Sbus
        F = np.concatenate([mis[pvpq].real, mis[pq].imag])
        if np.abs(F).max() < 1e-12:
            break
        dx = spl.splu(_jacobian(g, V)).solve(-F)
        va, vm = np.angle(V), np.abs(V)
        va[pvpq] += dx[:pvpq.size]
        vm[pq] += dx[pvpq.size:]
        V = vm * np.exp(1j * va)
    return V, _inverse(torch.as_tensor(_jacobian(g, V).toarray(), device=DEVICE))


def _inverse(A):
    """Dense inverse by halves (the factorization libraries take no 12,218 x 12,218 matrix)."""
    k = A.shape[0] // 2
    if k < 2048:
        return torch.linalg.inv(A)
    P = _inverse(A[:k, :k].contiguous())
    PB = P @ A[:k, k:]
    CP = A[k:, :k] @ P
    Q = _inverse(A[k:, k:] - A[k:, :k] @ PB)
    return torch.cat([torch.cat([P + PB @ (Q @ CP), -(PB @ Q)], 1), torch.cat([-(Q @ CP), Q], 1)], 0)


def _newton_row(g, S, trips, V):
    """Newton's method with its own Jacobian for one row (scipy); None if it ends nowhere."""
    import dataclasses
    import scipy.sparse.linalg as spl
    keep = np.ones(g.n_branch, bool)
    keep[list(trips)] = False
    Y = syn.build_ybus(g.n_bus, g.branch_from[keep], g.branch_to[keep], g.yff[keep], g.yft[keep], g.ytf[keep],
                       g.ytt[keep])
    g = dataclasses.replace(g, Ybus=Y)
    pvpq, pq = np.sort(np.concatenate([g.pv, g.pq])), g.pq
    for _ in range(15):
        mis = V * np.conj(Y @ V) - S
        F = np.concatenate([mis[pvpq].real, mis[pq].imag])
        if np.abs(F).max() < 1e-12:
            return V
        dx = spl.splu(_jacobian(g, V)).solve(-F)
        va, vm = np.angle(V), np.abs(V)
        va[pvpq] += dx[:pvpq.size]
        vm[pq] += dx[pvpq.size:]
        V = vm * np.exp(1j * va)
    return None


def _trip_correction(g, Vb, Jinv, pos, R, rr, f, t, y):
    """What R rows' trips (branch f -> t of row rr, admittances y) change in the base
    Jacobian, as the low-rank update (I + M C)^-1 M of its inverse: the touched
    unknowns [8, R] (-1: none), the 8 x 8 gains, and the inverse's columns there."""
    V = torch.as_tensor(Vb, device=DEVICE)
    yff, yft, ytf, ytt = y
    rows = rr.cpu().numpy()
    first = torch.as_tensor(np.r_[True, rows[1:] != rows[:-1]], device=DEVICE)
    slot = torch.where(first, 0, 4)
    at = torch.full((8, R), -1, dtype=torch.int64, device=DEVICE)
    M = torch.zeros((R, 8, 8), dtype=torch.float64, device=DEVICE)
    ends = ((f, t, yff, yft), (t, f, ytt, ytf))
    for e, (a, b, yaa, yab) in enumerate(ends):
        at[slot + 2 * e, rr], at[slot + 2 * e + 1, rr] = pos[0, a], pos[1, a]
        va, vb = V[a], V[b]
        w = va * (yab * vb).conj()
        own = va / va.abs() * (yaa * va + yab * vb).conj() + va * (yaa * va / va.abs()).conj()
        for q, dS in ((2 * e, 1j * w), (2 * e + 1, own), (2 - 2 * e, -1j * w), (3 - 2 * e, w / vb.abs())):
            M[rr, slot + 2 * e, slot + q] = -dS.real
            M[rr, slot + 2 * e + 1, slot + q] = -dS.imag
    none = at < 0
    cols = Jinv[:, at.clamp(min=0).reshape(-1)].reshape(-1, 8, R)
    cols[:, none] = 0.0
    C = cols.gather(0, at.clamp(min=0)[:, None, :].expand(8, 8, R)).permute(2, 0, 1).contiguous()
    M.masked_fill_(none.T[:, :, None] | none.T[:, None, :], 0.0)
    eye = torch.eye(8, dtype=torch.float64, device=DEVICE)
    return at, torch.linalg.solve(eye + M @ C, M), cols


def _solve_exact(n, S, trips=None):
    """V [rows, n] on the device for Sbus S: Newton's method with the base case's
    Jacobian throughout, which ends at the same root, then with their own for the
    rows that it does not take there; None if some row gets nowhere or too many are left."""
    g = _grid(n)
    Vb, Jinv = _base(n)
    Y = g.Ybus.tocoo()
    ti = lambda a: torch.as_tensor(np.asarray(a, np.int64), device=DEVICE)  # noqa: E731
    yi, yj, yx = ti(Y.row), ti(Y.col), torch.as_tensor(Y.data, device=DEVICE)[:, None]
    pvpq_h = np.sort(np.concatenate([g.pv, g.pq]))
    pvpq, pq, npv = ti(pvpq_h), ti(g.pq), pvpq_h.size
    pos = torch.full((2, n), -1, dtype=torch.int64, device=DEVICE)  # unknown of each bus's angle and |V|
    pos[0, pvpq] = torch.arange(npv, device=DEVICE)
    pos[1, pq] = npv + torch.arange(pq.numel(), device=DEVICE)
    out = torch.empty_like(S)
    left = []
    step = 512 if trips is not None else 2048
    for r0 in range(0, S.shape[0], step):
        Sc = S[r0:r0 + step].T.contiguous()
        R = Sc.shape[1]
        ed = fix = None
        if trips is not None:
            rows = [(r, b) for r, t in enumerate(trips[r0:r0 + R]) for b in t]
            if rows:
                rr, br = ti([r for r, _ in rows]), np.array([b for _, b in rows])
                y = [torch.as_tensor(a[br], device=DEVICE) for a in (g.yff, g.yft, g.ytf, g.ytt)]
                ed = rr, ti(g.branch_from[br]), ti(g.branch_to[br]), y
                fix = _trip_correction(g, Vb, Jinv, pos, R, *ed)
        V = torch.as_tensor(Vb, device=DEVICE)[:, None].repeat(1, R)
        va, vm = torch_angle(V), V.abs()
        for _ in range(80):
            I = torch.zeros_like(V)
            I.index_add_(0, yi, yx * V[yj])
            if ed is not None:
                rr, f, t, (yff, yft, ytf, ytt) = ed
                I.index_put_((f, rr), -(yff * V[f, rr] + yft * V[t, rr]), accumulate=True)
                I.index_put_((t, rr), -(ytf * V[f, rr] + ytt * V[t, rr]), accumulate=True)
            mis = V * I.conj() - Sc
            F = torch.cat([mis.real[pvpq], mis.imag[pq]])
            m = F.abs().amax(0)
            lost = ~(m < 10.0)  # diverging: left to its own Jacobian
            if not bool(((m > 5e-13) & ~lost).any()):
                break
            dx = Jinv @ torch.where(lost[None], torch.zeros_like(F), F)
            if fix is not None:
                at, gain, cols = fix
                z = torch.where(at < 0, torch.zeros((), dtype=dx.dtype, device=DEVICE), dx.gather(0, at.clamp(min=0)))
                w = torch.linalg.vecdot(gain, z.T[:, None, :].expand_as(gain))
                dx = dx - (cols * w.T[None]).sum(1)
            va[pvpq] -= dx[:npv]
            vm[pq] -= dx[npv:]
            V = torch.polar(vm, va)
        out[r0:r0 + R] = V.T
        left += (r0 + torch.nonzero(~(m < 1e-11)).flatten().cpu().numpy()).tolist()
    if len(left) > 150:
        return None
    for r in left:
        V = _newton_row(g, S[r].cpu().numpy(), trips[r] if trips is not None else [], Vb.copy())
        if V is None:
            return None
        out[r] = torch.as_tensor(V, device=DEVICE)
    return out


def exact(case, seed):
    kind, n = case["kind"], case["n"]
    g = _grid(n)
    if kind == "pf":
        V = _solve_exact(n, _injections(n, 1, seed))
        return None if V is None else V[0].cpu().numpy()
    if kind in ("sweep", "warm", "serve"):
        V = _solve_exact(n, _injections(n, case["rows"], seed), _outages(case, seed))
        if V is None:
            return None
        return dict(V=V.cpu().numpy() if kind == "serve" else V, status=None)
    if kind == "n1":
        trips = _n1_trips(case, seed)
        V = _solve_exact(n, _injections(n, 1, seed).repeat(len(trips), 1), trips)
        if V is None:
            return None
        out = dict(V=V, status=None)
        if case["flows"]:
            base = torch.as_tensor(_bases(g), device=DEVICE)
            f, t = (torch.as_tensor(np.asarray(a, np.int64), device=DEVICE) for a in (g.branch_from, g.branch_to))
            y = [torch.as_tensor(a, device=DEVICE) for a in (g.yff, g.yft, g.ytf, g.ytt)]
            orr = (y[0] * V[:, f] + y[1] * V[:, t]).abs() * base
            ex = (y[2] * V[:, f] + y[3] * V[:, t]).abs() * base
            for r, tr in enumerate(trips):
                orr[r, tr] = 0.0
                ex[r, tr] = 0.0
            out["or_amps"], out["ex_amps"] = orr.cpu().numpy(), ex.cpu().numpy()
        return out
    if kind == "adjoint":
        import scipy.sparse.linalg as spl
        V = _solve_exact(n, _injections(n, case["rows"], seed))
        if V is None:
            return None
        V, rhs = V.cpu().numpy(), _adjoint_rhs(case, seed)
        return np.stack([spl.splu(_jacobian(g, v)).solve(b, trans="T") for v, b in zip(V, rhs)])
    return _train_exact(case, seed)


def _train_exact(case, seed):
    _, _, n_out, p, X, T = _train_data(case, seed)
    p = {k: v.double() for k, v in p.items()}
    m = {k: torch.zeros_like(v) for k, v in p.items()}
    v2 = {k: torch.zeros_like(v) for k, v in p.items()}
    b, losses = case["batch"], []
    gelu = lambda z: 0.5 * z * (1.0 + torch.erf(z / math.sqrt(2.0)))  # noqa: E731
    dgelu = lambda z: (0.5 * (1.0 + torch.erf(z / math.sqrt(2.0)))  # noqa: E731
                       + z * torch.exp(-0.5 * z * z) / math.sqrt(2.0 * math.pi))
    for k in range(case["steps"]):
        x, t = X[k * b:(k + 1) * b].double(), T[k * b:(k + 1) * b].double()
        z1 = x @ p["W1"] + p["b1"]
        h1 = gelu(z1)
        z2 = h1 @ p["W2"] + p["b2"]
        h2 = gelu(z2)
        d = h2 @ p["W3"] + p["b3"] - t
        losses.append(float((d * d).mean()))
        dy = 2.0 * d / d.numel()
        dz2 = (dy @ p["W3"].T) * dgelu(z2)
        dz1 = (dz2 @ p["W2"].T) * dgelu(z1)
        gr = dict(W1=x.T @ dz1, b1=dz1.sum(0), W2=h1.T @ dz2, b2=dz2.sum(0), W3=h2.T @ dy, b3=dy.sum(0))
        norm = math.sqrt(sum(float((q * q).sum()) for q in gr.values()))
        s = CLIP / norm if norm > CLIP else 1.0
        c1, c2 = 1.0 / (1.0 - 0.9 ** (k + 1)), 1.0 / (1.0 - 0.999 ** (k + 1))
        for q in p:
            gq = gr[q] * s
            m[q].mul_(0.9).add_(gq, alpha=0.1)
            v2[q].mul_(0.999).addcmul_(gq, gq, value=0.001)
            p[q] -= _rate(k) * (m[q] * c1) / ((v2[q] * c2).sqrt() + 1e-8)
    return dict(losses=torch.tensor(losses), **{k: v.cpu().numpy() for k, v in p.items()})
