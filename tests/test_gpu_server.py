"""Request server (fmmhip_server_*): every request in a concurrent mix returns what the single
call returns.

Bars: fmm! requests bit-identical to fmm!(system) through one evaluation (every FMM pass is
deterministic: integer atomics only); FastGaussSeidel solves within 1e-10 relative of the single
solve with the same sweep count (a sweep level adds right-hand-side updates with floating-point
atomics, whose order varies run to run). The single calls are themselves pinned against the
oracle by the parity and FastGaussSeidel tests."""
import ctypes

import numpy as np
import pytest

import fastmultipole_amd as F
from fastmultipole_amd import _lib, workloads as W

pytestmark = pytest.mark.gpu


class _Rows:
    """A system given by its source rows and built-in kernel (duck-typed like the host systems)."""

    def __init__(self, kernel, rows):
        self.fmm_kernel = kernel
        self.rows = np.ascontiguousarray(rows, dtype=np.float64)

    def source_buffer(self):
        return self.rows


FMM_CASES = [
    ("sources-20k", _lib.POINT_SOURCE, lambda: W.uniform_sources(20000, seed=11), dict(expansion_order=5)),
    ("ring-8k-p10", _lib.POINT_VORTEX, lambda: W.vortex_ring(8000, seed=12), dict(expansion_order=10, leaf_size=40)),
    ("plummer-30k-hess", _lib.POINT_SOURCE, lambda: W.plummer_sources(30000, seed=13),
     dict(expansion_order=6, scalar_potential=True, hessian=True)),
    ("sources-500", _lib.POINT_SOURCE, lambda: W.uniform_sources(500, seed=14), dict(expansion_order=4, leaf_size=10)),
    ("dipoles-4k", _lib.POINT_DIPOLE, lambda: W.uniform_dipoles(4000, seed=15), dict(expansion_order=7)),
]
SOLVE_CASES = [
    ("quads-sphere", lambda: W.sphere_panels(10, quads=True), dict(leaf_size=30, expansion_order=6), -1.0),
    ("tris-sphere-normal", lambda: W.sphere_panels(8, quads=False),
     dict(leaf_size=20, expansion_order=6, influence=_lib.INFLUENCE_NORMAL_GRADIENT), None),
]


def _single_fmm(kernel, rows, kw):
    ev = F.Evaluation()
    ev.set_systems(kernel, None, rows)
    ls = kw.get("leaf_size", 20)
    opt = F.make_options(kw.get("expansion_order", 5), ls, ls, 0.4, None, True, None,
                         kw.get("scalar_potential", False), True, kw.get("hessian", False))
    ev.fmm(opt)
    out = ev.targets()
    ev.close()
    return out


def _solve_inputs(gen, ext_value):
    rows, kind = gen()
    n = len(rows)
    ext = np.full(n, ext_value) if ext_value is not None else -np.random.default_rng(3).standard_normal(n)
    return kind, rows, ext


def _single_solve(kind, rows, ext, kw):
    s = _Rows(kind, rows)
    fgs = F.FastGaussSeidel(s, expansion_order=kw.get("expansion_order", 4), leaf_size=kw.get("leaf_size", 30),
                            influence=kw.get("influence", _lib.INFLUENCE_POTENTIAL))
    strengths, targets, sweeps, _ = fgs.solve(ext, max_iterations=6, tolerance=1e-12)
    fgs.ev.close()
    return strengths, targets, sweeps


def _submit_all(server, fmm_inputs, solve_inputs):
    tickets = []
    for (name, kernel, rows, kw) in fmm_inputs:
        tickets.append(("fmm", name, server.submit_fmm(_Rows(kernel, rows), **kw)))
    for (name, kind, rows, ext, kw) in solve_inputs:
        skw = {k: v for k, v in kw.items()}
        tickets.append(("solve", name, server.submit_solve(_Rows(kind, rows), ext, max_iterations=6,
                                                           tolerance=1e-12, **skw)))
    return tickets


def test_server_mix_matches_single_calls():
    print("[gpu] server mix: single calls", flush=True)
    fmm_inputs = [(name, k, gen(), kw) for name, k, gen, kw in FMM_CASES]
    solve_inputs = []
    for name, gen, kw, ev in SOLVE_CASES:
        kind, rows, ext = _solve_inputs(gen, ev)
        solve_inputs.append((name, kind, rows, ext, kw))
    want_fmm = {name: _single_fmm(k, rows, kw) for name, k, rows, kw in fmm_inputs}
    want_solve = {name: _single_solve(kind, rows, ext, kw) for name, kind, rows, ext, kw in solve_inputs}
    print("[gpu] server mix: 4 slots, two rounds of every request", flush=True)
    with F.Server(n_slots=4, hbm_budget_bytes=32 * 2**30) as server:
        tickets = _submit_all(server, fmm_inputs, solve_inputs)
        tickets += _submit_all(server, fmm_inputs[::-1], solve_inputs[::-1])
        for kind, name, t in tickets:
            targets, strengths, st = server.wait(t)
            assert st["latency_ms"] >= st["run_ms"] > 0.0
            if kind == "fmm":
                assert st["status"] == _lib.FMMHIP_OK and st["error_success"] == 1, (name, st)
                np.testing.assert_array_equal(targets, want_fmm[name], err_msg=name)
            else:
                s_ref, t_ref, sw_ref = want_solve[name]
                assert st["sweeps"] == sw_ref, name
                # six sweeps never reach the 1e-12 residual: results delivered, tolerance missed
                assert st["converged"] == 0 and st["status"] == _lib.FMMHIP_ETOL, (name, st)
                assert np.abs(strengths - s_ref).max() <= 1e-10 * np.abs(s_ref).max(), name
                for lo, hi in ((3, 4), (4, 7)):
                    sc = np.abs(t_ref[:, lo:hi]).max()
                    assert np.abs(targets[:, lo:hi] - t_ref[:, lo:hi]).max() <= 1e-10 * sc, (name, lo)
        stats = server.stats()
        assert stats["completed"] == len(tickets) and stats["queued"] == 0 and stats["running"] == 0
        assert 0.0 < stats["p50_ms"] <= stats["p99_ms"] <= stats["span_ms"]


def test_server_budget_serialises_requests():
    """A budget below every request's footprint runs one request at a time (the oldest first)
    and still completes all of them."""
    print("[gpu] server tiny budget", flush=True)
    rows = [W.uniform_sources(n, seed=21 + i) for i, n in enumerate((3000, 6000, 1500))]
    want = [_single_fmm(_lib.POINT_SOURCE, r, dict(expansion_order=4)) for r in rows]
    with F.Server(n_slots=3, hbm_budget_bytes=1.0) as server:
        ts = [server.submit_fmm(_Rows(_lib.POINT_SOURCE, r), expansion_order=4) for r in rows]
        spans = []
        for t, w in zip(ts, want):
            targets, _, st = server.wait(t)
            np.testing.assert_array_equal(targets, w)
            spans.append((st["start_ms"], st["end_ms"]))
    spans.sort()
    for (s0, e0), (s1, _) in zip(spans, spans[1:]):
        assert s1 >= e0, spans     # no overlap: each starts after the previous ended


def _free_bytes():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert _lib.load().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0   # the runtime the library is linked to
    return free.value


def test_admission_estimate_counts_the_m2l_workspace_and_the_panel_records(monkeypatch):
    """The estimate's share of the M2L's partial expansions is at least what they take: the difference of two orders' estimates,
    the lower without such a workspace, less the difference of their two trees' expansions. A panel request's is
    its rows and records above a point request's."""
    print("[gpu] server admission estimate", flush=True)
    n, leaf, mac = 400000, 20, 0.5
    rows = W.uniform_vortices(n, seed=31)
    with F.Server(n_slots=1) as server:
        def estimate(kernel, r, **kw):
            return server.wait(server.submit_fmm(_Rows(kernel, r), multipole_acceptance=mac, **kw))[2]["footprint_bytes"]
        fp = {p: estimate(_lib.POINT_VORTEX, rows, leaf_size=leaf, expansion_order=p) for p in (4, 12)}
        panels, _ = W.sphere_panels(20, quads=True)
        points = estimate(_lib.POINT_SOURCE, W.uniform_sources(len(panels), seed=32), leaf_size=30)
        fp_panels = estimate(_lib.PANEL_SOURCE_QUAD, panels, leaf_size=30)
    ev = F.Evaluation()
    ev.set_systems(_lib.POINT_VORTEX, None, rows)
    for engine in ("wave", "mx"):   # the same handle: all other buffers have their size after the first
        monkeypatch.setenv("FMMHIP_M2L_KERNEL", engine)
        before = _free_bytes()
        ev.fmm(F.make_options(expansion_order=12, leaf_size_source=leaf, multipole_acceptance=mac))
        workspace = before - _free_bytes()
    ev.close()
    coefficients = lambda p: (p + 1) * (p + 2) // 2
    branches = 2.3 * n / leaf + 64
    assert workspace > 1e9
    assert fp[12] - fp[4] - 2 * branches * 32 * (coefficients(12) - coefficients(4)) >= workspace
    assert fp_panels - points >= len(panels) * 8 * ((17 - 5) + 35)


def test_server_rejects_bad_requests():
    with F.Server(n_slots=1) as server:
        with pytest.raises(ValueError):
            server.submit_solve(_Rows(_lib.POINT_SOURCE, W.uniform_sources(100, seed=1)), np.zeros(5))
        t = server.submit_solve(_Rows(_lib.POINT_VORTEX, W.vortex_ring(200, seed=1)), np.zeros(200))
        with pytest.raises(_lib.FmmHipError):
            server.wait(t)
    with pytest.raises(_lib.FmmHipError):
        F.Server(n_slots=0)


def test_server_reports_missed_tolerance():
    """A request whose tolerance cannot be met still delivers its results, with status FMMHIP_ETOL:
    an FMM at an order cap of 3 with a 1e-14 error tolerance (error_success false, as fmm! returns it)
    and a solve stopped after one sweep short of its residual tolerance; a reachable tolerance
    returns FMMHIP_OK."""
    print("[gpu] server missed tolerance", flush=True)
    rows = W.uniform_sources(4000, seed=31)
    tol_miss = dict(expansion_order=3, error_tolerance=F.PowerAbsoluteGradient(1e-14))
    tol_ok = dict(expansion_order=12, error_tolerance=F.PowerAbsoluteGradient(1e-3))
    ev = F.Evaluation()
    ev.set_systems(_lib.POINT_SOURCE, None, rows)
    st_single = ev.fmm(F.make_options(3, 20, 20, 0.4, None, True, F.PowerAbsoluteGradient(1e-14)))
    want = ev.targets()
    ev.close()
    assert st_single.error_success == 0 and st_single.pmax == 4
    prow, pkind = W.sphere_panels(8, quads=True)
    ext = np.full(len(prow), -1.0)
    with F.Server(n_slots=2) as server:
        t_miss = server.submit_fmm(_Rows(_lib.POINT_SOURCE, rows), **tol_miss)
        t_ok = server.submit_fmm(_Rows(_lib.POINT_SOURCE, rows), **tol_ok)
        t_solve = server.submit_solve(_Rows(pkind, prow), ext, max_iterations=1, tolerance=1e-30)
        targets, _, st = server.wait(t_miss)
        assert st["status"] == _lib.FMMHIP_ETOL and st["error_success"] == 0 and st["pmax"] == 4, st
        np.testing.assert_array_equal(targets, want)
        _, _, st = server.wait(t_ok)
        assert st["status"] == _lib.FMMHIP_OK and st["error_success"] == 1, st
        _, strengths, st = server.wait(t_solve)
        assert st["status"] == _lib.FMMHIP_ETOL and st["converged"] == 0 and st["sweeps"] == 1, st
        assert np.all(np.isfinite(strengths))


def test_server_batched_uneven_instances_match_oracle():
    """The batched-instances workload at test size: 32 independent systems with N log-uniform in
    [1e3, 5e3], even ones uniform-cube sources (potential + gradient, p 8, MAC 0.5), odd ones vortex rings
    (velocity + gradient, p 10, MAC 0.4), all submitted at once to 8 slots in both precision forms.
    Every request returns FMMHIP_OK; every FP64 result matches the oracle's fmm! to 1e-11 relative and
    every mixed-form result (FP32 nearfield) stays within 1e-5 of it."""
    import math
    from oracle import oracle as O
    print("[gpu] server batched uneven instances (32 systems)", flush=True)
    rng = np.random.default_rng(4)
    sizes = np.floor(np.exp(rng.uniform(math.log(1e3), math.log(5e3), 32))).astype(int)
    systems = []
    for i, n in enumerate(sizes):
        if i % 2 == 0:
            systems.append((_lib.POINT_SOURCE, W.uniform_sources(int(n), seed=500 + i),
                            dict(expansion_order=8, leaf_size=30, multipole_acceptance=0.5, scalar_potential=True)))
        else:
            systems.append((_lib.POINT_VORTEX, W.vortex_ring(int(n), seed=500 + i),
                            dict(expansion_order=10, leaf_size=40, multipole_acceptance=0.4)))
    with F.Server(n_slots=8) as server:
        tickets = [(i, prec, server.submit_fmm(_Rows(k, rows), precision=prec, **kw))
                   for prec in ("fp64", "mixed") for i, (k, rows, kw) in enumerate(systems)]
        results = {}
        for i, prec, t in tickets:
            targets, _, st = server.wait(t)
            assert st["status"] == _lib.FMMHIP_OK and st["error_success"] == 1, (i, prec, st)
            results[(i, prec)] = targets
    for i, (k, rows, kw) in enumerate(systems):
        okind = O.KIND_SOURCE if k == _lib.POINT_SOURCE else O.KIND_VORTEX
        ref = O.Run(okind, rows[:, :3], rows, p=kw["expansion_order"], leaf_size_source=kw["leaf_size"],
                    multipole_acceptance=kw["multipole_acceptance"],
                    scalar_potential=kw.get("scalar_potential", False)).fmm().targets()
        lo, hi = 4, 7
        sc = np.abs(ref[:, lo:hi]).max()
        e64 = np.abs(results[(i, "fp64")][:, lo:hi] - ref[:, lo:hi]).max() / sc
        e32 = np.abs(results[(i, "mixed")][:, lo:hi] - ref[:, lo:hi]).max() / sc
        assert e64 < 1e-11, (i, e64)
        assert e32 < 1e-5, (i, e32)


def test_server_batches_waiting_requests_like_single_calls():
    """FMM requests with the same kernel and options that wait together run as one batch evaluation. Two
    option sets (a relative tolerance some systems miss at p <= 10, and a fixed order) plus a solve are
    submitted at once to one worker: each request's targets are bit-identical to its own fmm! call, and its
    status, pmax and error_success are that call's. Requests that ran together share start and end times:
    with one worker and everything queued, at least one batch holds several requests, and no batch mixes
    the two option sets. With batch_requests=1 every request runs alone."""
    print("[gpu] server batching of waiting requests", flush=True)
    rel = dict(leaf_size=30, expansion_order=10, multipole_acceptance=0.5,
               error_tolerance=F.PowerRelativeGradient(1e-9))
    fixed = dict(leaf_size=20, expansion_order=6, multipole_acceptance=0.4)
    sizes = [3000, 1, 9000, 500, 20000, 2, 4000, 12000, 800, 6000]
    reqs = []
    for i, n in enumerate(sizes):
        rows = W.vortex_ring(n, seed=600 + i) if i % 2 == 0 else W.uniform_vortices(n, seed=600 + i)
        reqs.append((_Rows(_lib.POINT_VORTEX, rows), rel if i % 3 != 2 else fixed))

    def single(sysm, kw):
        ev = F.Evaluation()
        _, ev, *_ = F.fmm(sysm, evaluation=ev, update_target_systems=False, **kw)
        out, st = ev.targets(), ev.last_stats
        ev.close()
        return out, st.pmax, st.error_success

    singles = [single(s, kw) for s, kw in reqs]
    kind, srows, ext = _solve_inputs(SOLVE_CASES[0][1], SOLVE_CASES[0][3])
    for batch_requests in (64, 1):
        with F.Server(n_slots=1, batch_requests=batch_requests) as server:
            tickets = [server.submit_fmm(s, **kw) for s, kw in reqs]
            tsolve = server.submit_solve(_Rows(kind, srows), ext, **SOLVE_CASES[0][2])
            got = [server.wait(t) for t in tickets]
            server.wait(tsolve)
        groups = {}
        for i, ((out, _, st), (ref, pmax, ok)) in enumerate(zip(got, singles)):
            np.testing.assert_array_equal(out, ref, err_msg=f"request {i} (n={sizes[i]})")
            assert st["pmax"] == pmax and st["error_success"] == ok, (i, st, pmax, ok)
            assert st["status"] == (_lib.FMMHIP_OK if ok else _lib.FMMHIP_ETOL), (i, st)
            groups.setdefault((st["start_ms"], st["end_ms"]), []).append(i)
        sets = [{id(reqs[i][1]) for i in g} for g in groups.values()]
        assert all(len(s) == 1 for s in sets), groups
        if batch_requests == 1:
            assert all(len(g) == 1 for g in groups.values()), groups
        else:
            assert max(len(g) for g in groups.values()) > 1, groups
        print(f"[gpu] batch_requests={batch_requests}: groups {sorted(groups.values())}", flush=True)
