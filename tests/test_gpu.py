"""GPU parity: every stage kernel and the full NR loop against the oracle.

Tolerances (floating point, FP64 unless stated):
  Ybus               bit-exact (same operation order, no FMA contraction)
  P, Q               |d| <= 1e-11 * (1 + max|P|, |Q|)  (complex form vs polar form)
  Jacobian           |d| <= 1e-11 * max|J|, identical sparsity pattern
  LU solve           |dx| <= 1e-9 * max|x|  (FP64; FP32 factor + 2 FP64 refinements)
  NR final state     |dV| <= 1e-6 pu, |dtheta| <= 1e-6 rad, same final PV->PQ set
"""
import os
import sys

import numpy as np
import pytest

from conftest import GOLDEN, IEEE, csr_to_dense

pytestmark = pytest.mark.gpu

CASES_SMALL = ["c14", "c118", "ieee14", "ieee57", "ieee118"]


def _path(cases, name):
    if name.startswith("ieee"):
        return os.path.join(IEEE, name + ".cdf")
    if name in ("c14", "c118"):
        return os.path.join(GOLDEN, name + ".cdf")
    return cases.path(name)


def _say(*a):
    print("[gpu]", *a, flush=True)
    sys.stdout.flush()


def _solver(pf, net, **kw):
    o = pf.options(tolerancia=1e-8, no_max_iter=100, **kw)
    return pf.Solver(net, o)


def _rand_state(net, seed):
    rng = np.random.default_rng(seed)
    V = 1.0 + 0.05 * rng.standard_normal(net.nB)
    th = 0.2 * rng.standard_normal(net.nB)
    return V, th


def _limq(net, seed):
    rng = np.random.default_rng(seed)
    return rng.random(net.nPV) < 0.3


@pytest.mark.parametrize("name", CASES_SMALL + ["c1888"])
def test_ybus_bitexact(pf, oracle, cases, name):
    p = _path(cases, name)
    _say("ybus", name)
    s = _solver(pf, pf.Network(p))
    rp, ci, y = s.ybus()
    rpo, cio, yo = oracle.Case(p).ybus()
    assert np.array_equal(rp, rpo) and np.array_equal(ci, cio)
    assert np.array_equal(y.real, yo.real) and np.array_equal(y.imag, yo.imag)


@pytest.mark.parametrize("name", CASES_SMALL + ["c1888"])
def test_pq(pf, oracle, cases, name):
    p = _path(cases, name)
    _say("pq", name)
    net = pf.Network(p)
    s = _solver(pf, net)
    rp, ci, y = oracle.Case(p).ybus()
    for seed in range(3):
        V, th = _rand_state(net, seed)
        P, Q = s.pq(V, th)
        Po, Qo = oracle.pq(rp, ci, y, V, th)
        scale = 1 + max(np.abs(Po).max(), np.abs(Qo).max())
        assert np.abs(P - Po).max() <= 1e-11 * scale
        assert np.abs(Q - Qo).max() <= 1e-11 * scale


@pytest.mark.parametrize("name", ["c14", "ieee57", "ieee118", "c1888"])
def test_flows(pf, oracle, cases, name):
    """Reported branch flows (the reference's formula and lookups) on the GPU
    against the oracle: at random states through the stage entry point, and at
    the solver's own answer.  Tolerance 1e-11 x (1 + max|flow|): the GPU's sin
    and cos are not the host's."""
    p = _path(cases, name)
    _say("flows", name)
    net = pf.Network(p)
    oc = oracle.Case(p)
    s = _solver(pf, net)
    for seed in range(2):
        V, th = _rand_state(net, seed)
        got = s.flows(V, th)
        ref = oc.flows(V, th)
        scale = 1 + max(np.abs(r).max() for r in ref)
        for g, e in zip(got, ref):
            assert np.abs(g - e).max() <= 1e-11 * scale
    s.reset()   # the stage calls left a random state on the device
    r = s.solve()
    assert r["converged"]
    V, th, _ = s.state()
    got = s.flows()
    ref = oc.flows(V, th)
    scale = 1 + max(np.abs(x).max() for x in ref)
    for g, e in zip(got, ref):
        assert np.abs(g - e).max() <= 1e-11 * scale


@pytest.mark.parametrize("name", ["c14", "c118", "ieee118"])
def test_mismatch(pf, oracle, cases, name):
    p = _path(cases, name)
    _say("mismatch", name)
    net = pf.Network(p)
    s = _solver(pf, net)
    oc = oracle.Case(p)
    rp, ci, y = oc.ybus()
    for seed in range(3):
        V, th = _rand_state(net, seed)
        lq = _limq(net, seed)
        ql = net.Qliq.copy()
        ql[net.pv[lq]] = 0.1 * (seed + 1)
        g, m = s.mismatch(V, th, lq, ql)
        Po, Qo = oracle.pq(rp, ci, y, V, th)
        pqlim = np.sort(np.concatenate([net.pq, net.pv[lq]]))
        go = oracle.mismatch(net.nB, net.slack, net.Pliq, ql, Po, Qo, pqlim)
        assert g.shape == go.shape
        assert np.abs(g - go).max() <= 1e-11 * (1 + np.abs(go).max())
        assert abs(m - np.abs(go).max()) <= 1e-11 * (1 + np.abs(go).max())


@pytest.mark.parametrize("name", ["c14", "c118", "ieee118", "c944"])
def test_jacobian(pf, oracle, cases, name):
    p = _path(cases, name)
    _say("jacobian", name)
    net = pf.Network(p)
    s = _solver(pf, net)
    oc = oracle.Case(p)
    rp, ci, y = oc.ybus()
    for seed in range(2):
        V, th = _rand_state(net, seed)
        lq = _limq(net, seed)
        rpJ, cJ, vJ = s.jacobian(V, th, lq)
        Po, Qo = oracle.pq(rp, ci, y, V, th)
        pqlim = np.sort(np.concatenate([net.pq, net.pv[lq]]))
        rpo, co, vo = oracle.jacobian(net.nB, net.slack, rp, ci, y, V, th, Po, Qo, pqlim)
        assert np.array_equal(rpJ, rpo) and np.array_equal(cJ, co)
        assert np.abs(vJ - vo).max() <= 1e-11 * np.abs(vo).max()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("name", ["c14", "c118", "ieee118", "c1888"])
def test_lu_solve(pf, oracle, cases, name, precision):
    p = _path(cases, name)
    _say("lu_solve", name, precision)
    net = pf.Network(p)
    s = _solver(pf, net, precision=pf.MIXED if precision == "mixed" else pf.FP64)
    oc = oracle.Case(p)
    rp, ci, y = oc.ybus()
    V = 1.0 + 0.01 * np.random.default_rng(1).standard_normal(net.nB)
    th = 0.05 * np.random.default_rng(2).standard_normal(net.nB)
    lq = _limq(net, 3)
    Po, Qo = oracle.pq(rp, ci, y, V, th)
    pqlim = np.sort(np.concatenate([net.pq, net.pv[lq]]))
    rpo, co, vo = oracle.jacobian(net.nB, net.slack, rp, ci, y, V, th, Po, Qo, pqlim)
    n = len(rpo) - 1
    b = np.random.default_rng(4).standard_normal(n)
    x = s.lu_solve(V, th, lq, b)
    xr = oracle.sparse_solve(rpo, co, vo, b)
    if n <= 1000:
        xr2 = np.linalg.solve(csr_to_dense(rpo, co, vo, n), b)
        assert np.abs(xr - xr2).max() <= 1e-10 * np.abs(xr2).max()
    assert np.abs(x - xr).max() <= 1e-9 * np.abs(xr).max()


@pytest.mark.parametrize("name", ["c14", "c118", "c944"])
def test_limits(pf, oracle, cases, name):
    p = _path(cases, name)
    _say("limits", name)
    net = pf.Network(p)
    s = _solver(pf, net, lim_inj_reat=1)
    oc = oracle.Case(p)
    rng = np.random.default_rng(11)
    for trial in range(4):
        V = net.V.copy()
        V[net.pv] = net.Vset + rng.choice([-2e-4, 0.0, 2e-4], net.nPV)
        span = net.Qmax - net.Qmin
        qg = net.Qmin + span * rng.uniform(-0.3, 1.3, net.nPV)
        Q = np.zeros(net.nB)
        Q[net.pv] = qg - net.Qload[net.pv]
        lq = rng.random(net.nPV) < 0.4
        ql = net.Qliq.copy()
        up = rng.random(net.nPV) < 0.5
        ql[net.pv[lq & up]] = (net.Qmax - net.Qload[net.pv])[lq & up]
        ql[net.pv[lq & ~up]] = (net.Qmin - net.Qload[net.pv])[lq & ~up]
        for mode in (0, 1):
            a = s.limits(mode, V, Q, lq, ql)
            b = oc.limits(mode, Q, V, lq, ql)
            assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1]) and a[2] == b[2]


def _nr_check(pf, oracle, p, lim, method, precision=0, graph=0, exact_iters=True, tol=1e-8):
    net = pf.Network(p)
    s = _solver(pf, net, lim_inj_reat=int(lim), metodo=method, precision=precision, use_graph=graph)
    r = s.solve()
    V, th, lq = s.state()
    o = oracle.Case(p).solve(tol=tol, lim=lim, reuse_symbolic=True)
    assert o["converged"]
    assert r["converged"], r
    assert r["max_mismatch"] <= tol
    assert np.abs(V - o["V"]).max() <= 1e-6
    assert np.abs(th - o["theta"]).max() <= 1e-6
    assert np.array_equal(lq, o["limQ"])
    if exact_iters:
        assert r["iterations"] == o["iterations"], (r, o["iterations"])
    else:
        assert abs(r["iterations"] - o["iterations"]) <= 3
    return r, o



@pytest.mark.parametrize("lim", [False, True])
@pytest.mark.parametrize("name", CASES_SMALL)
def test_nr_esparso(pf, oracle, cases, name, lim):
    if name == "ieee118" and lim:
        # does not converge in the reference logic: compared by
        # test_nr_ieee118_limits_trajectory instead
        return
    _say("nr esparso", name, lim)
    _nr_check(pf, oracle, _path(cases, name), lim, pf.ESPARSO)


def test_nr_ieee118_limits_trajectory(pf, oracle):
    """The bundled ieee118 case with Q limits does not converge under the
    reference rules: its PV->PQ switching cycles and the iterates grow to tens
    of pu, where 1e-13 changes the state at iteration 100.  The first 12
    iterations are well conditioned (a 1e-13 perturbation of the start moves
    them by < 1e-11) and hold three rounds of switching, back-switches
    included: there the FP64 GPU path must match the oracle state, the limQ
    set and the switch count.  At 100 iterations only the outcome is
    compared (not converged, 100 iterations, the switch count)."""
    p = os.path.join(IEEE, "ieee118.cdf")
    net = pf.Network(p)
    oc = oracle.Case(p)
    for mi in (12, 100):
        s = pf.Solver(net, pf.options(tolerancia=1e-8, no_max_iter=mi, lim_inj_reat=1))
        r = s.solve()
        V, th, lq = s.state()
        o = oc.solve(tol=1e-8, lim=True, max_iter=mi, reuse_symbolic=True)
        dv = float(np.abs(V - o["V"]).max())
        dt = float(np.abs(th - o["theta"]).max())
        _say("ieee118 limits", mi, "iters", r["iterations"], o["iterations"], "flips", r["n_switch_events"],
             o["n_switch_events"], "limited", int(lq.sum()), int(o["limQ"].sum()), "dV", dv, "dth", dt)
        assert not r["converged"] and not o["converged"]
        assert r["iterations"] == o["iterations"] == mi
        assert r["n_switch_events"] == o["n_switch_events"]
        if mi == 12:
            assert np.array_equal(lq, o["limQ"])
            assert dv <= 1e-6 and dt <= 1e-6


@pytest.mark.parametrize("name", ["c14", "c118", "c944"])
def test_nr_graph(pf, oracle, cases, name):
    _say("nr graph", name)
    _nr_check(pf, oracle, _path(cases, name), True, pf.ESPARSO, graph=1)


@pytest.mark.parametrize("name", ["c14", "c118", "c944"])
def test_nr_mixed(pf, oracle, cases, name):
    _say("nr mixed", name)
    _nr_check(pf, oracle, _path(cases, name), True, pf.ESPARSO, precision=pf.MIXED, graph=1,
              exact_iters=False)


@pytest.mark.parametrize("name", ["c14", "c118"])
def test_nr_denso(pf, oracle, cases, name):
    _say("nr denso", name)
    _nr_check(pf, oracle, _path(cases, name), True, pf.DENSO)


@pytest.mark.parametrize("name", ["c14", "c118", "c944"])
def test_nr_hibrido(pf, oracle, cases, name):
    _say("nr hibridoC", name)
    _nr_check(pf, oracle, _path(cases, name), True, pf.HIBRIDO_C)


@pytest.mark.parametrize("metodo", ["hibridoA", "hibridoB"])
@pytest.mark.parametrize("name", ["c14", "c118"])
def test_nr_hibrido_ab(pf, oracle, cases, name, metodo):
    """The GPU build's hibridoA (sparse path) and hibridoB (sparse Jacobian
    made dense, dense LU) solve like the oracle, in the same iterations."""
    _say("nr", metodo, name)
    _nr_check(pf, oracle, _path(cases, name), True, pf.HIBRIDO_A if metodo == "hibridoA" else pf.HIBRIDO_B)


def test_nr_15104(pf, oracle, cases):
    p = cases.path("c15104")
    _say("nr 15104 fp64 graph")
    r, o = _nr_check(pf, oracle, p, True, pf.ESPARSO, graph=1)
    _say("nr 15104 mixed graph", r["solve_ms"])
    r2, _ = _nr_check(pf, oracle, p, True, pf.ESPARSO, precision=pf.MIXED, graph=1, exact_iters=False)
    _say("15104 ms fp64", r["solve_ms"], "mixed", r2["solve_ms"])


def test_nr_not_converged_and_reset(pf, cases):
    net = pf.Network(os.path.join(GOLDEN, "c118.cdf"))
    s = _solver(pf, net, lim_inj_reat=1)
    s.opts.no_max_iter = 1
    s2 = pf.Solver(net, pf.options(tolerancia=1e-8, no_max_iter=1, lim_inj_reat=1))
    r = s2.solve()
    assert r["status"] == pf.PF_NOT_CONVERGED and not r["converged"] and r["iterations"] == 1
    r = s.solve()
    assert r["converged"]
    V1 = s.state()[0]
    s.reset()
    r2 = s.solve()
    assert r2["converged"] and r2["iterations"] == r["iterations"]
    assert np.array_equal(s.state()[0], V1)


@pytest.mark.parametrize("variant", ["eager", "graph", "mixed", "denso", "hibridoC", "batch"])
def test_nr_traced_limits(pf, oracle, variant):
    """The 3-bus case whose switch at iteration 1 and back-switch at
    iteration 2 are traced by hand in test_oracle.py: every solver path takes
    the same decisions at the same passes and keeps the back-switched |V|."""
    p = os.path.join(GOLDEN, "c3_limits.cdf")
    net = pf.Network(p)
    o = oracle.Case(p).solve(tol=1e-8, lim=True, reuse_symbolic=True)
    _say("traced limits", variant)
    if variant == "batch":
        b = pf.Batch([net], pf.options(tolerancia=1e-8, no_max_iter=100, lim_inj_reat=1))
        b.set_scenarios(np.zeros(1, np.int32), net.Pliq, net.Qliq, net.Qload)
        b.solve()
        V, th, it, cv, mm = b.results()
        lq, fl = b.limq()
        r = {"iterations": int(it[0]), "converged": bool(cv[0]), "n_switch_events": int(fl[0])}
        lq = lq[0]
    else:
        kw = {"eager": {}, "graph": {"use_graph": 1}, "mixed": {"use_graph": 1, "precision": pf.MIXED},
              "denso": {"metodo": pf.DENSO}, "hibridoC": {"metodo": pf.HIBRIDO_C}}[variant]
        s = _solver(pf, net, lim_inj_reat=1, **kw)
        r = s.solve()
        V, th, lq = s.state()
    assert r["converged"] and o["converged"]
    assert r["iterations"] == o["iterations"] == 4
    assert r["n_switch_events"] == o["n_switch_events"] == 2
    assert np.array_equal(lq, o["limQ"])
    assert np.abs(V - o["V"]).max() <= 1e-9 and np.abs(th - o["theta"]).max() <= 1e-9


@pytest.mark.parametrize("name", ["ieee14", "ieee30", "ieee57", "c118", "c944"])
def test_dense_lu_solve(pf, oracle, cases, name):
    """metodo denso's LU at unknown counts around its panels of 32 columns (26
    to 234) and in its panels of 8 (1,886), whose rows sit four per thread:
    backward error within n times the rounding unit times the growth that
    partial pivoting shows in practice."""
    p = _path(cases, name)
    _say("dense lu_solve", name)
    net = pf.Network(p)
    s = _solver(pf, net, metodo=pf.DENSO)
    oc = oracle.Case(p)
    rp, ci, y = oc.ybus()
    V = 1.0 + 0.01 * np.random.default_rng(1).standard_normal(net.nB)
    th = 0.05 * np.random.default_rng(2).standard_normal(net.nB)
    lq = _limq(net, 3)
    Po, Qo = oracle.pq(rp, ci, y, V, th)
    pqlim = np.sort(np.concatenate([net.pq, net.pv[lq]]))
    rpo, co, vo = oracle.jacobian(net.nB, net.slack, rp, ci, y, V, th, Po, Qo, pqlim)
    n = len(rpo) - 1
    J = csr_to_dense(rpo, co, vo, n)
    b = np.random.default_rng(4).standard_normal(n)
    x = s.lu_solve(V, th, lq, b)
    r = np.abs(J @ x - b).max()
    assert r <= 10 * n * 2.0 ** -53 * (np.abs(J).sum(1).max() * np.abs(x).max() + np.abs(b).max())


def test_dense_lu_singular(pf, cases):
    """A column without a finite pivot ends the dense solve as singular."""
    net = pf.Network(_path(cases, "c118"))
    s = _solver(pf, net, metodo=pf.DENSO)
    V = np.ones(net.nB)
    V[net.pq[3]] = np.nan
    with pytest.raises(pf.PfError) as e:
        s.lu_solve(V, np.zeros(net.nB), None, np.ones(net.nB - 1 + net.nPQ))
    assert e.value.status == pf.PF_SINGULAR


@pytest.mark.parametrize("copies,precision", [(1, "fp64"), (8, "fp64"), (8, "mixed"), (24, "mixed"), (40, "fp64"),
                                              (128, "fp64"), (128, "mixed")])
def test_lu_solve_dense_tops(pf, synth, tmp_path, copies, precision):
    """The sparse factor over networks whose dense tops take each tile of the
    register inverse: the FP64 residual of a solve, in the binding's own
    Jacobian, to the accuracy of FP64 and of FP32 with two FP64 refinements."""
    known = {1: synth.case118, 8: synth.case944, 128: synth.case15104}
    path = str(tmp_path / "net.cdfx")
    synth.write_cdf(known[copies]() if copies in known else synth.multi_copy(copies, 118000, 2 * copies, copies),
                    path, wide=True)
    net = pf.Network(path)
    _say("dense top", copies, precision, pf.SymbolicProbe(net).chain)
    s = _solver(pf, net, precision=pf.MIXED if precision == "mixed" else pf.FP64)
    V = 1.0 + 0.01 * np.random.default_rng(1).standard_normal(net.nB)
    th = 0.05 * np.random.default_rng(2).standard_normal(net.nB)
    rp, cj, v = s.jacobian(V, th, None)
    n = len(rp) - 1
    b = np.random.default_rng(4).standard_normal(n)
    x = s.lu_solve(V, th, None, b)
    r = np.zeros(n)
    np.add.at(r, np.repeat(np.arange(n), np.diff(rp)), v * x[cj])
    assert np.abs(r - b).max() <= 1e-9 * np.abs(v).max() * np.abs(x).max()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("name", ["c14", "ieee57", "c118", "ieee118"])
def test_nr_one_workgroup(pf, cases, name, precision):
    """Networks that one CU holds take the whole loop in one workgroup; with stage timing on, the
    kernels across the GPU run.  Both take the same Newton steps, so after each pass count the
    states agree to the rounding of the steps: within 1e-9 in FP64, the FP32 factors with one
    refinement leave about (100 * 6e-8)^2 of a step, 1e-7 after the passes here.
    """
    tol = 1e-9 if precision == "fp64" else 1e-7
    net = pf.Network(_path(cases, name))
    for lim in (0, 1):
        for max_iter in (0, 1, 3, 4):
            both = []
            for timing in (False, True):
                s = pf.Solver(net, pf.options(tolerancia=1e-8, no_max_iter=max_iter, lim_inj_reat=lim, refine_steps=1,
                                              precision=pf.MIXED if precision == "mixed" else pf.FP64))
                pf.lib().pf_solver_set_timing(s.h, int(timing))
                r = [s.solve(), s.solve()]          # from the start, and on from where that one ended
                both.append((r, s.state(), np.concatenate(s.flows())))
            (ra, sa, fa), (rb, sb, fb) = both
            for x, y in zip(ra, rb):
                for k in ("status", "iterations", "converged", "singular", "n_switch_events"):
                    assert x[k] == y[k], (name, lim, max_iter, k, x, y)
            assert np.abs(sa[0] - sb[0]).max() <= tol and np.abs(sa[1] - sb[1]).max() <= tol
            assert np.array_equal(sa[2], sb[2])
            assert np.abs(fa - fb).max() <= 1e4 * tol     # branch admittances up to some 1e3


def test_nr_one_workgroup_singular(pf, cases):
    """A flat zero voltage has no pivot: both paths say so after the same pass."""
    net = pf.Network(_path(cases, "c14"))
    got = []
    for timing in (False, True):
        s = pf.Solver(net, pf.options(tolerancia=1e-8, no_max_iter=10))
        pf.lib().pf_solver_set_timing(s.h, int(timing))
        s.set_state(np.zeros(net.nB), np.zeros(net.nB))
        r = s.solve()
        got.append((r["status"], r["iterations"], r["converged"], r["singular"]))
    assert got[0] == got[1] and got[0][3]


@pytest.mark.parametrize("precision,refine", [("fp64", 1), ("mixed", 0), ("mixed", 1), ("mixed", 2)])
def test_nr_head_in_one_launch(pf, cases, precision, refine):
    """Stage timing runs P/Q, limits, mismatch and decision one by one; without it one launch does the first
    three and one the decision, and the last correction is added where the state is updated.  Same bits."""
    net = pf.Network(_path(cases, "c944"))
    for lim in (0, 1):
        got = []
        for timing in (False, True):
            s = pf.Solver(net, pf.options(tolerancia=1e-6, no_max_iter=40, lim_inj_reat=lim, refine_steps=refine,
                                          precision=pf.MIXED if precision == "mixed" else pf.FP64))
            pf.lib().pf_solver_set_timing(s.h, int(timing))
            r = s.solve()
            got.append([r[k] for k in ("status", "iterations", "converged", "n_switch_events", "max_mismatch")]
                       + [x.tobytes() for x in s.state()])
        assert got[0] == got[1] and got[0][2]


@pytest.mark.parametrize("name,precision,metodo", [("c944", "fp64", "ESPARSO"), ("c944", "mixed", "ESPARSO"),
                                                   ("c118", "fp64", "DENSO")])
def test_nr_singular_with_a_pass_ahead(pf, cases, name, precision, metodo):
    """The host queues a pass before it has read the last one's outcome; behind a pass whose pivot failed
    nothing runs, so outcome and state are those of the solver that waits (stage timing)."""
    net = pf.Network(_path(cases, name))
    got = []
    for timing in (False, True):
        s = pf.Solver(net, pf.options(tolerancia=1e-8, no_max_iter=10, metodo=getattr(pf, metodo),
                                      precision=pf.MIXED if precision == "mixed" else pf.FP64))
        pf.lib().pf_solver_set_timing(s.h, int(timing))
        s.set_state(np.zeros(net.nB), np.zeros(net.nB))
        r = s.solve()
        got.append([r[k] for k in ("status", "iterations", "converged", "singular")] + [x.tobytes() for x in s.state()])
    assert got[0] == got[1] and got[0][3]


def test_state_read_by_several_threads(pf, cases):
    """Threads that read one solver's state at once each get all of it."""
    import threading
    net = pf.Network(_path(cases, "c944"))
    s = pf.Solver(net, pf.options(tolerancia=1e-8, no_max_iter=20))
    s.solve(check=True)
    want, got = s.state(), []

    def read():
        for _ in range(20):
            got.append(s.state())

    threads = [threading.Thread(target=read) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(got) == 80
    assert all(np.array_equal(x, y) for g in got for x, y in zip(want, g))


@pytest.mark.parametrize("name,precision,metodo", [("c14", "fp64", "ESPARSO"), ("c118", "mixed", "ESPARSO"),
                                                   ("c944", "fp64", "ESPARSO"), ("c944", "mixed", "ESPARSO"),
                                                   ("c118", "fp64", "DENSO"), ("c118", "fp64", "HIBRIDO_C")])
def test_nr_singular_keeps_the_state(pf, cases, name, precision, metodo):
    """A failed pivot ends the solve alike however its passes run (in one workgroup, launched one by one,
    as a replayed graph, with stage timing): after the same pass, the state as it was before that step."""
    net = pf.Network(_path(cases, name))
    V0, th0 = np.zeros(net.nB), np.linspace(-0.1, 0.1, net.nB)
    for graph in (0, 1):
        for timing in (False, True):
            s = pf.Solver(net, pf.options(tolerancia=1e-8, no_max_iter=10, use_graph=graph,
                                          metodo=getattr(pf, metodo),
                                          precision=pf.MIXED if precision == "mixed" else pf.FP64))
            pf.lib().pf_solver_set_timing(s.h, int(timing))
            s.set_state(V0, th0)
            r = s.solve()
            _say(name, precision, metodo, "graph", graph, "timing", timing, r)
            assert (r["status"], r["iterations"], r["converged"], r["singular"]) == (pf.PF_SINGULAR, 1, False, True)
            V, th, _ = s.state()
            assert np.array_equal(V, V0) and np.array_equal(th, th0)


@pytest.mark.parametrize("name", ["ieee14", "ieee30", "ieee57"])
def test_dense_lu_solve_rounding(pf, cases, name):
    """metodo denso rounds as plain elimination with partial pivoting does: every multiply-add and every
    quotient once.  The same steps on the host in exact rational arithmetic, rounded after each, give the
    same bits (26, 58 and 112 unknowns: less than a panel of 32, two, four)."""
    from fractions import Fraction as F
    net = pf.Network(_path(cases, name))
    s, pr = _solver(pf, net, metodo=pf.DENSO), pf.SymbolicProbe(net)
    V = 1.0 + 0.01 * np.random.default_rng(1).standard_normal(net.nB)
    th = 0.05 * np.random.default_rng(2).standard_normal(net.nB)
    rp, cj, v = s.jacobian(V, th, None)
    J = csr_to_dense(rp, cj, v, len(rp) - 1)
    b = np.random.default_rng(4).standard_normal(len(J))
    # the blocked system, two unknowns a bus in elimination order; buses without a Q equation keep dV = 0
    bus = pr.perm + (pr.perm >= net.slack)
    place = {int(k): i for i, k in enumerate(np.sort(net.pq))}
    at = []
    for k in bus:
        at += [int(k) - (k > net.slack), net.nB - 1 + place[int(k)] if int(k) in place else -1]
    n = len(at)
    A = np.eye(n)
    kept = [i for i in range(n) if at[i] >= 0]
    A[np.ix_(kept, kept)] = J[np.ix_([at[i] for i in kept], [at[i] for i in kept])]
    A = [row + [float(b[at[i]]) if at[i] >= 0 else 0.0] for i, row in enumerate(A.tolist())]

    def fnma(l, u, a):
        return float(F(a) - F(l) * F(u)) if l and u else a

    for k in range(n):
        p = max(range(k, n), key=lambda i: (abs(A[i][k]), -i))
        A[k], A[p] = A[p], A[k]
        for i in range(k + 1, n):
            if A[i][k]:
                A[i][k] /= A[k][k]
                for c in range(k + 1, n + 1):
                    A[i][c] = fnma(A[i][k], A[k][c], A[i][c])
    x = [row[n] for row in A]
    for k in range(n - 1, -1, -1):
        x[k] /= A[k][k]
        for i in range(k):
            x[i] = fnma(A[i][k], x[k], x[i])
    want = np.zeros(len(J))
    want[[at[i] for i in kept]] = [x[i] for i in kept]
    assert np.array_equal(s.lu_solve(V, th, None, b), want)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_lu_solve_longest_dense_top(pf, synth, tmp_path, precision):
    """A complete graph of 120 buses: a dense top of 101 nodes in FP64 and 119 in FP32, past the 96 that
    square tiles of the register inverse cover.  Accuracy as for the shorter ones."""
    rng = np.random.default_rng(120)
    nb = 120
    buses = [synth.Bus(i + 1, 3 if i == 0 else 0, pload=round(float(rng.uniform(0, 2)), 1) * (i > 0),
                       qload=round(float(rng.uniform(0, 0.5)), 1) * (i > 0)) for i in range(nb)]
    branches = [synth.Branch(i + 1, j + 1, 1.0, round(float(rng.uniform(5, 9)), 3))
                for i in range(nb) for j in range(i + 1, nb)]
    path = str(tmp_path / "dense.cdf")
    synth.write_cdf(synth.Case(buses, branches), path)
    net = pf.Network(path)
    assert pf.SymbolicProbe(net).chain[0] == 101
    s = _solver(pf, net, precision=pf.MIXED if precision == "mixed" else pf.FP64)
    V = 1.0 + 0.01 * np.random.default_rng(1).standard_normal(nb)
    th = 0.05 * np.random.default_rng(2).standard_normal(nb)
    rp, cj, v = s.jacobian(V, th, None)
    n = len(rp) - 1
    b = np.random.default_rng(4).standard_normal(n)
    x = s.lu_solve(V, th, None, b)
    r = np.zeros(n)
    np.add.at(r, np.repeat(np.arange(n), np.diff(rp)), v * x[cj])
    assert np.abs(r - b).max() <= 1e-9 * np.abs(v).max() * np.abs(x).max()
