"""The work this library is used for, as cases that can be timed and compared.

A study solves power flows: one case file from scratch, one network again and
again as its injections move, or many perturbed scenarios of one or more
networks at once; the learned warm start is trained on such solutions and
writes starting points for the next batch.  Every kind below is one of these,
through the library's Python binding, on networks from 14 to 15,104 buses
(the ones the repository's tests and benchmark use; ``areas<k>``: k tied
118-bus areas).

Scenarios are a day's operating points: a system load level of 0.9 to 1.0 and
a per-bus factor clip(exp(0.1 N(0, 1)), 0.8, 1.2), dispatch following load.
All of them converge.  The mismatch left over at convergence is not among the
outputs: it is rounding noise below the tolerance.
"""
import ctypes
import functools
import importlib
import importlib.util
import math
import os
import sys
import tempfile

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "experience-of-using-gpu-in-power-flow-computation_amd")
TOL, MAX_ITER = 1e-8, 60
FOLGA = 1e-4        # tolerance of the reactive limits
HIDDEN, LAYERS = 512, 3


def _package():
    if "pfamd" not in sys.modules:
        spec = importlib.util.spec_from_file_location("pfamd", os.path.join(PKG, "__init__.py"),
                                                      submodule_search_locations=[PKG])
        m = importlib.util.module_from_spec(spec)
        sys.modules["pfamd"] = m
        spec.loader.exec_module(m)
    return sys.modules["pfamd"], importlib.import_module("pfamd.synth")


def listed():
    return [
        # the smallest call: a textbook network solved once more, default options
        dict(name="solve 14", kind="solve", net="case14", precision="fp64", graph=False, limits=True),
        # a case file solved once and reported, as the command line does it: analysis, solve, flows
        dict(name="report 118", kind="report", net="areas1", precision="fp64", limits=True),
        # the dense method (the reference's metodo = denso)
        dict(name="dense 118", kind="dense", net="areas1", limits=False),
        # a mid-size network followed through the day
        dict(name="solve 1888", kind="solve", net="areas16", precision="fp64", graph=True, limits=True),
        # the largest network: default options, and the fastest ones
        dict(name="solve 15104", kind="solve", net="areas128", precision="fp64", graph=False, limits=True),
        dict(name="solve 15104 mixed", kind="solve", net="areas128", precision="mixed", graph=True, limits=True),
        # a serving loop: a handful of scenarios in the caller's own GPU memory, nothing allocated
        dict(name="serve 24x57", kind="serve", net="ieee57", n=24, precision="fp64", limits=True),
        # a contingency-sized batch with default precision, a ragged count
        dict(name="batch 333x118", kind="batch", net="areas1", n=333, net2="", n2=0, precision="fp64", limits=True),
        # the benchmark's batch: many small scenarios beside fewer large ones
        dict(name="batch 2048x118 128x1888", kind="batch", net="areas1", n=2048, net2="areas16", n2=128,
             precision="mixed", limits=True),
        # the GPU full of large scenarios
        dict(name="batch 512x1888", kind="batch", net="areas16", n=512, net2="", n2=0, precision="mixed",
             limits=False),
        # inference straight into a batch's start, then the solve
        dict(name="warm 2048x944", kind="warm", net="areas8", n=2048, precision="mixed", limits=False),
        # training of the warm start on solved scenarios
        dict(name="train 944", kind="train", net="areas8", n=2048, batch=256),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["solve", "solve", "solve", "batch", "batch", "batch", "batch", "serve", "warm", "train",
                       "report", "dense"])
    precision, limits = rng.choice(["fp64", "mixed"]), rng.random() < 0.5
    small = ["case14", "ieee30", "ieee57"]
    if kind == "solve":
        net = rng.choice(small) if rng.random() < 0.2 else "areas%d" % _log(rng, 1, 120)
        return dict(kind=kind, net=net, precision=precision, graph=rng.random() < 0.5, limits=_limits(net, limits))
    if kind == "report":
        net = rng.choice(small) if rng.random() < 0.3 else "areas%d" % _log(rng, 1, 20)
        return dict(kind=kind, net=net, precision="fp64", limits=_limits(net, limits))
    if kind == "dense":
        net = rng.choice(small + ["ieee118", "areas2"])
        return dict(kind=kind, net=net, limits=_limits(net, limits))
    if kind == "serve":
        net = rng.choice(small + ["areas1", "areas2"])
        return dict(kind=kind, net=net, n=_log(rng, 4, 300), precision=precision, limits=_limits(net, limits))
    if kind == "batch":
        k = rng.choice([0, 0, 1, 1, 1, 2, 3, 5, 8, 12, 16])
        net = rng.choice(small) if k == 0 else "areas%d" % k
        n = _log(rng, 8, min(2048, 2048 // max(1, k)))
        c = dict(kind=kind, net=net, n=n, net2="", n2=0, precision=precision, limits=_limits(net, limits))
        if rng.random() < 0.3:
            c.update(net2="areas%d" % rng.choice([1, 4, 6, 9]), n2=_log(rng, 4, 64))
        return c
    k = rng.choice([1, 2, 4, 8])
    if kind == "warm":
        return dict(kind=kind, net="areas%d" % k, n=8 * _log(rng, 4, 200), precision="mixed", limits=False)
    return dict(kind=kind, net="areas%d" % k, n=_log(rng, 256, 2000), batch=8 * rng.choice([4, 9, 16, 25, 32]))


def _limits(net, limits):
    return limits and net != "ieee118"     # its published limits cycle: no method of this kind settles there


# ---------------------------------------------------------------- networks

@functools.lru_cache(maxsize=None)
def _network(name):
    """The network of a case, from a file as a user has it."""
    pf, synth = _package()
    if name.startswith("ieee"):
        return pf.Network(os.path.join(ROOT, "tests", "golden", "ieee", name + ".cdf"))
    d = os.path.join(tempfile.gettempdir(), "pf_cases_%d" % os.getuid())
    os.makedirs(d, exist_ok=True)
    path = os.path.join(d, name + ".cdfx")
    if not os.path.exists(path):
        k = 0 if name == "case14" else int(name[5:])
        known = {0: synth.case14, 1: synth.case118, 8: synth.case944, 16: synth.case1888, 128: synth.case15104}
        case = known[k]() if k in known else synth.multi_copy(k, 118000, 2 * k, k)
        own = "%s.%d.cdfx" % (path, os.getpid())
        synth.write_cdf(case, own, wide=True)
        os.replace(own, path)
    return pf.Network(path)


def _scenarios(net, n, seed):
    """n operating points of a network: net injections P, Q and the loads' Q, each [n, buses]."""
    rng = np.random.default_rng([seed, net.nB])
    f = np.clip(np.exp(0.1 * rng.standard_normal((n, net.nB))), 0.8, 1.2) * rng.uniform(0.9, 1.0, (n, 1))
    pv = np.zeros(net.nB, bool)
    pv[net.pv] = True
    p, q = net.Pload * f, net.Qload * f
    total = net.Pload.sum()
    ratio = p.sum(1, keepdims=True) / total if total else 1.0
    return np.where(pv, net.Pg * ratio, net.Pg) - p, net.Qg - q, q


def _inputs(case, seed):
    """(networks, network of each scenario, their injections)."""
    nets, n = [_network(case["net"])], [case.get("n", 1)]
    if case.get("net2"):
        nets.append(_network(case["net2"]))
        n.append(case["n2"])
    return nets, np.repeat(np.arange(len(nets), dtype=np.int32), n), [_scenarios(a, k, seed) for a, k in zip(nets, n)]


def _options(case):
    pf, _ = _package()
    mixed = case.get("precision") == "mixed"
    return pf.options(tolerancia=TOL, no_max_iter=MAX_ITER, lim_inj_reat=int(case["limits"]),
                      precision=pf.MIXED if mixed else pf.FP64, refine_steps=1, use_graph=int(case.get("graph", False)),
                      metodo=pf.DENSO if case["kind"] == "dense" else pf.ESPARSO)


def _features(net, P, Q):
    """The warm start's rows: injections and setpoints, padded to a multiple of 8."""
    vset = np.zeros(net.nB)
    vset[net.pv] = net.Vset
    vset[net.slack] = net.V[net.slack]
    X = np.zeros((len(P), -(-3 * net.nB // 8) * 8), np.float32)
    X[:, :3 * net.nB] = np.concatenate([P, Q, np.repeat(vset[None], len(P), 0)], 1)
    return X


def _rows(net, n, seed):
    """Solved-looking rows for training: features, and voltages that move with the injections
    (angles as in a DC power flow on a fixed operating point), with their normalisation."""
    P, Q, _ = _scenarios(net, n, seed)
    X = _features(net, P, Q)
    Y = np.zeros((n, -(-2 * net.nB // 8) * 8), np.float32)
    B = np.zeros((net.nB, net.nB))
    w = 1.0 / net.x
    np.add.at(B, (net.frm, net.to), -w)
    np.add.at(B, (net.to, net.frm), -w)
    np.add.at(B, (net.frm, net.frm), w)
    np.add.at(B, (net.to, net.to), w)
    keep = np.arange(net.nB) != net.slack
    S = np.linalg.inv(B[np.ix_(keep, keep)])
    Y[:, :net.nB] = 1.0
    Y[:, :net.nB][:, keep] = 1.0 + 0.1 * (Q[:, keep] - Q[:, keep].mean(0)) @ S
    Y[:, net.nB:2 * net.nB][:, keep] = P[:, keep] @ S
    return X, Y, (X.mean(0), X.std(0) + 1e-6, Y.mean(0), Y.std(0) + 1e-6)


# --------------------------------------------------------------- the calls

def prepare(case, seed):
    pf, _ = _package()
    kind = case["kind"]
    s = dict(kind=kind)
    if kind == "train":
        net = _network(case["net"])
        X, Y, norm = _rows(net, case["n"], seed)
        w = pf.WarmStart(X.shape[1], Y.shape[1], HIDDEN, LAYERS, seed=11)
        w.set_norm(*norm)
        return dict(s, w=w, X=X, Y=Y, batch=case["batch"])
    nets, net_of, inj = _inputs(case, seed)
    opts = _options(case)
    if kind == "report":
        return dict(s, net=nets[0], opts=opts, inj=[a[0] for a in inj[0]])
    if kind in ("solve", "dense"):
        solver = pf.Solver(nets[0], opts)
        solver.set_injections(*[a[0] for a in inj[0]])
        return dict(s, solver=solver)
    b = pf.Batch(nets, opts)
    P, Q, L = (np.concatenate([x[i].ravel() for x in inj]) for i in range(3))
    if kind == "serve":
        pv = sum(nets[i].nPV for i in net_of)
        gpu = [torch.from_numpy(a).cuda() for a in (net_of, P, Q, L)]
        out = [torch.zeros(k, dtype=t, device="cuda") for k, t in
               ((len(P), torch.float64), (len(P), torch.float64), (len(net_of), torch.int32),
                (len(net_of), torch.int32), (len(net_of), torch.float64), (pv, torch.uint8),
                (len(net_of), torch.int32))]
        return dict(s, b=b, n=len(net_of), gpu=gpu, out=out)
    b.set_scenarios(net_of, P, Q, L)
    s.update(b=b)
    if kind == "warm":
        # a network whose outputs stay near a known operating point
        net = nets[0]
        base = pf.Solver(net, opts)
        base.solve()
        V, th, _ = base.state()
        X = _features(net, *inj[0][:2])
        w = pf.WarmStart(X.shape[1], -(-2 * net.nB // 8) * 8, HIDDEN, LAYERS, seed=11)
        ym, ys = np.zeros(w.n_out), np.full(w.n_out, 0.02)
        ym[:net.nB], ym[net.nB:2 * net.nB] = V.round(6), th.round(6)
        w.set_norm(X.mean(0), X.std(0) + 1e-6, ym, ys)
        w.stage(X)
        s.update(w=w, nB=net.nB)
    return s


def run(s):
    pf, _ = _package()
    kind = s["kind"]
    if kind in ("solve", "dense"):
        s["solver"].reset()
        r = s["solver"].solve()
        V, th, lq = s["solver"].state()
        return dict(V=V, theta=th, limQ=lq, iterations=r["iterations"], converged=r["converged"])
    if kind == "report":
        solver = pf.Solver(s["net"], s["opts"])
        solver.set_injections(*s["inj"])
        solver.reset()
        r = solver.solve()
        V, th, lq = solver.state()
        return dict(V=V, theta=th, limQ=lq, iterations=r["iterations"], converged=r["converged"],
                    flows=list(solver.flows()))
    if kind == "train":
        loss = s["w"].fit(s["X"], s["Y"], epochs=1, batch=s["batch"], lr=1e-3, weight_decay=1e-5)
        return dict(loss=loss, params=s["w"].params())
    if kind == "serve":
        p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
        st = pf.lib().pf_batch_solve_noalloc(s["b"].h, ctypes.c_int(s["n"]), *[p(t) for t in s["gpu"]], None, None,
                                             *[p(t) for t in s["out"]], None)
        if st != pf.PF_OK:
            raise pf.PfError(st, "pf_batch_solve_noalloc " + pf.last_error())
        V, th, it, cv, _, lq, fl = s["out"]
        return dict(V=V, theta=th, iterations=it, converged=cv, limQ=lq, flips=fl)
    if kind == "warm":
        s["w"].predict_into(s["b"], 0, s["nB"])
    s["b"].solve()
    V, th, it, cv, _ = s["b"].results()
    lq, fl = s["b"].limq()
    return dict(V=V, theta=th, iterations=it, converged=cv, limQ=np.concatenate(lq), flips=fl)


# ---------------------------------------------------------- work and answers

@functools.lru_cache(maxsize=None)
def _counts(name):
    """Of one network: values in its Ybus pattern, and the factorisation's and one solve's operations."""
    pf, _ = _package()
    net = _network(name)
    c = np.diff(pf.SymbolicProbe(net).colptr).astype(float)
    return net.nB + 2 * net.nL, float((16 * c * c + 28 * c).sum()), float((16 * c + 6).sum())


def work(case):
    """One input and output of everything, and the operations of the fewest Newton steps such a case takes
    (4 from a flat start, 2 more where limits switch buses, 3 from a predicted one)."""
    kind, net = case["kind"], _network(case["net"])
    if kind == "train":
        k_in, k_out, rows = -(-3 * net.nB // 8) * 8, -(-2 * net.nB // 8) * 8, case["n"] // case["batch"] * case["batch"]
        weights = k_in * HIDDEN + (LAYERS - 1) * HIDDEN * HIDDEN + HIDDEN * k_out
        steps = rows // case["batch"]
        return {"bytes": 4.0 * rows * (k_in + k_out) + 28.0 * weights * steps, "flops": 6.0 * rows * weights}
    steps = 3 if kind == "warm" else 4 + 2 * case["limits"]
    total = {"bytes": 0.0, "flops": 0.0}
    for name, n in ((case["net"], case.get("n", 1)), (case.get("net2"), case.get("n2", 0))):
        if not name:
            continue
        a = _network(name)
        y, factor, solve = _counts(name)
        if kind == "dense":
            m = 2.0 * (a.nB - 1)
            factor, solve = 2.0 / 3.0 * m ** 3, 2.0 * m * m
        total["bytes"] += n * (5 * 8 * a.nB + a.nPV) + 20.0 * y + 64.0 * a.nB
        total["flops"] += n * steps * (factor + solve + 60.0 * y)
        if kind == "warm":
            k_in, k_out = 3 * a.nB, 2 * a.nB
            weights = k_in * HIDDEN + (LAYERS - 1) * HIDDEN * HIDDEN + HIDDEN * k_out
            total["bytes"] += 4.0 * n * k_in + 2.0 * weights
            total["flops"] += 2.0 * n * weights
    return total


def _newton(net, P, Q, L, limits, start=None):
    """Newton-Raphson in polar form with dense 64-bit algebra, all scenarios of a network together: the power
    balance, PV buses turned PQ at their reactive limits and back, and a last step without switching."""
    n, B = P.shape
    y = 1.0 / (net.r + 1j * net.x)
    t = net.tap_re + 1j * net.tap_im
    Y = np.zeros((B, B), complex)
    np.add.at(Y, (net.frm, net.frm), (y + 0.5j * net.bch) / abs(t) ** 2)
    np.add.at(Y, (net.frm, net.to), -y / t.conj())
    np.add.at(Y, (net.to, net.frm), -y / t)
    np.add.at(Y, (net.to, net.to), y + 0.5j * net.bch)
    Y[np.arange(B), np.arange(B)] += net.gsh + 1j * net.bsh
    V, th = np.repeat(net.V[None], n, 0), np.repeat(net.theta[None], n, 0)
    pq0 = np.zeros(B, bool)
    pq0[net.pq] = True
    isq, qlim, lq = np.repeat(pq0[None], n, 0), Q.copy(), np.zeros((n, net.nPV), bool)
    it, conv, live, flips = np.zeros(n, int), np.zeros(n, bool), np.ones(n, bool), np.zeros(n, int)
    last = np.zeros(n)
    pv, lo, hi = net.pv, net.Qmin, net.Qmax
    diag = np.arange(B)

    def power(s):
        E = V[s] * np.exp(1j * th[s])
        I = E @ Y.T
        return E, I, E * I.conj()

    def switch(s, check, q):
        """limits of scenarios s; check: also PV to PQ"""
        load, was = L[s][:, pv], lq[s]
        low = check[:, None] & ~was & (q[:, pv] + load < lo - FOLGA)
        high = check[:, None] & ~was & ~low & (q[:, pv] + load > hi + FOLGA)
        at_max = qlim[s][:, pv] == hi - load
        back = was & np.where(at_max, V[s][:, pv] > net.Vset + FOLGA, V[s][:, pv] < net.Vset - FOLGA)
        new = qlim[s]
        new[:, pv] = np.where(low, lo - load, np.where(high, hi - load, np.where(back, Q[s][:, pv], new[:, pv])))
        qlim[s] = new
        lq[s] = (was | low | high) & ~back
        q_row = isq[s]
        q_row[:, pv] = lq[s]
        isq[s] = q_row
        flips[s] += (low | high | back).sum(1)

    def step(s, E, I, S):
        for i, k in enumerate(s):
            D = E[i][:, None] * Y.conj() * E[i].conj()[None]
            dth = -1j * D
            dth[diag, diag] += 1j * S[i]
            dV = D / V[k][None]
            dV[diag, diag] += S[i] / V[k]
            keep_p, keep_q = diag != net.slack, isq[k]
            J = np.block([[dth.real[np.ix_(keep_p, keep_p)], dV.real[np.ix_(keep_p, keep_q)]],
                          [dth.imag[np.ix_(keep_q, keep_p)], dV.imag[np.ix_(keep_q, keep_q)]]])
            g = np.concatenate([(P[k] - S[i].real)[keep_p], (qlim[k] - S[i].imag)[keep_q]])
            x = np.linalg.solve(J, g)
            a = keep_p.sum()
            th[k, keep_p] += x[:a]
            V[k, keep_q] += x[a:]
            last[k] = np.abs(x).max()

    while live.any():
        s = np.flatnonzero(live)
        E, I, S = power(s)
        if limits and it[s[0]] >= 1:
            chk = last[s] < 0.1
            act = chk | lq[s].any(1)
            if act.any():
                switch(s[act], chk[act], S.imag[act])
        gp = np.where(diag == net.slack, 0.0, P[s] - S.real)
        gq = np.where(isq[s], qlim[s] - S.imag, 0.0)
        g = np.maximum(np.abs(gp).max(1), np.abs(gq).max(1))
        qg = S.imag[:, pv] + L[s][:, pv]
        bad = ((qg < lo - FOLGA) | (qg > hi + FOLGA)).any(1) & limits
        at = g <= TOL
        again, end = at & bad, at & ~bad
        if again.any():
            switch(s[again], np.ones(again.sum(), bool), S.imag[again])
            last[s[again]] = 0.0
        if end.any():
            step(s[end], E[end], I[end], S[end])
        conv[s[end]] = True
        if (~at).any():
            step(s[~at], E[~at], I[~at], S[~at])
        it[s[~end]] += 1
        live[s] = ~end & (it[s] < MAX_ITER)
    return V, th, it, conv, lq, flips


def _flows(net, V, th):
    """Branch flows in the reference's form: its sign, and the full line charging."""
    out = []
    first = {}
    for l in range(net.nL):
        first.setdefault((net.frm[l], net.to[l]), l)
    y = 1.0 / (net.r + 1j * net.x)
    t = net.tap_re + 1j * net.tap_im
    if np.abs(net.tap_im).max() > 0 or len(first) < net.nL:
        return [None] * 4
    for k, m in ((net.frm, net.to), (net.to, net.frm)):
        Y = -y / t
        a = th[k] - th[m]
        P = V[k] ** 2 * Y.real - V[k] * V[m] * (Y.real * np.cos(a) + Y.imag * np.sin(a))
        q = -V[k] ** 2 * (Y.imag + net.bch) + V[k] * V[m] * (Y.imag * np.cos(a) - Y.real * np.sin(a))
        out += [P, q]
    return out


def _gelu(z):
    return 0.5 * z * (1 + torch.erf(z * math.sqrt(0.5)))


def _train(case, seed):
    """One epoch of AdamW on the mean squared error of the normalised rows, in 64 bits."""
    X, Y, (xm, xs, ym, ys) = _rows(_network(case["net"]), case["n"], seed)
    t = lambda a: torch.from_numpy(np.asarray(a, np.float64))  # noqa: E731
    X, Y = (t(X) - t(np.float32(xm))) / t(np.float32(xs)), (t(Y) - t(np.float32(ym))) / t(np.float32(ys))
    state = 11

    def mix():
        nonlocal state
        state = (state + 0x9E3779B97F4A7C15) & (2 ** 64 - 1)
        z = state
        z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & (2 ** 64 - 1)
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & (2 ** 64 - 1)
        return z ^ (z >> 31)

    def draws(n):       # the same stream, n values at once
        nonlocal state
        s = np.uint64(state) + np.arange(1, n + 1, dtype=np.uint64) * np.uint64(0x9E3779B97F4A7C15)
        state = int(s[-1])
        z = (s ^ (s >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        return (z ^ (z >> np.uint64(31))) >> np.uint64(11)

    sizes = [X.shape[1]] + [HIDDEN] * LAYERS + [Y.shape[1]]
    params = []
    for l, (a, b) in enumerate(zip(sizes, sizes[1:])):
        lim = np.float32(math.sqrt(6.0 / a)) * np.float32(0.1 if l == LAYERS else 1.0)
        u = draws(a * b).astype(np.float64) / 2 ** 53
        params += [t(np.float32((2 * u - 1) * lim)).reshape(a, b), torch.zeros(b, dtype=torch.float64)]
    state = 7
    perm = list(range(len(X)))
    for i in range(len(X) - 1, 0, -1):
        j = mix() % (i + 1)
        perm[i], perm[j] = perm[j], perm[i]
    params = [p.requires_grad_() for p in params]
    opt = torch.optim.AdamW(params, lr=1e-3, betas=(0.9, 0.999), eps=1e-8, weight_decay=1e-5)
    steps, total = len(X) // case["batch"], 0.0
    for k in range(steps):
        rows = perm[k * case["batch"]:(k + 1) * case["batch"]]
        h = X[rows]
        for l in range(LAYERS + 1):
            h = h @ params[2 * l] + params[2 * l + 1]
            if l < LAYERS:
                h = _gelu(h)
        loss = ((h - Y[rows]) ** 2).mean()
        opt.zero_grad()
        loss.backward()
        opt.step()
        total += float(loss.detach())
    return dict(loss=np.array([total / steps]), params=torch.cat([p.detach().reshape(-1) for p in params]))


def exact(case, seed):
    if case["kind"] == "train":
        return _train(case, seed)
    nets, net_of, inj = _inputs(case, seed)
    if sum(len(a[0]) * (net.nB / 118) ** 3 for net, a in zip(nets, inj)) > 5000:
        return None        # dense algebra would take minutes
    got = [_newton(net, *a, bool(case["limits"])) for net, a in zip(nets, inj)]
    V, th, it, cv, lq, fl = (np.concatenate([g[i].ravel() for g in got]) for i in range(6))
    if case["kind"] in ("solve", "dense", "report"):
        out = dict(V=V, theta=th, limQ=lq, iterations=int(it[0]), converged=bool(cv[0]))
        if case["kind"] == "report":
            out["flows"] = _flows(nets[0], V, th)
        return out
    return dict(V=V, theta=th, iterations=it, converged=cv, limQ=lq, flips=fl)
