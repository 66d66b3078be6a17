"""What a program that simulates circuits with this framework has the GPU
do, as cases that can be timed and compared: the device load of one Newton
iteration, the Newton linear solve, and fixed-step transients.

Circuits are the framework's own generators: CMOS rings (MOSFET level 1 and
BSIM3), random BSIM3 NAND/NOR logic with RC interconnect, resistive power
grids with switching BSIM3 inverters, and RC ladders with junction diodes,
alone or merged into batches of independent circuits.  A case fixes the
circuit's topology (``seed0``); the seed of ``prepare`` draws the component
values, voltages, states and right-hand sides.

Everything is FP64.  A load writes F, Q, the limiter vectors, both Jacobians
and the next state and store.  A solve returns dx and the per-circuit
statistics.  A transient returns its time points, the probed waveforms and
the final solution, state and store.
"""
import ctypes

import numpy as np
import torch

from xyce_amd import circuits
from xyce_amd._lib import check, lib
from xyce_amd.loader import DeviceLoad
from xyce_amd.transient import Transient

DT = 1e-12          # time step of the Newton systems and the transients
VDD = 1.2

# The listed cases, each for what it stands for:
LISTED = [
    # one small circuit's load, zero-then-add as a caller that keeps the
    # reference's "+=" loads does it: launch latency
    dict(name="load-ring-mos1", kind="load", circuit="ring_mos1", size=101, count=1,
         overwrite=False, dc=False, seed0=1),
    # the device load of a 20,000-transistor circuit, every output written
    dict(name="load-logic", kind="load", circuit="logic", size=5000, count=1,
         overwrite=True, dc=False, seed0=2),
    # a large load dominated by its mesh, zero-then-add
    dict(name="load-grid", kind="load", circuit="grid", size=160, count=10000,
         overwrite=False, dc=False, seed0=5),
    # linear devices and diodes only, at the operating point
    dict(name="load-ladders", kind="load", circuit="ladder", size=10000, count=8,
         overwrite=True, dc=False, seed0=4),
    # the Newton solve of a Monte-Carlo batch of small circuits
    dict(name="solve-rings", kind="solve", circuit="rings", size=301, count=256, seed0=3),
    # of one large, irregular circuit
    dict(name="solve-logic", kind="solve", circuit="logic", size=5000, count=1, seed0=2),
    # of a two-dimensional mesh with clocked inverters
    dict(name="solve-grid", kind="solve", circuit="grid", size=100, count=4000, seed0=5),
    # of a batch of long chains
    dict(name="solve-ladders", kind="solve", circuit="ladder", size=10000, count=8, seed0=4),
    # one small circuit's transient: the latency of a single request
    dict(name="tran-ring", kind="tran", circuit="ring", size=31, count=1, steps=100,
         uic=False, seed0=3),
    # a Monte-Carlo batch's transient
    dict(name="tran-rings", kind="tran", circuit="rings", size=301, count=256, steps=100,
         uic=False, seed0=3),
    # a served batch of random-logic requests, supply ramped from zero
    dict(name="tran-logics", kind="tran", circuit="logics", size=1250, count=8, steps=50,
         uic=True, seed0=4),
    # one large circuit's transient, supply ramped from zero
    dict(name="tran-logic", kind="tran", circuit="logic", size=5000, count=1, steps=16,
         uic=True, seed0=2),
]


def listed():
    return [dict(c) for c in LISTED]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["load", "load", "solve", "solve", "tran"])
    seed0 = rng.randrange(1, 1 << 20)
    if kind == "load":
        circuit = rng.choice(["ring_mos1", "ring", "logic", "grid", "ladder"])
        case = dict(kind=kind, circuit=circuit, count=1, overwrite=rng.random() < 0.6,
                    dc=rng.random() < 0.25, seed0=seed0)
    elif kind == "solve":
        circuit = rng.choice(["rings", "logic", "grid", "ladder"])
        case = dict(kind=kind, circuit=circuit, count=1, seed0=seed0)
    else:
        circuit = rng.choice(["ring", "rings", "logics"])
        case = dict(kind=kind, circuit=circuit, count=1, steps=rng.randrange(16, 51),
                    uic=circuit == "logics", seed0=seed0)
    if circuit in ("ring_mos1", "ring"):
        case["size"] = _log_int(rng, 11, 301)
    elif circuit == "rings":
        case["size"] = rng.randrange(31, 302)
        case["count"] = _log_int(rng, 2, 256)
    elif circuit == "logic":
        case["size"] = _log_int(rng, 100, 4000)
    elif circuit == "logics":
        case["size"] = rng.randrange(150, 1251)
        case["count"] = _log_int(rng, 1, 8)
    elif circuit == "grid":
        case["size"] = _log_int(rng, 12, 100)
        case["count"] = max(4, int(case["size"] ** 2 * rng.uniform(0.1, 0.4)))
    else:
        case["size"] = _log_int(rng, 200, 10000)
        case["count"] = _log_int(rng, 1, 8)
    return case


# ---- circuits

def _netlist(case, seed):
    """The case's circuit: topology from seed0, component values from seed."""
    name, size, count, seed0 = case["circuit"], case["size"], case["count"], case["seed0"]
    rng = np.random.default_rng([seed, seed0])
    top = np.random.default_rng(seed0)
    ramp = 50e-12 if case["kind"] == "tran" else 0.0
    if name == "ring_mos1":
        nl = circuits.ring_oscillator_mos1(size, seed=int(rng.integers(1 << 30)))
    elif name == "ring":
        nl = circuits.ring_oscillator_bsim3(size, dvth0=0.030, dtox=0.02, ramp=ramp, rng=rng)
    elif name == "rings":
        # a Monte-Carlo batch; every transistor its own card where devices
        # are evaluated
        mc = dict(dvth0=0.030, dtox=0.02) if case["kind"] == "tran" else {}
        stages = top.integers(11, size + 1, count)
        nl = circuits.merge([circuits.ring_oscillator_bsim3(int(s), ramp=ramp, rng=rng,
                                                            prefix="m", **mc)
                             for s in stages])
    elif name == "logic":
        nl = circuits.random_logic_bsim3(size, seed=seed0, ramp=ramp)
    elif name == "logics":
        gates = top.integers(min(125, size), size + 1, count)
        nl = circuits.merge([circuits.random_logic_bsim3(int(g), seed=seed0 + k, ramp=ramp)
                             for k, g in enumerate(gates)])
    elif name == "grid":
        nl = circuits.power_grid_bsim3(size, size, count, seed=seed0)
    elif name == "ladder":
        nl = circuits.merge([circuits.rc_ladder_diodes(size, max(1, size // 10),
                                                       seed=seed0 + k)
                             for k in range(count)])
    else:
        raise ValueError(name)
    for rows in (nl.res, nl.caps):
        f = rng.uniform(0.9, 1.1, len(rows))
        rows[:] = [(nm, a, b, v * float(q)) for (nm, a, b, v), q in zip(rows, f)]
    return nl.layout(), rng


def _state(nl, rng):
    """A point the load meets: supplies up (a power grid's mesh with some
    drop), signal nodes mostly near a rail, some switching; the store holds
    the junction voltages of the previous time point, the solution is a
    step further, with a few nodes far enough for the limiters to act."""
    n = nl.n_nodes
    vdd = max([VDD] + [v.dc for v in nl.vsrc])
    prev = np.where(rng.random(n + 1) < 0.5, 0.0, vdd)
    sw = rng.random(n + 1) < 0.2
    prev[sw] = rng.uniform(0.0, vdd, int(sw.sum()))
    if nl.diodes:
        prev = rng.uniform(0.0, 0.7, n + 1)
    x = prev + rng.normal(0.0, 0.01, n + 1)
    far = rng.random(n + 1) < 0.05
    x[far] += rng.uniform(-0.3, 0.3, int(far.sum())) * vdd
    up = [nl.node(v.p) for v in nl.vsrc if v.dc]
    if nl.title.startswith("power grid"):
        up += [i for name, i in nl.node_ids.items() if name[0] == "g"]
    prev[up] = vdd - rng.uniform(0.0, 0.02, len(up))
    x[up] = prev[up] + rng.normal(0.0, 0.001, len(up))
    br = np.asarray(nl.vsrc_branch, dtype=np.int64)
    x[br] = rng.normal(0.0, 1e-3, len(br))
    prev[n] = x[n] = 0.0
    sto = np.zeros(nl.n_store)
    for recs in (nl.mos1, nl.bsim3):
        if not recs:
            continue
        lid = np.array([r["lids"][:4] for r in recs])
        typ = np.array([nl.models[r["model"]].dtype for r in recs], dtype=float)
        base = np.array([r["sto"] for r in recs])
        vd, vg, vs, vb = (prev[lid[:, k]] for k in range(4))   # ground: the last entry
        for k, v in enumerate((vb - vd, vb - vs, vg - vs, vd - vs)):
            sto[base + k] = typ * v
        sto[base + 4] = 0.4
    for (_, a, b, _m, _p), st in zip(nl.diodes, nl.diode_sto):
        sto[st] = prev[nl.node(a)] - prev[nl.node(b)]
    sta = rng.uniform(-1e-15, 1e-15, nl.n_state)
    return x, sta, sto


def _stamps(nl, rng):
    """(row, column, value) of a Newton matrix of the circuit as a transient
    step of DT meets it: conductances and C / DT of the linear devices,
    small-signal conductances and capacitances of the transistors and diodes
    drawn over their working range, +-1 of the sources.  Ground is -1."""
    rows, cols, vals = [], [], []

    def add(r, c, v):
        rows.append(np.asarray(r))
        cols.append(np.asarray(c))
        vals.append(np.broadcast_to(v, np.shape(r)).astype(float))

    def two(a, b, g):
        for r, c, s in ((a, a, 1.0), (b, b, 1.0), (a, b, -1.0), (b, a, -1.0)):
            add(r, c, s * g)

    log_u = lambda lo, hi, k: np.exp(rng.uniform(np.log(lo), np.log(hi), k))
    for devs, val in ((nl.res, lambda v: 1.0 / v), (nl.caps, lambda v: v / DT)):
        if devs:
            two(np.array([nl.node(d[1]) for d in devs]), np.array([nl.node(d[2]) for d in devs]),
                val(np.array([d[3] for d in devs])))
    if nl.diodes:
        two(np.array([nl.node(d[1]) for d in nl.diodes]),
            np.array([nl.node(d[2]) for d in nl.diodes]), log_u(1e-12, 1e-2, len(nl.diodes)))
    for recs in (nl.mos1, nl.bsim3):
        if not recs:
            continue
        d, g, s, b = np.array([r["lids"][:4] for r in recs]).T
        k = len(recs)
        two(d, s, log_u(1e-9, 1e-3, k))
        gm = log_u(1e-8, 2e-3, k)
        for ctl, q in ((g, gm), (b, 0.2 * gm)):
            add(d, ctl, q)
            add(d, s, -q)
            add(s, ctl, -q)
            add(s, s, q)
        for a, c in ((g, s), (g, d), (g, b), (d, b), (s, b)):
            two(a, c, rng.uniform(0.05e-15, 0.5e-15, k) / DT)
    br = np.array(nl.vsrc_branch)
    p = np.array([nl.node(v.p) for v in nl.vsrc])
    m = np.array([nl.node(v.n) for v in nl.vsrc])
    for r, c, v in ((p, br, 1.0), (m, br, -1.0), (br, p, 1.0), (br, m, -1.0)):
        add(r, c, v)
    r, c, v = (np.concatenate(q) for q in (rows, cols, vals))
    keep = (r >= 0) & (c >= 0)
    return r[keep], c[keep], v[keep]


def _system(nl, rng):
    """(rows, columns, values) of the Newton matrix and its right-hand side:
    current residuals, and for the sources' rows voltage errors."""
    n = nl.n_nodes
    r, c, v = _stamps(nl, rng)
    key, inv = np.unique(r.astype(np.int64) * n + c, return_inverse=True)
    vals = np.bincount(inv, v, len(key))
    rhs = np.zeros(n + 1)
    rhs[:n] = rng.normal(0.0, 1e-5, n)
    br = np.asarray(nl.vsrc_branch, dtype=np.int64)
    rhs[br] = rng.normal(0.0, 1e-2, len(br))
    return key // n, key % n, vals, rhs


# ---- the protocol

def _cu(a):
    return torch.tensor(np.asarray(a, dtype=np.float64), dtype=torch.float64, device="cuda")


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


def prepare(case, seed):
    nl, rng = _netlist(case, seed)
    if case["kind"] == "tran":
        tr = Transient(nl)
        probes = {"ring": ["out0", "out5"], "logic": ["g0", "g1"]}.get(case["circuit"])
        if probes is None:
            probes = ["s%d_%s" % (k, "out0" if case["circuit"] == "rings" else "g0")
                      for k in range(case["count"])]
        return dict(case=case, tr=tr, probes=probes)
    dev = DeviceLoad(nl)
    dev.set_stream(torch.cuda.current_stream().cuda_stream)
    n1 = nl.n_nodes + 1
    if case["kind"] == "load":
        x, sta, sto = _state(nl, rng)
        dev.set_output_mode(case["overwrite"])
        if case["dc"]:
            dev.set_solver_state(dcop=1, tranop=1)
        else:
            dev.set_solver_state(transient=1)
        dev.set_time(0.3e-9)
        out = torch.zeros(4 * n1 + 2 * dev.nnz, dtype=torch.float64, device="cuda")
        outs = [out[k * n1:(k + 1) * n1] for k in range(4)]
        outs += [out[4 * n1:4 * n1 + dev.nnz], out[4 * n1 + dev.nnz:]]
        return dict(case=case, dev=dev, out=out, outs=outs,
                    ins=[_cu(x), _cu(sta), _cu(sto), _cu(sta), _cu(sto)])
    # solve
    r, c, v, rhs = _system(nl, rng)
    rp, ci = dev.pattern()
    have = np.repeat(np.arange(n1, dtype=np.int64), np.diff(rp)) * n1 + ci
    at = np.searchsorted(have, r * n1 + c)
    vals = np.zeros(dev.nnz)
    vals[at] = v
    nc = ctypes.c_int32()
    check(lib().xg_components(dev.h, ctypes.byref(nc), None), "components")
    return dict(case=case, dev=dev, J=_cu(vals), rhs=_cu(rhs), dx=_cu(np.zeros(n1)),
                w=_cu(np.full(n1, VDD)), stats=_cu(np.zeros(4 * nc.value)))


def run(state):
    case = state["case"]
    if case["kind"] == "tran":
        tr = state["tr"]
        if case["uic"]:
            tr.sto_n.zero_()   # a start from zero reads the next store, too
        t, w = tr.run(case["steps"] * DT, DT, state["probes"], uic=case["uic"])
        return dict(times=t, waves=w, x=tr.x_curr, sta=tr.sta_c, sto=tr.sto_c)
    dev = state["dev"]
    if case["kind"] == "load":
        if not case["overwrite"]:
            state["out"].zero_()
        dev.load_all(*state["ins"], *state["outs"])
        F, Q, FL, QL, JF, JQ = state["outs"]
        return dict(F=F, Q=Q, dFdxdVp=FL, dQdxdVp=QL, dFdx=JF, dQdx=JQ,
                    sta=state["ins"][3], sto=state["ins"][4])
    dx = state["dx"].zero_()
    check(lib().xg_lu_solve(dev.h, _p(state["J"]), _p(state["rhs"]), _p(dx), _p(state["w"]),
                            _p(state["w"]), 1e-2, 1e-6, None, _p(state["stats"])), "solve")
    return dict(dx=dx, stats=state["stats"])


def _counts(case):
    """Sizes of the case's circuit: unknowns, CSR entries, BSIM3, MOSFET1,
    linear devices, factorisation flops (of the orderings that fit these
    circuits: chains linear, meshes and random logic cubic in their size)."""
    name, s, k = case["circuit"], case["size"], case["count"]
    if name in ("ring_mos1", "ring", "rings"):
        s = s * k if name != "rings" else k * (s + 11) // 2
        b3 = 0 if name == "ring_mos1" else 2 * s
        return s + 2 * k, 7 * s, b3, 2 * s - b3, s + k, 40 * s
    if name in ("logic", "logics"):
        g = s if name == "logic" else (s + min(s, 125)) / 2
        return (int(k * (4 * g + 130)), int(30 * k * g), int(4 * k * g), 0, int(k * (4 * g + 65)),
                int(k * (0.022 * g ** 3 + 200 * g)))
    if name == "grid":
        return s * s + 3 * k, 5 * s * s + 10 * k, 2 * k, 0, 3 * s * s + 2 * k, 24 * s ** 3
    return k * (s + 1), 5 * k * s, 0, 0, k * (2 * s + s // 10), 10 * k * s


def work(case):
    n, nnz, b3, m1, lin, fl = _counts(case)
    # a device's own record, its indices and its old and new state
    load_b = 8 * (5 * n + 2 * nnz) + b3 * (99 * 8 + 38 * 4 + 22 * 8) + \
        m1 * (25 * 8 + 38 * 4 + 18 * 8) + lin * 32
    load_f = 6000 * b3 + 600 * m1 + 12 * lin
    solve_b, solve_f = 8 * (nnz + 4 * n), fl + 4 * nnz
    if case["kind"] == "load":
        return {"bytes": load_b, "flops": load_f}
    if case["kind"] == "solve":
        return {"bytes": solve_b, "flops": solve_f}
    # a step: the predictor's load, one Newton iteration and its load
    asm_b, asm_f = 8 * (3 * nnz + 9 * n), 4 * nnz + 10 * n
    return {"bytes": case["steps"] * (2 * (load_b + asm_b) + solve_b),
            "flops": case["steps"] * (2 * (load_f + asm_f) + solve_f)}


def tolerance(case):
    if case["kind"] == "load":
        # 64-bit sums; numpy's differ by 2e-17 (2-norm) and 2e-15 (largest)
        return {"rel": 1e-14, "max": 1e-13}
    if case["kind"] == "solve":
        # LAPACK's solution differs by up to 2.3e-15 and 4.3e-14
        return {"rel": 1e-14, "max": 2e-13}
    # component values moved by 1e-15 of themselves change the results by
    # up to 2e-15 and 1e-14, moved by 1e-13 by 1e-13 and 3e-13
    return {"rel": 2e-13, "max": 2e-12}


# ---- the same in plain numpy

def _exact_load_ladder(case, seed):
    """R, C, V and the junction diode (level 1, IS and N only)."""
    nl, rng = _netlist(case, seed)
    x, _, sto = _state(nl, rng)
    n = nl.n_nodes
    gmin, vt = 1e-12, 1.3806226e-23 * 300.15 / 1.6021918e-19
    node = lambda devs, k: np.array([nl.node(d[k]) for d in devs])
    F, Q, FL, QL = (np.zeros(n + 1) for _ in range(4))
    key, jf, jq = [], [], []

    def vec(out, a, b, v):
        np.add.at(out, a, v)
        np.add.at(out, b, -v)

    def mat(a, b, f, q):
        for r, c, s in ((a, a, 1.0), (a, b, -1.0), (b, a, -1.0), (b, b, 1.0)):
            key.append((r % (n + 1)) * (n + 1) + c % (n + 1))
            jf.append(s * f)
            jq.append(s * q)

    a, b = node(nl.res, 1), node(nl.res, 2)
    g = 1.0 / np.array([d[3] for d in nl.res])
    vec(F, a, b, g * (x[a] - x[b]))
    mat(a, b, g, 0.0 * g)
    a, b = node(nl.caps, 1), node(nl.caps, 2)
    c = np.array([d[3] for d in nl.caps])
    vec(Q, a, b, c * (x[a] - x[b]))
    mat(a, b, 0.0 * c, c)
    sta = np.zeros(nl.n_state)
    sta[nl.cap_sta] = c * (x[a] - x[b])
    a, b = node(nl.diodes, 1), node(nl.diodes, 2)
    v0 = x[a] - x[b]
    i_s = 1e-14
    vcrit = vt * np.log(vt / (np.sqrt(2.0) * i_s))
    old = v0 if case["dc"] else sto[nl.diode_sto]
    with np.errstate(invalid="ignore", divide="ignore"):
        arg = 1 + (v0 - old) / vt
        lim = np.where(old > 0, np.where(arg > 0, old + vt * np.log(arg), vcrit),
                       vt * np.log(v0 / vt))
        v = np.where((v0 > vcrit) & (np.abs(v0 - old) > 2 * vt), lim, v0)
        rev = (3.0 * vt / (v * np.exp(1.0))) ** 3
        e = np.exp(np.minimum(100.0, v / vt))
        on = v >= -3.0 * vt
        i_d = np.where(on, i_s * (e - 1.0), -i_s * (1.0 + rev)) + gmin * v
        g_d = np.where(on, i_s * e / vt, i_s * 3.0 * rev / v) + gmin
    vec(F, a, b, i_d)
    vec(FL, a, b, g_d * (v - v0))
    mat(a, b, g_d, 0.0 * g_d)
    br = np.array(nl.vsrc_branch)
    p, m = (np.array([nl.node(getattr(s, q)) for s in nl.vsrc]) for q in "pn")
    F[:] += np.bincount(p % (n + 1), x[br], n + 1) - np.bincount(m % (n + 1), x[br], n + 1)
    # at 0.3 ns every PULSE(0 vdd 0 20p 20p 1n 2n) is at its high level
    F[br] = x[p] - x[m] - np.array([s.pulse.v2 for s in nl.vsrc])
    for r, c2, s in ((p, br, 1.0), (m, br, -1.0), (br, p, 1.0), (br, m, -1.0)):
        key.append((r % (n + 1)) * (n + 1) + c2 % (n + 1))
        jf.append(np.full(len(br), s))
        jq.append(np.zeros(len(br)))
    key, inv = np.unique(np.concatenate(key), return_inverse=True)
    JF = np.bincount(inv, np.concatenate(jf), len(key))
    JQ = np.bincount(inv, np.concatenate(jq), len(key))
    ground = (key // (n + 1) == n) | (key % (n + 1) == n)
    JF[ground] = JQ[ground] = 0.0
    for out in (F, Q, FL, QL):
        out[n] = 0.0
    return dict(F=F, Q=Q, dFdxdVp=FL, dQdxdVp=QL, dFdx=JF, dQdx=JQ, sta=sta, sto=None)


def _chain_solve(r, c, v, b):
    """Elimination of a sparse system in descending order of its unknowns
    (no fill on chains)."""
    n = len(b)
    rows = [dict() for _ in range(n)]
    for i, j, q in zip(r.tolist(), c.tolist(), v.tolist()):
        rows[i][j] = q
    b = b.tolist()
    for k in range(n - 1, -1, -1):
        pv = rows[k][k]
        for i in [j for j in rows[k] if j < k]:   # symmetric pattern
            f = rows[i].pop(k, 0.0) / pv
            for j, q in rows[k].items():
                if j < k:
                    rows[i][j] = rows[i].get(j, 0.0) - f * q
            b[i] -= f * b[k]
    x = [0.0] * n
    for k in range(n):
        x[k] = (b[k] - sum(q * x[j] for j, q in rows[k].items() if j < k)) / rows[k][k]
    return np.array(x)


def _exact_solve(case, seed):
    nl, rng = _netlist(case, seed)
    r, c, v, rhs = _system(nl, rng)
    n = nl.n_nodes
    dx = np.zeros(n + 1)
    # nodes held by grounded sources are known: dx = their row's value;
    # their current rows give the branch currents afterwards
    br = np.asarray(nl.vsrc_branch, dtype=np.int64)
    held = np.array([nl.node(s.p) for s in nl.vsrc], dtype=np.int64)
    dx[held] = rhs[br]
    free = np.ones(n, bool)
    free[held] = free[br] = False
    ids = np.cumsum(free) - 1
    b = rhs[:n] - np.bincount(r, v * dx[c], n)
    m = free[r] & free[c]
    fr, fc, fv = ids[r[m]], ids[c[m]], v[m]
    k = int(free.sum())
    if case["circuit"] == "ladder":
        dx[:n][free] = _chain_solve(fr, fc, fv, b[free])
    elif case["circuit"] == "rings":
        # independent circuits: one dense solve per ring
        comp = np.zeros(n, np.int64)
        for name, i in nl.node_ids.items():
            comp[i] = int(name[1:name.index("_")])
        cf = comp[free]
        start = np.searchsorted(cf, np.arange(case["count"] + 1))
        order = np.argsort(cf[fr], kind="stable")
        fr, fc, fv = fr[order], fc[order], fv[order]
        ptr = np.searchsorted(cf[fr], np.arange(case["count"] + 1))
        sol, bf = np.zeros(k), b[free]
        for q in range(case["count"]):
            s0, s1, e = start[q], start[q + 1], slice(ptr[q], ptr[q + 1])
            A = np.zeros((s1 - s0, s1 - s0))
            A[fr[e] - s0, fc[e] - s0] = fv[e]
            sol[s0:s1] = np.linalg.solve(A, bf[s0:s1])
        dx[:n][free] = sol
    elif k <= 21000:
        A = np.zeros((k, k))
        A[fr, fc] = fv
        dx[:n][free] = np.linalg.solve(A, b[free])
    else:
        return None
    # branch currents from the held nodes' rows
    res = rhs[:n] - np.bincount(r, v * dx[c], n)
    dx[br] = res[held]
    return dict(dx=dx, stats=None)


def exact(case, seed):
    if case["kind"] == "load" and case["circuit"] == "ladder":
        return _exact_load_ladder(case, seed)
    if case["kind"] == "solve":
        return _exact_solve(case, seed)
    # the transistor models and whole transients have no closed form in
    # a few lines of numpy
    return None
