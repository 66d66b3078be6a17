"""Dense fronts at the sizes where their forms change: a clique of n nodes is
one front of n fully summed columns, a clique hanging off a smaller one gives
a front with rows below its fully summed block.  Random values (pivoting at
most columns) against LAPACK by the normwise backward error, and the same
bits from the wavefront, one-workgroup and many-workgroup forms."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _clique_circuit(n, extra):
    """n fully connected nodes, the first `extra` of them also connected to
    extra + 3 further nodes."""
    from xyce_amd import circuits
    nl = circuits.Netlist("clique %d + %d" % (n, extra))
    a = ["a%d" % i for i in range(n)]
    b = ["b%d" % i for i in range(extra + 3 if extra else 0)]
    for nodes in (a, a[:extra] + b):
        for i in range(len(nodes)):
            for j in range(i):
                nl.add_res("R%d" % len(nl.res), nodes[i], nodes[j], 1.0)
    nl.add_res("RG", a[0], "0", 1.0)
    return nl.layout()


# edges of the 4-column steps, the 16-row tiles, the 8-row thread form, the
# 64-row wavefront form, the 32-column panels and the panel's row classes
# (64, 256, 512), each with its neighbours
@pytest.mark.parametrize("n,extra", [(2, 0), (3, 1), (7, 2), (8, 3), (9, 4), (15, 5), (16, 0),
                                     (17, 8), (31, 9), (32, 4), (33, 16), (47, 5), (48, 0),
                                     (63, 0), (64, 0), (65, 7), (96, 31), (97, 40), (255, 20),
                                     (257, 64), (513, 3)])
def test_front_forms_at_their_edges(n, extra):
    import torch
    from xyce_amd._lib import check, lib
    from xyce_amd.loader import DeviceLoad, _ptr
    nl = _clique_circuit(n, extra)
    print("case: clique %d + %d" % (n, extra), flush=True)
    dev = DeviceLoad(nl, lu_fronts=True)
    rp, ci = dev.pattern()
    N = dev.n_rows - 1
    rng = np.random.default_rng(n)
    vals = rng.standard_normal(len(ci))
    rhs = rng.standard_normal(N + 1)
    rhs[N] = 0.0
    A = np.zeros((N, N))
    rows = np.repeat(np.arange(N + 1), np.diff(rp))
    keep = (rows < N) & (ci < N)
    np.add.at(A, (rows[keep], ci[keep]), vals[keep])
    cu = lambda v: torch.tensor(v, dtype=torch.float64, device="cuda")
    out = []
    for big_m in (64, 1, 8, 1 << 30):
        check(lib().xg_lu_front_set_big(dev.h, big_m), "set big")
        J, R, X, W = cu(vals), cu(rhs), cu(np.zeros(N + 1)), cu(np.ones(N + 1))
        nc = ctypes.c_int32()
        check(lib().xg_components(dev.h, ctypes.byref(nc), None), "components")
        st = cu(np.zeros(4 * nc.value))
        check(lib().xg_lu_solve(dev.h, _ptr(J), _ptr(R), _ptr(X), _ptr(W), _ptr(W), 0.0, 1.0,
                                None, _ptr(st)), "lu solve")
        dev.sync()
        x = X.cpu().numpy()
        assert not st.cpu().numpy().reshape(-1, 4)[:, 2].any()
        if dev.lu_info()["fallbacks"] == 0:   # (a weak pivot block may need it)
            out.append(x)
        berr = np.abs(A @ x[:N] - rhs[:N]).max() / (np.abs(A).sum(1).max() * np.abs(x[:N]).max() +
                                                    np.abs(rhs[:N]).max())
        # n rounding errors of growth-bounded elimination: far below 1e-12,
        # the bound the solve itself accepts
        assert berr < 1e-12, (big_m, berr)
    assert len(out) in (0, 4)   # every form accepts or hands over the same system
    for x in out[1:]:
        assert x.tobytes() == out[0].tobytes()
    dev.close()


def _random_graph(n, degree):
    """n nodes, each joined to `degree` earlier ones at random: the last front
    takes most of them."""
    from xyce_amd import circuits
    rng = np.random.default_rng(1)
    nl = circuits.Netlist("random graph")
    for i in range(1, n):
        for j in rng.integers(0, i, min(degree, i)):
            nl.add_res("R%d" % len(nl.res), "n%d" % i, "n%d" % int(j), 1.0)
    nl.add_res("R%d" % len(nl.res), "n0", "0", 1.0)
    return nl.layout()


# the panel's classes above the cliques': 1024 and 2048 fully summed rows, with
# a root just above each and one near the largest front's
@pytest.mark.parametrize("n,degree,low,high", [(2500, 5, 1024, 1200), (2900, 16, 2048, 2200),
                                               (4100, 20, 3400, 3481)])
def test_tall_panels(n, degree, low, high):
    import torch
    from xyce_amd._lib import check, lib
    from xyce_amd.loader import DeviceLoad, _ptr
    nl = _random_graph(n, degree)
    dev = DeviceLoad(nl, lu_fronts=True)
    root = int(dev.front_plan()["k"].max())
    print("case: random graph of", n, "largest front", root, flush=True)
    assert low < root <= high
    rp, ci = dev.pattern()
    rows = np.repeat(np.arange(n + 1), np.diff(rp))
    keep = (rows < n) & (ci < n)
    r, c = rows[keep], ci[keep]
    rng = np.random.default_rng(n)
    vals = rng.standard_normal(len(ci)) + 2.0 * (rows == ci)
    rhs = np.append(rng.standard_normal(n), 0.0)
    v = vals[keep]
    nc = ctypes.c_int32()
    check(lib().xg_components(dev.h, ctypes.byref(nc), None), "components")
    cu = lambda q: torch.tensor(q, dtype=torch.float64, device="cuda")
    out = []
    for big_m in (64, 1 << 30):
        check(lib().xg_lu_front_set_big(dev.h, big_m), "set big")
        J, R, X, W = cu(vals), cu(rhs), cu(np.zeros(n + 1)), cu(np.ones(n + 1))
        st = cu(np.zeros(4 * nc.value))
        check(lib().xg_lu_solve(dev.h, _ptr(J), _ptr(R), _ptr(X), _ptr(W), _ptr(W), 0.0, 1.0,
                                None, _ptr(st)), "lu solve")
        dev.sync()
        x = X.cpu().numpy()[:n]
        print("threshold", big_m, flush=True)
        assert not st.cpu().numpy().reshape(-1, 4)[:, 2].any()
        ax = np.bincount(r, v * x[c], n)
        berr = np.abs(ax - rhs[:n]).max() / (np.bincount(r, np.abs(v), n).max() * np.abs(x).max() +
                                             np.abs(rhs[:n]).max())
        assert berr < 1e-12   # the bound the solve itself accepts
        out.append(x)
    assert out[1].tobytes() == out[0].tobytes()
    dev.close()
