"""Dense fronts at the sizes where their forms change.  A star of cliques, all
joined to one separator, is a front per clique, of its nodes (fully summed)
and the separator's, and a front of the separator; a single clique is one front
without rows below.  The plan is checked to be that.  Random values (pivoting at
most columns) by the normwise backward error, and the same bits from the
thread, wavefront, one-workgroup and many-workgroup forms."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _star(sizes, sep):
    """A clique of each size, all joined to the same `sep` nodes."""
    from xyce_amd import circuits
    nl = circuits.Netlist("star of %d cliques" % len(sizes))
    s = ["s%d" % i for i in range(sep)]
    r = lambda a, b: nl.add_res("R%d" % len(nl.res), a, b, 1.0)
    for i in range(sep):
        for other in s[:i]:
            r(s[i], other)
    for q, size in enumerate(sizes):
        a = ["c%d_%d" % (q, i) for i in range(size)]
        for i in range(size):
            for other in a[:i] + s:
                r(a[i], other)
    r(s[0] if sep else "c0_0", "0")
    return nl.layout()


def _check(nl, want, thresholds, seed, diagonal):
    """The plan's (rows, fully summed columns) are `want`; every threshold's
    solve stands without the dense fallback, to the bound that the solve itself
    accepts, with the same bits."""
    import torch
    from xyce_amd._lib import check, lib
    from xyce_amd.loader import DeviceLoad, _ptr
    dev = DeviceLoad(nl, lu_fronts=True)
    fp = dev.front_plan()
    assert sorted(zip(fp["m"].tolist(), fp["k"].tolist())) == sorted(want)
    rp, ci = dev.pattern()
    n = dev.n_rows - 1
    rows = np.repeat(np.arange(n + 1), np.diff(rp))
    keep = (rows < n) & (ci < n)
    r, c = rows[keep], ci[keep]
    rng = np.random.default_rng(seed)
    vals = rng.standard_normal(len(ci)) + diagonal * (rows == ci)
    rhs = np.append(rng.standard_normal(n), 0.0)
    v = vals[keep]
    nc = ctypes.c_int32()
    check(lib().xg_components(dev.h, ctypes.byref(nc), None), "components")
    cu = lambda q: torch.tensor(q, dtype=torch.float64, device="cuda")
    out = []
    for big_m in thresholds:
        check(lib().xg_lu_front_set_big(dev.h, big_m), "set big")
        J, R, X, W = cu(vals), cu(rhs), cu(np.zeros(n + 1)), cu(np.ones(n + 1))
        st = cu(np.zeros(4 * nc.value))
        check(lib().xg_lu_solve(dev.h, _ptr(J), _ptr(R), _ptr(X), _ptr(W), _ptr(W), 0.0, 1.0,
                                None, _ptr(st)), "lu solve")
        dev.sync()
        x = X.cpu().numpy()[:n]
        assert not st.cpu().numpy().reshape(-1, 4)[:, 2].any()
        assert dev.lu_info()["fallbacks"] == 0, big_m
        ax = np.bincount(r, v * x[c], n)
        berr = np.abs(ax - rhs[:n]).max() / (np.bincount(r, np.abs(v), n).max() * np.abs(x).max() +
                                             np.abs(rhs[:n]).max())
        assert berr < 1e-12, (big_m, berr)
        out.append(x)
    for x in out[1:]:
        assert x.tobytes() == out[0].tobytes()
    dev.close()


# cliques: the edges of the four-column steps, the 16-row tiles, the wavefront
# form, the 32-column panels and the panel's row classes (64, 256, 512)
@pytest.mark.parametrize("n", [2, 3, 4, 5, 15, 16, 17, 31, 32, 33, 47, 48, 63, 64, 65, 96, 97,
                               255, 256, 257, 513])
def test_fronts_without_rows_below(n):
    print("case: clique of", n, flush=True)
    _check(_star([n], 0), [(n, n)], (64, 1, 8, 1 << 30), n, 1.0)


# stars by their largest front: the edges of the wavefront form's tile counts
# (15, 31, 47, 63 rows and the right-hand side), of the wavefront form, of the
# update's 64-row tiles and of the panels, each with few and with many rows below
@pytest.mark.parametrize("rows,sep", [(8, 1), (8, 5), (15, 2), (16, 3), (16, 9), (31, 1), (32, 5),
                                      (32, 24), (47, 2), (48, 8), (48, 40), (63, 1), (64, 3),
                                      (64, 32), (64, 60), (65, 1), (65, 40), (96, 31), (97, 32),
                                      (97, 64), (128, 63), (129, 64), (160, 128), (288, 31)])
def test_fronts_with_rows_below(rows, sep):
    print("case: fronts of up to", rows, "rows,", sep, "below", flush=True)
    k = rows - sep
    # (as many as keep the planner from joining them: more serial columns than
    # it allows, also where one column of each is left)
    sizes = [k] * (18 // k + 3) + [max(1, k - d) for d in (1, 2, 3, 4, 5, 7)]
    want = [(q + sep, q) for q in sizes] + [(sep, sep)]
    _check(_star(sizes, sep), want, (64, 1, 8, 1 << 30), rows, 3.0)


def test_level_of_many_fronts():
    """More than 2048 small fronts in a level: a thread each up to 8 rows, a
    wavefront each by tile count above."""
    sep = 3
    sizes = [1 + i % 5 for i in range(1500)] + [6 + i % 24 for i in range(600)] + \
        [30 + i % 32 for i in range(64)]
    print("case: level of", len(sizes), flush=True)
    _check(_star(sizes, sep), [(q + sep, q) for q in sizes] + [(sep, sep)],
           (64, 1, 20, 1 << 30), 9, 3.0)


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
    from xyce_amd.loader import DeviceLoad
    nl = _random_graph(n, degree)
    plan = DeviceLoad(nl, plan_only=True, lu_fronts=True)
    fp = plan.front_plan()
    plan.close()
    root = int(fp["k"].max())
    print("case: random graph of", n, "largest front", root, flush=True)
    assert low < root <= high
    _check(nl, list(zip(fp["m"].tolist(), fp["k"].tolist())), (64, 1 << 30), n, 2.0)
