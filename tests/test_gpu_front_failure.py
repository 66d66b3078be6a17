"""One front of several that share a launch fails: a star of cliques, every
clique one front above the many-workgroup threshold (or below it, a wavefront
each), all in one level.  The failing clique's component is reported singular
with its iterate left alone when it is too large for the dense fallback, goes
to the fallback when not, and the other component is solved as if nothing had
happened -- in every form, and the same again on the next solve."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _star(nl, tag, cliques, size, sep):
    """`cliques` cliques of `size` nodes, all joined to the same `sep`."""
    s = ["%ss%d" % (tag, i) for i in range(sep)]
    for i in range(sep):
        for j in range(i):
            nl.add_res("R%d" % len(nl.res), s[i], s[j], 1.0)
    nl.add_res("R%d" % len(nl.res), s[0], "0", 1.0)
    for q in range(cliques):
        a = ["%sc%d_%d" % (tag, q, i) for i in range(size)]
        for i in range(size):
            for other in a[:i] + s:
                nl.add_res("R%d" % len(nl.res), a[i], other, 1.0)


@pytest.mark.parametrize("size,many,few", [(90, 24, 6), (30, 80, 20)])
@pytest.mark.parametrize("kind", ["zero column", "infinity", "nan"])
def test_one_singular_front_among_many(size, many, few, kind):
    import torch
    from xyce_amd import circuits
    from xyce_amd._lib import check, lib
    from xyce_amd.loader import DeviceLoad, _ptr
    print("case: %s, cliques of %d" % (kind, size), flush=True)
    sep = 5
    nl = circuits.Netlist("stars")
    _star(nl, "b", many, size, sep)    # above the dense fallback's 2048 unknowns
    _star(nl, "f", few, size, sep)
    nl.layout()
    dev = DeviceLoad(nl, lu_fronts=True)
    fp = dev.front_plan()
    level0 = fp["m"][fp["lv"][fp["lv_ptr"][0]:fp["lv_ptr"][1]]]
    assert np.count_nonzero(level0 == size + sep) >= (many + few) * 3 // 4
    rp, ci = dev.pattern()
    n = dev.n_rows - 1
    rows = np.repeat(np.arange(n + 1), np.diff(rp))
    keep = (rows < n) & (ci < n)
    nc = ctypes.c_int32()
    check(lib().xg_components(dev.h, ctypes.byref(nc), None), "components")
    comp = np.zeros(n, np.int32)
    check(lib().xg_components(dev.h, ctypes.byref(nc), comp.ctypes.data), "components")
    node = lambda name: nl.node_ids[name]
    cb, cf = comp[node("bs0")], comp[node("fs0")]
    assert np.count_nonzero(comp == cb) > 2048 >= np.count_nonzero(comp == cf)
    rng = np.random.default_rng(size)
    vals = rng.standard_normal(len(ci))
    vals[rows == ci] += 2.0 * size
    rhs = rng.standard_normal(n + 1)
    rhs[n] = 0.0
    x0 = rng.standard_normal(n + 1)

    def spoil(v, tag):
        """The matrix with clique 3's column 7 emptied within the clique (the
        separator rows keep theirs: singular for the front, not as a whole),
        or one entry of it not finite."""
        v = v.copy()
        mine = np.array([node("%sc3_%d" % (tag, i)) for i in range(size)])
        col = ci == mine[7]
        if kind == "zero column":
            v[col & np.isin(rows, mine)] = 0.0
        else:
            v[col & (rows == mine[11])] = np.inf if kind == "infinity" else np.nan
        return v

    cu = lambda a: torch.tensor(a, dtype=torch.float64, device="cuda")

    def solve(v):
        J, R, X, W = cu(v), cu(rhs), cu(x0), cu(np.ones(n + 1))
        st = cu(np.zeros(4 * nc.value))
        check(lib().xg_lu_solve(dev.h, _ptr(J), _ptr(R), _ptr(X), _ptr(W), _ptr(W), 0.0, 1.0,
                                None, _ptr(st)), "lu solve")
        dev.sync()
        return X.cpu().numpy(), st.cpu().numpy().reshape(-1, 4)

    def backward_error(v, dx, of):
        A = np.zeros((n, n))
        A[rows[keep], ci[keep]] = v[keep]
        m = comp == of
        A, b, dx = A[np.ix_(m, m)], rhs[:n][m], dx[:n][m]
        return np.abs(A @ dx - b).max() / (np.abs(A).sum(1).max() * np.abs(dx).max() +
                                           np.abs(b).max())

    for big_m in (64, 1, 1 << 30):
        print("threshold", big_m, flush=True)
        check(lib().xg_lu_front_set_big(dev.h, big_m), "set big")
        want, st = solve(vals)
        assert not st[:, 2].any() and dev.lu_info()["fallbacks"] == 0
        for c in (cb, cf):   # the bound that the solve itself accepts
            assert backward_error(vals, want - x0, c) < 1e-12
        # the large component fails: reported, untouched, the other one whole
        for _ in range(2):
            x, st = solve(spoil(vals, "b"))
            assert st[cb, 2] == 1 and st[cf, 2] == 0
            assert x[:n][comp == cb].tobytes() == x0[:n][comp == cb].tobytes()
            assert x[:n][comp == cf].tobytes() == want[:n][comp == cf].tobytes()
        # the small one fails: the dense fallback solves it
        bad = spoil(vals, "f")
        x, st = solve(bad)
        assert dev.lu_info()["fallbacks"] == 1 and st[cb, 2] == 0
        assert x[:n][comp == cb].tobytes() == want[:n][comp == cb].tobytes()
        if kind == "zero column":
            assert st[cf, 2] == 0 and backward_error(bad, x - x0, cf) < 1e-12
        # and nothing is left behind
        x, st = solve(vals)
        assert x.tobytes() == want.tobytes() and not st[:, 2].any()
    dev.close()
