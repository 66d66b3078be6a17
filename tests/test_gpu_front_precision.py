"""The dense fronts' error on resistive meshes, whose rows nearly cancel, so
that every rounding at an entry's full size shows in the solution: no larger
than 0.75 times that of LAPACK's partial-pivoting LU, on the mean over meshes
and values.  (Measured: 0.60; fronts of a single supernode each, updated in
one chain over all pivots, 0.71; joined up to a wavefront's rows and updated
in one chain 0.79.)  The exact solution is LAPACK's, refined with residuals in
long double."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _mesh(nx, ny, pitch):
    """nx x ny resistors; every pitch-th node carries a two-node tap, so that
    leaves of several sizes hang off the mesh.  One node is grounded."""
    from xyce_amd import circuits
    nl = circuits.Netlist("mesh %d x %d" % (nx, ny))
    r = lambda a, b: nl.add_res("R%d" % len(nl.res), a, b, 1.0)
    for i in range(nx):
        for j in range(ny):
            n = "n%d_%d" % (i, j)
            if i:
                r(n, "n%d_%d" % (i - 1, j))
            if j:
                r(n, "n%d_%d" % (i, j - 1))
            if (i * ny + j) % pitch == 0:
                r(n, "t" + n)
                r("t" + n, "u" + n)
    r("n0_0", "0")
    return nl.layout()


def test_error_on_meshes_is_below_lapacks():
    import torch
    from xyce_amd._lib import check, lib
    from xyce_amd.loader import DeviceLoad, _ptr
    cu = lambda a: torch.tensor(a, dtype=torch.float64, device="cuda")
    LD, norm = np.longdouble, np.linalg.norm
    ratios = []
    for nx, pitch, seeds in ((20, 2, 12), (28, 3, 12), (40, 4, 8)):
        nl = _mesh(nx, nx, pitch)
        dev = DeviceLoad(nl, lu_fronts=True)
        rp, ci = dev.pattern()
        n = dev.n_rows - 1
        rows = np.repeat(np.arange(n + 1), np.diff(rp))
        keep = (rows < n) & (ci < n)
        r, c = rows[keep], ci[keep]
        nc = ctypes.c_int32()
        check(lib().xg_components(dev.h, ctypes.byref(nc), None), "components")
        ours = lapack = 0.0
        for seed in range(seeds):
            rng = np.random.default_rng([seed, nx])
            g = np.exp(rng.uniform(np.log(1e-4), np.log(1e-2), len(r)))
            A = np.zeros((n, n))
            A[r, c] = np.where(r != c, -g, 0.0)
            A = (A + A.T) / 2
            A[np.arange(n), np.arange(n)] = 1e-6 - A.sum(1)   # a weak load to ground
            vals = np.zeros(len(ci))
            vals[keep] = A[r, c]
            b = np.append(rng.normal(0.0, 1e-5, n), 0.0)
            J, R, X, W = cu(vals), cu(b), cu(np.zeros(n + 1)), cu(np.ones(n + 1))
            st = cu(np.zeros(4 * nc.value))
            check(lib().xg_lu_solve(dev.h, _ptr(J), _ptr(R), _ptr(X), _ptr(W), _ptr(W), 0.0, 1.0,
                                    None, _ptr(st)), "lu solve")
            dev.sync()
            assert not st.cpu().numpy().reshape(-1, 4)[:, 2].any()
            assert dev.lu_info()["fallbacks"] == 0
            lap = np.linalg.solve(A, b[:n])
            x = lap.astype(LD)
            for _ in range(3):
                res = b[:n].astype(LD)
                np.subtract.at(res, r, A[r, c].astype(LD) * x[c])
                x = x + np.linalg.solve(A, res.astype(np.float64))
            ours += float(norm(X.cpu().numpy()[:n] - x) / norm(x))
            lapack += float(norm(lap - x) / norm(x))
        ratios.append(ours / lapack)
        print("mesh %d: error %.3g, LAPACK %.3g, ratio %.3f" %
              (nx, ours / seeds, lapack / seeds, ratios[-1]), flush=True)
        dev.close()
    assert np.mean(ratios) < 0.75, ratios
