"""The ordered fold at the lengths where its forms change: a hub node with n
resistors, so that its row of F and its diagonal of dFdx sum n sources (one
thread to 32, a wavefront with a lane per chunk of 32 to 2048, two passes
above).  Against the exactly rounded sum: a sum of s terms in any order, each
term within 2 roundings, differs from the exact one by at most
(s + 3) 2^-53 times the sum of the magnitudes."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("overwrite", [False, True])
@pytest.mark.parametrize("n", [1, 31, 32, 33, 63, 64, 65, 127, 2015, 2016, 2017, 2047, 2048,
                               2049, 4097])
def test_hub_row_at_the_edges_of_the_forms(n, overwrite):
    import torch
    from xyce_amd import circuits
    from xyce_amd.loader import DeviceLoad
    print("case: hub of", n, flush=True)
    rng = np.random.default_rng(n)
    nl = circuits.Netlist("hub %d" % n)
    r = 10.0 ** rng.uniform(0, 4, n)
    for i in range(n):
        nl.add_res("R%d" % i, "h", "a%d" % i, float(r[i]))
    nl.layout()
    dev = DeviceLoad(nl)
    dev.set_output_mode(overwrite)
    n1 = nl.n_nodes + 1
    rp, ci = dev.pattern()
    hub, leaf = nl.node_ids["h"], [nl.node_ids["a%d" % i] for i in range(n)]
    x = rng.uniform(-1, 1, n1)
    x[-1] = 0.0
    f0, j0 = rng.uniform(-1, 1, n1), rng.uniform(-1, 1, dev.nnz)
    cu = lambda a: torch.tensor(a, dtype=torch.float64, device="cuda")
    F, Q, FL, QL = cu(f0), cu(np.zeros(n1)), cu(np.zeros(n1)), cu(np.zeros(n1))
    JF, JQ = cu(j0), cu(np.zeros(dev.nnz))
    st = [cu(np.zeros(max(1, k))) for k in (nl.n_state, nl.n_store)]
    dev.set_solver_state(transient=1, newtonIter=1)
    dev.load_all(cu(x), st[0], st[1], st[0].clone(), st[1].clone(), F, Q, FL, QL, JF, JQ)
    dev.sync()
    F, JF = F.cpu().numpy(), JF.cpu().numpy()
    u, g = 2.0 ** -53, 1.0 / r
    row = slice(rp[hub], rp[hub + 1])
    diag = rp[hub] + int(np.flatnonzero(ci[row] == hub)[0])
    for got, start, t in ((JF[diag], j0[diag], list(g)),
                          (F[hub], f0[hub], list(g * (x[hub] - x[leaf])))):
        t += [] if overwrite else [start]
        assert abs(got - math.fsum(t)) <= (len(t) + 3) * u * math.fsum(map(abs, t))
    dev.close()
