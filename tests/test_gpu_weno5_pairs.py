"""FP64 WENO5 sweeps on states whose stencils have no differences on one side of an interface: a
uniform gas with isolated jumps on a grid of unit spacing, so that all other differences are exactly
zero and the indicators of one split side vanish while the other's do not.  Stage residual against the
oracle at the smallest extents and at the edges of the tiles, both metrics, default and classical
epsilon (the sweeps form the split fluxes without their factor 1/2, so a given epsilon acts as a
quarter of it does on the halved fluxes).  The state is O(1) and a stage residual is a sum of some hundred rounded terms of that size:
1e-13 of the largest entry."""
import numpy as np
import pytest

import orc
from helpers import interior
from shock_amd import cases, shockx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("eps", [0.0, 1e-6])
@pytest.mark.parametrize("inviscid", [True, False])
@pytest.mark.parametrize("n,quirks", [((6, 6, 6), 3), ((31, 8, 63), 3), ((32, 33, 64), 3), ((9, 62, 65), 3),
                                      ((17, 7, 33), 0), ((6, 65, 1), 0), ((33, 6, 1), 0)])
def test_isolated_jumps(n, quirks, inviscid, eps):
    dims = 2 if n[2] == 1 else 3
    kw = dict(dims=dims, n=n, time_order=4, mach=0.5, reynolds=1000.0, inviscid=inviscid, quirks=quirks)
    o = orc.Oracle(S=5, eps_override=eps / 4.0, **kw)
    coords = cases.periodic_ext_coords(dims, 5, n, lambda a, b, c: (a * n[0], b * n[1], c * n[2]),
                                       period=(n[0], n[1], n[2]))
    met = o.metric_from_coords(*coords)
    o.ghost_periodic(met)
    rng = np.random.default_rng(sum(n))
    prim = [np.full(o.shape, a) for a in (1.0, 0.5, 0.25, 0.125 if dims == 3 else 0.0, 8.0)]
    g = o.g
    for m in (0, 1, 2, 3, 4):                      # one jump per field, each at its own node
        at = tuple(g + int(rng.integers(0, n[d])) if d < dims else 0 for d in range(3))
        if m != 3 or dims == 3:
            prim[m][at] += 0.5
    o.ghost_periodic(prim)
    want, _, _ = o.rhs(met, prim)
    with shockx.Case(space_order=5, eps_override=eps, **kw) as c:
        c.build_metric(*coords)
        c.upload_state(prim)
        got = c.rhs()
    sl = interior(o, dims, n)
    for m in range(5):
        assert np.isfinite(got[m][sl]).all()
        scale = max(float(np.max(np.abs(want[m][sl]))), 1.0)
        assert float(np.max(np.abs(got[m][sl] - want[m][sl]))) <= 1e-13 * scale, m
