"""Steps of all-periodic inviscid 3D cases, whose sweeps read ghosts at their periodic image: three steps
against the oracle at the smallest extents and the edges of the tiles (1e-12 relative, the bar of the other
parity tests), and the whole downloaded state, ghosts included, equal to that of a case whose ghosts are
filled."""
import numpy as np
import pytest

import orc
from helpers import conserved, interior, rel_linf, smooth_periodic_state
from shock_amd import cases, shockx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(6, 6, 6), (7, 9, 33), (32, 8, 64), (8, 33, 65)])
@pytest.mark.parametrize("S,quirks,time_order", [(5, 3, 4), (5, 0, 3), (9, 3, 3), (9, 0, 4)])
def test_steps(n, S, quirks, time_order):
    if S == 9:
        n = tuple(max(a, 10) for a in n)
    kw = dict(dims=3, n=n, mach=0.5, reynolds=400.0, inviscid=True, quirks=quirks, time_order=time_order)
    o = orc.Oracle(S=S, **kw)
    coords = cases.periodic_ext_coords(3, S, n, lambda a, b, z: (a, b, z), period=(1.0, 1.0, 1.0))
    met = o.metric_from_coords(*coords)
    o.ghost_periodic(met)
    prim = smooth_periodic_state(o, n, 9, 0.5)
    with shockx.Case(space_order=S, **kw) as c, shockx.Case(space_order=S, **kw) as d:
        states = []
        for k in (c, d):
            k.build_metric(*coords)
            k.upload_state(prim)
            if k is d:
                d.post()                           # d keeps p and c from here on, so its ghosts are filled
            tau = c.cfl_dt(0.3) if k is c else tau
            k.run(tau, 3)
            states.append(k.download_state())
    got, filled = states
    want = o.run(tau, met, prim, 3)
    assert max(rel_linf(conserved(got), conserved(want), interior(o, 3, n))) <= 1e-12
    for a, b in zip(got, filled):
        assert np.array_equal(a, b)
