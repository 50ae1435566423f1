"""The two tiles of the sweeps along the contiguous axis (4 x 64 and 8 x 32 threads) at the ends of their
rows.  A launch over several cases takes one tile by the threads of all of them, so a case alone on one
tile and in a batch beside a case that turns the rule runs both: the arithmetic per node is the same,
and the states are equal bit for bit.  The first sizes take 8 x 32 alone and 4 x 64 in the batch, the
others the reverse."""
import numpy as np
import pytest

import orc
from helpers import interior, smooth_periodic_state
from shock_amd import cases, shockx

pytestmark = pytest.mark.gpu


def _case(n, S, precision, inviscid, quirks, seed):
    kw = dict(dims=3, n=n, mach=0.5, reynolds=400.0, inviscid=inviscid, quirks=quirks)
    o = orc.Oracle(S=S, **kw)
    c = shockx.Case(space_order=S, time_order=4, precision=precision, **kw)
    c.build_metric(*cases.periodic_ext_coords(3, S, n, lambda a, b, z: (a, b, z), period=(1.0, 1.0, 1.0)))
    prim = smooth_periodic_state(o, n, seed, 0.5)
    c.upload_state(prim)
    return o, c, prim


@pytest.mark.parametrize("n,beside", [((6, 16, 65), (24, 16, 63)), ((7, 9, 64), (30, 12, 60)),
                                      ((6, 15, 128), (40, 8, 63)), ((6, 20, 63), (8, 16, 128)),
                                      ((6, 12, 32), (7, 16, 65))])
@pytest.mark.parametrize("S,precision,inviscid,quirks", [(5, shockx.FP64, False, 3), (9, shockx.FP64, False, 3),
                                                         (5, shockx.MIXED, False, 3), (9, shockx.MIXED, False, 3),
                                                         (5, shockx.FP64, True, 3), (9, shockx.FP64, True, 0)])
def test_tiles_agree(n, beside, S, precision, inviscid, quirks):
    if S == 9:
        n, beside = tuple(max(a, 10) for a in n), tuple(max(a, 10) for a in beside)
    o, c, prim = _case(n, S, precision, inviscid, quirks, 5)
    _, d, _ = _case(beside, S, precision, inviscid, quirks, 6)
    tau = 0.5 * c.cfl_dt(0.4)
    c.run(tau, 2)
    alone = c.download_state()
    c.upload_state(prim)
    with shockx.Batch([c, d], [tau, 0.5 * d.cfl_dt(0.4)]) as b:
        b.run(2)
        b.synchronize()
        got = c.download_state()
    sl = interior(o, 3, n)
    for m in range(5):
        assert np.isfinite(got[m][sl]).all()
        assert float(np.max(np.abs(got[m][sl] - alone[m][sl]))) == 0.0, m
    c.close()
    d.close()
