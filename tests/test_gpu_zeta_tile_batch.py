"""Both tiles of the sweeps along the contiguous axis (4 x 64 and 8 x 32 threads) in single and in batched
launches: a case whose tile alone is the one and, in a batch beside a larger case, the other, either way
round.  The arithmetic per node is the same, and the states are equal bit for bit."""
import numpy as np
import pytest

import orc
from helpers import interior, smooth_periodic_state
from shock_amd import cases, shockx

pytestmark = pytest.mark.gpu


def narrow(sizes):
    """The library's rule: 8 x 32 where it takes fewer than 7/8 of the threads."""
    up = lambda a, b: -(-a // b)  # noqa: E731
    w = sum(n[0] * up(n[1], 4) * up(n[2], 63) for n in sizes)
    return 8 * sum(n[0] * up(n[1], 8) * up(n[2], 31) for n in sizes) < 7 * w


def _case(n, S, precision, inviscid, quirks, seed):
    kw = dict(dims=3, n=n, mach=0.5, reynolds=400.0, inviscid=inviscid, quirks=quirks)
    o = orc.Oracle(S=S, **kw)
    c = shockx.Case(space_order=S, time_order=4, precision=precision, **kw)
    c.build_metric(*cases.periodic_ext_coords(3, S, n, lambda a, b, z: (a, b, z), period=(1.0, 1.0, 1.0)))
    prim = smooth_periodic_state(o, n, seed, 0.5)
    c.upload_state(prim)
    return o, c, prim


@pytest.mark.parametrize("n,beside,alone", [((10, 16, 65), (24, 16, 63), True), ((11, 11, 31), (30, 16, 63), True),
                                            ((10, 20, 63), (60, 16, 65), False), ((10, 12, 62), (48, 24, 64), False),
                                            ((11, 10, 32), (40, 16, 70), False)])
@pytest.mark.parametrize("S,precision,inviscid,quirks", [(5, shockx.FP64, False, 3), (9, shockx.FP64, False, 3),
                                                         (5, shockx.MIXED, False, 3), (9, shockx.MIXED, False, 3),
                                                         (5, shockx.FP64, True, 3), (9, shockx.FP64, True, 0)])
def test_other_tile_in_the_batch(n, beside, alone, S, precision, inviscid, quirks):
    assert narrow([n]) == alone and narrow([n, beside]) != alone
    o, c, prim = _case(n, S, precision, inviscid, quirks, 5)
    _, d, _ = _case(beside, S, precision, inviscid, quirks, 6)
    tau = 0.5 * c.cfl_dt(0.4)
    c.run(tau, 2)
    want = c.download_state()
    c.upload_state(prim)
    with shockx.Batch([c, d], [tau, 0.5 * d.cfl_dt(0.4)]) as b:
        b.run(2)
        b.synchronize()
        got = c.download_state()
    sl = interior(o, 3, n)
    for m in range(5):
        assert np.isfinite(got[m][sl]).all()
        assert np.array_equal(got[m][sl], want[m][sl]), m
    c.close()
    d.close()
