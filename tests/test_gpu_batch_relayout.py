"""A case whose post-processing runs inside a live batch keeps its pressure from then on, which changes
the batch's launches at the next set_tau: the states (and the stored pressure that post reads) are those
of the cases stepped alone, bit for bit."""
import numpy as np
import pytest

from helpers import interior, setup_2d_mms, setup_3d_turb
from shock_amd import shockx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,S,inviscid,time_order", [(2, 5, False, 4), (2, 9, False, 3), (2, 5, True, 4),
                                                        (3, 5, True, 4), (3, 5, False, 4)])
def test_post_under_a_batch(dims, S, inviscid, time_order):
    setup = setup_2d_mms if dims == 2 else setup_3d_turb
    made = [setup(n=n, S=S, inviscid=inviscid, time_order=time_order) for n in (16, 21)]

    def fresh():                           # handles that do not keep their pressure yet
        out = []
        for o, coords, _, prim, nn in made:
            c = shockx.Case(dims=dims, space_order=S, time_order=time_order, n=nn, mach=o.c.mach,
                            reynolds=o.c.reynolds, inviscid=inviscid)
            c.build_metric(*coords)
            c.upload_state(prim)
            out.append(c)
        return out

    cs = fresh()
    taus = [c.cfl_dt(0.3) for c in cs]
    for c, tau in zip(cs, taus):
        c.run(tau, 2)
        if c is cs[0]:
            c.post()
        c.run(0.5 * tau, 2)
    alone = [c.download_state() for c in cs]
    mach = cs[0].post()[0]
    for c in cs:
        c.close()

    cs = fresh()
    with shockx.Batch(cs, taus) as b:
        b.run(2)
        b.synchronize()
        cs[0].post()
        b.set_tau([0.5 * t for t in taus])
        b.run(2)
        b.synchronize()
        for c, want, (o, _, _, _, nn) in zip(cs, alone, made):
            sl = interior(o, dims, nn)
            got = c.download_state()
            for m in range(5):
                assert np.isfinite(got[m][sl]).all()
                assert np.array_equal(got[m][sl], want[m][sl]), m
        sl = interior(made[0][0], dims, made[0][4])
        assert np.array_equal(cs[0].post()[0][sl], mach[sl])
    for c in cs:
        c.close()
