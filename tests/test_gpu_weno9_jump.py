"""FP64 WENO9 beside a jump: a uniform gas with a transverse velocity of 1e-12 noise and two jumps of 1
along one axis.  Where a stencil reaches a jump the smooth sub-stencils carry all the weight, and their
indicators are 1e-24 of the largest.  The transverse momentum's stage residual on the side without base
value (beyond it the reference's point-value indicators are the rounding of terms that cancel, in
extended precision too), against the oracle's source in extended precision: an interface adds some ten
rounded terms of the size of the jump times the spectral radius (2.5), a node takes two interfaces:
20 x 2.5 x 2^-53."""
import numpy as np
import pytest

import orc
from helpers import interior
from shock_amd import cases, shockx
from test_gpu_weno_pairs import extended  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("noise", [1e-10, 1e-12, 1e-13])
@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("quirks", [3, 0])
def test_noise_beside_a_jump(extended, axis, quirks, noise):  # noqa: F811
    n = [10, 11, 12]
    n[axis] = 40
    n = tuple(n)
    kw = dict(dims=3, n=n, mach=0.5, reynolds=1000.0, inviscid=True, quirks=quirks)
    o = orc.Oracle(S=9, **kw)
    coords = cases.periodic_ext_coords(3, 9, n, lambda a, b, c: (a * n[0], b * n[1], c * n[2]), period=n)
    met = o.metric_from_coords(*coords)
    o.ghost_periodic(met)
    sl = interior(o, 3, n)
    prim = o.zeros(5)
    prim[0][...] = 1.0
    prim[1 + axis][...] = 0.5
    t = 1 + (axis + 1) % 3
    line = noise * np.random.default_rng(axis).standard_normal(n[axis])
    line[14:27] += 1.0
    prim[t][sl] = line.reshape([n[d] if d == axis else 1 for d in range(3)])
    prim[4][...] = cases.energy(prim[1], prim[2], prim[3], np.ones(o.shape), prim[0], o.c.gamma, 0.5)
    o.ghost_periodic(prim)
    want = extended(o, met, prim)[t]
    with shockx.Case(space_order=9, time_order=4, **kw) as c:
        c.build_metric(*coords)
        c.upload_state(prim)
        got = c.rhs()[t]
    err = np.max(np.abs(got[sl] - want[sl]), axis=tuple(d for d in range(3) if d != axis))
    err[13:28] = 0.0                       # the nodes of the jumps' interfaces and those between them
    print(f"[jump] noise {noise:.0e} axis {axis}: {np.max(err):.1e}", flush=True)
    assert np.max(err) <= 20 * 2.5 * 2.0 ** -53
