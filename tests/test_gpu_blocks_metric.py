"""Joined blocks whose metrics differ in kind: one block's rows have entries that the other's own rows
lack (2D: z entries; 3D: off-diagonal ones), and the ghost rows it gets from its neighbour have them.
The box cut in two evolves as the whole box, bit for bit."""
import numpy as np
import pytest

import orc
from helpers import interior, smooth_periodic_state
from shock_amd import cases, shockx

pytestmark = pytest.mark.gpu

P, I = shockx.BC_PERIODIC, shockx.BC_INTERFACE


def _slab(a, axis, start, length):
    return np.ascontiguousarray(np.take(a, range(start, start + length), axis=axis))


@pytest.mark.parametrize("dims,n,axis,S,inviscid", [
    (2, (24, 20, 1), 0, 5, False), (2, (17, 36, 1), 1, 9, False), (2, (24, 20, 1), 1, 5, True),
    (3, (20, 12, 13), 0, 5, False), (3, (12, 20, 11), 1, 9, True)])
def test_mixed_kinds_equal_whole_box(dims, n, axis, S, inviscid):
    g, half = (S + 1) // 2, n[axis] // 2
    # (3D: without the zeta-index quirk, whose reads depend on the block's extents)
    kw = dict(dims=dims, mach=0.5, reynolds=200.0, inviscid=inviscid, quirks=0)
    o = orc.Oracle(S=S, n=n, **kw)
    ident = cases.periodic_ext_coords(dims, S, n, cases.cartesian_unit(dims))
    met = o.metric_from_coords(*ident)
    o.ghost_periodic(met)
    for m in (1, 2, 3, 5, 6, 7):                    # an exactly diagonal metric to start from
        met[m][...] = 0.0
    upper = tuple(slice(g + half, g + n[d]) if d == axis else interior(o, dims, n)[d] for d in range(3))
    for m in (2, 5) if dims == 2 else (1, 2, 3, 5, 6, 7):
        met[m][upper] = 0.3 * met[0][upper]
    o.ghost_periodic(met)
    if dims == 3:
        prim = smooth_periodic_state(o, n, 3, 0.5)
    else:
        x, y, _ = cases.interior_coords(2, S, n, *ident)
        prim = cases.mms_periodic_2d_state(np.ascontiguousarray(x), np.ascontiguousarray(y), mach=0.5)
        o.ghost_periodic(prim)

    def case(nn, bc, lo):
        c = shockx.Case(space_order=S, time_order=4, n=nn, bc=bc, **kw)
        c.upload_metric([_slab(m, axis, lo, nn[axis] + 2 * g) for m in met] if nn != n else met)
        c.upload_state([_slab(f, axis, lo, nn[axis] + 2 * g) for f in prim] if nn != n else prim)
        return c
    with case(n, (P,) * 6, 0) as whole:
        tau = whole.cfl_dt(0.3)
        whole.run(tau, 2)
        ref = [_slab(f, axis, g, n[axis]) for f in whole.download_state()]
    nb = tuple(half if d == axis else n[d] for d in range(3))
    bc = tuple(I if f // 2 == axis else P for f in range(6))
    lo, hi, t = 2 * axis, 2 * axis + 1, (1, 2, 3)
    conn = [(0, hi, 1, lo, t), (1, lo, 0, hi, t), (0, lo, 1, hi, t), (1, hi, 0, lo, t)]
    blocks = []
    try:
        for b in range(2):
            blocks.append(case(nb, bc, b * half))
            # the block's own rows alone: what its neighbours give is left to the transfer
            own = [_slab(m, axis, b * half, half + 2 * g) for m in met]
            for m in own:
                for s in (slice(0, g), slice(g + half, None)):
                    m[tuple(s if d == axis else slice(None) for d in range(3))] = 0.0
            blocks[b].upload_metric(own)
        with shockx.Blocks(blocks, conn) as grp:
            grp.transfer_metric()
            grp.run(tau, 2)
            got = [np.concatenate([_slab(blocks[b].download_state()[m], axis, g, half) for b in range(2)], axis=axis)
                   for m in range(5)]
    finally:
        for c in blocks:
            c.close()
    cut = tuple(slice(None) if d == axis else interior(o, dims, n)[d] for d in range(3))
    for m in range(5):
        assert np.isfinite(got[m][cut]).all()
        assert np.array_equal(got[m][cut], ref[m][cut]), m
