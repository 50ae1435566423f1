"""The 2D stage kernel (15 x 15 node tiles) against the oracle at the edges of its tiles: stage residual
(ghosts filled first) and steps (periodic cases read ghosts at their image), both orders, viscous and
inviscid, both time schemes, inflow / outflow / wall faces, a metric with z entries.
Bars of the other parity tests: 1e-12 relative; 1e-7 for the mixed form's step (FP32 deviation)."""
import numpy as np
import pytest

import orc
from helpers import conserved, interior, rel_linf
from shock_amd import cases, shockx

pytestmark = pytest.mark.gpu
SIZES = [(10, 10), (15, 15), (16, 14), (30, 31), (17, 46), (61, 29)]


def _setup(n, S, seed, bc=(0,) * 6, **kw):
    nn = (n[0], n[1], 1)
    kw = dict(dict(mach=0.5, reynolds=400.0), **kw)
    extra = dict(bc=bc, inflow=(1.0, 1.5, 0.0, 0.0, 1.0), T_wall=1.1)
    o = orc.Oracle(dims=2, S=S, n=nn, **kw, **extra)
    per = tuple(bc[2 * d] == 0 for d in range(3))
    tp = 2.0 * np.pi
    coords = cases.ext_coords(2, S, nn, lambda a, b, c: (a + 0.02 * np.sin(tp * a) * np.sin(tp * b),
                                                         b - 0.02 * np.sin(tp * a) * np.sin(tp * b), 0.0 * a), per)
    met = o.metric_from_coords(*coords)
    o.ghost_periodic(met)
    o.mirror_metric(met)
    rng = np.random.default_rng(seed)
    x, y, _ = cases.interior_coords(2, S, nn, *coords)
    ph = rng.uniform(0.0, tp, size=8)
    rho = 1.0 + 0.1 * np.sin(tp * x + ph[0]) * np.sin(tp * y + ph[1])
    u = 0.8 + 0.3 * np.sin(tp * (x + y) + ph[2])
    v = 0.3 * np.cos(tp * x + ph[3]) * np.sin(tp * y + ph[4])
    p = 1.0 + 0.1 * np.cos(tp * (x - y) + ph[5])
    prim = [rho, u, v, np.zeros_like(x), cases.energy(u, v, 0.0 * x, p, rho, 1.4, kw["mach"])]
    prim = [np.ascontiguousarray(a) for a in prim]
    o.ghost_periodic(prim)
    case = dict(dims=2, space_order=S, n=nn, bc=bc, **kw, inflow=extra["inflow"], T_wall=1.1)
    return o, coords, met, prim, case


def _live(errs):
    return max(errs[:3] + errs[4:])


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("S,inviscid", [(5, False), (5, True), (9, False)])
def test_residual(n, S, inviscid):
    o, coords, met, prim, case = _setup(n, S, 3, inviscid=inviscid)
    want, _, _ = o.rhs(met, [a.copy() for a in prim])
    with shockx.Case(**case) as c:
        c.upload_metric(met)
        c.upload_state(prim)
        got = c.rhs()
    assert _live(rel_linf(got, want, interior(o, 2, case["n"]))) <= 1e-12


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("S,time_order,precision", [(5, 4, shockx.FP64), (5, 3, shockx.FP64), (9, 4, shockx.FP64),
                                                    (5, 4, shockx.MIXED), (9, 3, shockx.MIXED)])
def test_periodic_steps(n, S, time_order, precision):
    """Two steps: every stage after the first reads a buffer whose ghosts nothing has filled; the
    downloaded ghosts are those of the last stage's input, as in the oracle's single array."""
    o, coords, met, prim, case = _setup(n, S, 4, time_order=time_order)
    tau = o.cfl_dt(0.4, met, prim)
    un, urk, scratch = [a.copy() for a in prim], [a.copy() for a in prim], o.zeros(30)
    for _ in range(2):
        o.step(tau, met, un, urk, None, scratch)
        for a, b in zip(un, urk):
            a[...] = b
    with shockx.Case(precision=precision, **case) as c:
        c.build_metric(*coords)
        c.upload_state(prim)
        c.run(tau, 2)
        got = c.download_state()
    every = tuple(slice(0, e) for e in o.shape)
    assert _live(rel_linf(conserved(got), conserved(un), every)) <= (1e-12 if precision == shockx.FP64 else 1e-7)


@pytest.mark.parametrize("n", [(16, 14), (30, 31)])
@pytest.mark.parametrize("bc", [(shockx.BC_INFLOW_SUPERSONIC, shockx.BC_OUTFLOW_RIEMANN, 0, 0, 0, 0),
                                (0, 0, shockx.BC_WALL_SLIP, shockx.BC_WALL_NOSLIP, 0, 0),
                                (0, 0, shockx.BC_WALL_NOSLIP, shockx.BC_WALL_ISOTHERMAL, 0, 0),
                                (shockx.BC_WALL_NOSLIP, shockx.BC_WALL_ISOTHERMAL, 0, 0, 0, 0)])
def test_faces_step(n, bc):
    o, coords, met, prim, case = _setup(n, 5, 5, bc=bc)
    tau = 0.5 * o.cfl_dt(0.4, met, prim)
    want = o.run(tau, met, prim, 1)
    with shockx.Case(**case) as c:
        c.build_metric(*coords)
        c.upload_state(prim)
        c.run(tau, 1)
        got = c.download_state()
    assert _live(rel_linf(conserved(got), conserved(want), interior(o, 2, case["n"]))) <= 1e-12


@pytest.mark.parametrize("S", [5, 9])
def test_metric_with_z_entries(S):
    o, coords, met, prim, case = _setup((17, 31), S, 6)
    for m in (2, 5):
        met[m][...] = 0.1 * met[m - 2 if m == 2 else 4]
    want, _, _ = o.rhs(met, [a.copy() for a in prim])
    with shockx.Case(**case) as c:
        c.upload_metric(met)
        c.upload_state(prim)
        got = c.rhs()
    assert _live(rel_linf(got, want, interior(o, 2, case["n"]))) <= 1e-12
