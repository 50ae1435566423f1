"""FP64 WENO sweeps at the edges of their tiles.

WENO5 on states whose stencils have no differences on one side of an interface: a
uniform gas with isolated jumps on a grid of unit spacing, so that all other differences are exactly
zero and the indicators of one split side vanish while the other's do not.  Stage residual against the
oracle at the smallest extents and at the edges of the tiles, both metrics, default and classical
epsilon (the sweeps form the split fluxes without their factor 1/2, so a given epsilon acts as a
quarter of it does on the halved fluxes).  The state is O(1) and a stage residual is a sum of some hundred rounded terms of that size:
1e-13 of the largest entry.

WENO9 on a smooth periodic field (where differences vanish the reference's indicators are the rounding
of terms that cancel, so its weights are not defined to compare with): the stage residual's bar of the
other parity tests, 1e-12, against the oracle's source built in extended precision.  The FP64 oracle
itself is up to 7e-12 from that on these states, for the same reason; the sweeps' indicators (sums of
squares of differences) are not."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import orc
from helpers import interior, rel_linf, smooth_periodic_state
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


@pytest.fixture(scope="module")
def extended(tmp_path_factory):
    """rhs(o, met, prim) by the oracle's source with every double replaced by long double."""
    d = tmp_path_factory.mktemp("extended")
    here = os.path.dirname(os.path.abspath(orc.__file__))
    for f in ("shx_oracle.c", "shx_oracle.h"):
        with open(os.path.join(here, f)) as src:
            (d / f).write_text(src.read().replace("long double", "double"))
    heads = ("float.h", "omp.h", "math.h", "stdlib.h", "string.h", "tgmath.h")
    (d / "pre.h").write_text("".join(f"#include <{h}>\n" for h in heads) + "#define double long double\n")
    lib = str(d / "libextended.so")
    subprocess.run(["gcc", "-O2", "-std=gnu99", "-fopenmp", "-fPIC", "-shared", "-ffp-contract=off", "-w", "-I", str(d),
                    "-include", str(d / "pre.h"), str(d / "shx_oracle.c"), "-o", lib, "-lm"], check=True)
    L = ctypes.CDLL(lib)
    L.orc_rhs_b.argtypes = [ctypes.c_void_p] * 6

    def wide(t):
        if t is ctypes.c_double:
            return ctypes.c_longdouble
        if getattr(t, "_type_", None) is ctypes.c_double:
            return ctypes.c_longdouble * t._length_
        return t

    class Cfg(ctypes.Structure):
        _fields_ = [(name, wide(t)) for name, t in orc.OrcCfg._fields_]

    def rhs(o, met, prim):
        c = Cfg()
        for name, t in orc.OrcCfg._fields_:
            v = getattr(o.c, name)
            if hasattr(v, "__len__"):
                getattr(c, name)[:] = list(v)
            else:
                setattr(c, name, v)
        assert L.orc_define(ctypes.byref(c)) == 0
        arrs = [[a.astype(np.longdouble) for a in f] for f in (met, prim, o.zeros(30))]
        ptrs = [(ctypes.c_void_p * len(f))(*[a.ctypes.data for a in f]) for f in arrs]
        L.orc_rhs_b(ctypes.byref(c), *ptrs, None, None)
        return [a.astype(np.float64) for a in arrs[2][20:25]]
    return rhs


@pytest.mark.parametrize("n,quirks", [((10, 31, 63), 3), ((16, 15, 64), 3), ((32, 10, 65), 3), ((17, 10, 33), 0)])
def test_w9_tile_edges(extended, n, quirks):
    o = orc.Oracle(dims=3, S=9, n=n, quirks=quirks, mach=0.5, reynolds=2000.0)
    coords = cases.periodic_ext_coords(3, 9, n, cases.sine_bump_3d(0.05))
    met = o.metric_from_coords(*coords)
    o.ghost_periodic(met)
    prim = smooth_periodic_state(o, n, 5, 0.5)
    want = extended(o, met, prim)
    with shockx.Case(dims=3, space_order=9, time_order=4, n=n, mach=0.5, reynolds=2000.0, quirks=quirks) as c:
        c.build_metric(*coords)
        c.upload_state(prim)
        got = c.rhs()
    assert max(rel_linf(got, want, interior(o, 3, n))) <= 1e-12
