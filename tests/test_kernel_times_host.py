"""Kernel classes that shx_kernel_times reports, over a stand-in runtime: a step's launches by what they
are, and no class that nothing launches."""
import pytest

import hoststub


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    return hoststub.build(tmp_path_factory.mktemp("stub"))


@pytest.mark.parametrize("n,kw,want", [
    ((16, 17, 1), "", {"plane_stage": 4}),
    ((16, 17, 1), "bc=(2, 3, 0, 0, 0, 0)",
     {"ghost_values": 4, "ghost_faces": 8, "plane_stage": 4}),
    ((12, 11, 10), "inviscid=True", {"weno_xi": 4, "weno_eta": 4, "weno_zeta": 4}),
    ((12, 11, 10), "", {"ghost_values": 4, "weno_xi": 4, "visc_grad_xi": 4, "weno_visc_eta": 4, "weno_visc_zeta": 4}),
    ((12, 11, 10), "space_order=9", {"ghost_values": 4, "weno_xi": 4, "weno_eta": 4, "visc_grad": 4, "visc_xi": 4,
                                     "visc_eta": 4, "weno_visc_zeta": 4})])
def test_classes_of_a_step(stub, n, kw, want):
    r = hoststub.run(stub, f"""
c = case({n}, {kw})
c.set_timing(True)
c.calc_runge_kutta(1e-3)
result = [{{k: v[1] for k, v in c.kernel_times().items() if v[1]}}, "rk_update" in c.kernel_times(),
          "rk" in shockx.BATCH_CLASSES]
""")
    assert r == [want, False, False]
