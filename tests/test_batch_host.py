"""Host side of shx_batch_set_tau over a stand-in runtime: where a case has changed under the batch what
its launches are, tables and graph are replaced together, and a failed replacement leaves the batch as
it was."""
import pytest

import hoststub


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    return hoststub.build(tmp_path_factory.mktemp("stub"))


# launches of a step before and after the case keeps its pressure: 2D, four stages of k_plane and the
# first one's ghost fill, then a fill (inviscid: and a pass for p and c) before every stage; 3D inviscid,
# three sweeps a stage in k_plane's place; a case whose ghosts are filled anyway
@pytest.mark.parametrize("n,kw,before,after", [
    ((32, 32, 1), "inviscid=False", 5, 8), ((17, 40, 1), "inviscid=False, time_order=3", 4, 6),
    ((32, 32, 1), "inviscid=True", 5, 12), ((12, 11, 10), "inviscid=True", 13, 20),
    ((12, 11, 10), "inviscid=False", 20, 20)])
def test_pressure_kept_under_a_batch(stub, n, kw, before, after):
    r = hoststub.run(stub, f"""
c, d = case({n}, {kw}), case((20, 20, 1))
b = shockx.Batch([c], [1e-3])
b.run(1)
result = [stub.stub_graph_nodes()]
c.post()
b.set_tau([2e-3])
b.run(1)
result += [stub.stub_graph_nodes()]
b.set_tau([1e-3])
b.run(1)
result += [stub.stub_graph_nodes(), stub.stub_overruns(), stub.stub_graph_bad()]
""")
    assert r == [before, after, after, 0, 0]


def test_tuned_case_leaves_its_group(stub):
    """Two cases of one group; a tile picked for one of them splits the group."""
    r = hoststub.run(stub, """
c, d = case((16, 16, 16)), case((16, 16, 16))
b = shockx.Batch([c, d], [1e-3, 1e-3])
b.run(1)
result = [stub.stub_graph_nodes()]
c.tune(1)
b.set_tau([2e-3, 2e-3])
b.run(1)
result += [stub.stub_graph_nodes() >= result[0], stub.stub_overruns(), stub.stub_graph_bad()]
""")
    assert r[1:] == [True, 0, 0]


def test_failed_replacement_keeps_the_batch(stub):
    r = hoststub.run(stub, """
c = case((32, 32, 1))
b = shockx.Batch([c], [1e-3])
c.post()
stub.stub_fail_captures(1)
try:
    b.set_tau([2e-3])
    result = ["taken"]
except shockx.ShxError:
    result = ["refused"]
b.run(1)
result += [stub.stub_graph_nodes()]
b.set_tau([2e-3])
b.run(1)
result += [stub.stub_graph_nodes(), stub.stub_overruns(), stub.stub_graph_bad()]
""")
    assert r == ["refused", 5, 8, 0, 0]
