"""Host side of state transfers over a stand-in runtime."""
import pytest

import hoststub


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    return hoststub.build(tmp_path_factory.mktemp("stub"))


@pytest.mark.parametrize("no_threads", [0, 1])
def test_caller_keeps_its_device(stub, no_threads):
    """A case of device 0 used while device 1 is current, with and without threads to be had."""
    r = hoststub.run(stub, f"""
c = case((48, 48, 48))
stub.stub_no_threads({no_threads})
stub.hipSetDevice(1)
d = ctypes.c_int(-1)
result = []
for call in (lambda: c.upload_state([np.ones(c.shape)] * 5), c.download_state, c.download_metric):
    call()
    stub.hipGetDevice(ctypes.byref(d))
    result.append(d.value)
""")
    assert r == [1, 1, 1]


# pinned memory of a case after its state has gone up and come back, in fields of the case (doubles of
# the padded grid): the whole state where that is 256 KB at most, else two slots of a field or of a third
# of the state, and with several threads half the state or four slots of 2 MB
@pytest.mark.parametrize("n,most", [((32, 32, 1), 5), ((64, 64, 1), 5), ((90, 90, 1), 3.4), ((18, 18, 18), 3.4),
                                    ((24, 24, 24), 2.5), ((32, 32, 32), 2), ((42, 42, 42), 2), ((48, 48, 48), 2.51),
                                    ((97, 85, 106), 1.1)])
def test_pinned_memory(stub, n, most):
    r = hoststub.run(stub, f"""
c = shockx.Case(dims={2 if n[2] == 1 else 3}, n={n})
before, ev = stub.stub_pinned(), stub.stub_events()
c.upload_state([np.ones(c.shape)] * 5)
c.download_state()
slots = stub.stub_events() - ev
field = 8 * int(np.prod(c.shape))
pinned = stub.stub_pinned() - before
c.close()
result = [pinned / field, pinned, slots, stub.stub_pinned(), stub.stub_overruns()]
""")
    fields, pinned, slots, left, overruns = r
    assert fields <= most and pinned <= 8 << 20 and slots <= 4
    assert left == 0 and overruns == 0


@pytest.mark.parametrize("n", [(32, 32, 1), (18, 18, 18), (42, 42, 42), (48, 48, 48), (97, 85, 106)])
@pytest.mark.parametrize("threads", [True, False])
def test_every_transfer_has_its_slots(stub, n, threads):
    """Each kind of transfer first (one, five and ten fields): every chunk's copy stays in its slot."""
    r = hoststub.run(stub, f"""
stub.stub_no_threads({int(not threads)})
result = 0
for first in range(3):
    c = shockx.Case(dims={2 if n[2] == 1 else 3}, n={n})
    one = [np.ones(c.shape)] * 10
    calls = [lambda: c.upload_state(one[:5]), lambda: c.upload_metric(one), lambda: c.upload_boundary_state(one[:6])]
    for q in range(3):
        calls[(first + q) % 3]()
    c.download_state(); c.download_metric()
    c.close()
result = [stub.stub_overruns(), stub.stub_pinned()]
""")
    assert r == [0, 0]
