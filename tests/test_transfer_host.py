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
