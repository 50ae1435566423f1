"""Downloads into arrays that coincide: the fields are written in order, so the array holds the last one,
whether the call's chunks are one thread's or several threads'."""
import ctypes

import numpy as np
import pytest

from shock_amd import shockx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(20, 20, 1), (18, 19, 20), (56, 60, 50)])
def test_last_field_wins(n):
    rng = np.random.default_rng(n[0])
    with shockx.Case(dims=2 if n[2] == 1 else 3, n=n) as c:
        state = [rng.random(c.shape) + 0.5 for _ in range(5)]
        met = [rng.random(c.shape) for _ in range(10)]
        c.upload_state(state)
        c.upload_metric(met)
        rho, rest = np.zeros(c.shape), np.zeros(c.shape)
        for _ in range(20):
            ptr = (ctypes.c_void_p * 5)(rho.ctypes.data, *[rest.ctypes.data] * 4)
            assert shockx.lib().shx_download_state(c.h, ptr) == 0
            assert np.array_equal(rho, state[0]) and np.array_equal(rest, state[4])
            ptr = (ctypes.c_void_p * 10)(*[rest.ctypes.data] * 10)
            assert shockx.lib().shx_download_metric(c.h, ptr) == 0
            assert np.array_equal(rest, met[9])
