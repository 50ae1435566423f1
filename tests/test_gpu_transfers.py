"""Host transfers: states and metrics go up and come back bit for bit at sizes below, at and above the
staging chunks (one chunk on the calling thread, several, several per slot and thread), in both
dimensions, and an upload follows a download through the same slots."""
import numpy as np
import pytest

from shock_amd import shockx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(6, 6, 1), (70, 88, 1), (160, 150, 1), (6, 6, 6), (26, 25, 26), (42, 51, 37), (90, 86, 95)])
def test_round_trip(n):
    dims = 2 if n[2] == 1 else 3
    rng = np.random.default_rng(n[0])
    with shockx.Case(dims=dims, n=n) as c:
        for _ in range(2):
            state = [rng.random(c.shape) + 0.5 for _ in range(5)]
            met = [rng.random(c.shape) for _ in range(10)]
            c.upload_state(state)
            c.upload_metric(met)
            got, gmet = c.download_state(), c.download_metric()
            assert all(np.array_equal(a, b) for a, b in zip(got + gmet, state + met))
