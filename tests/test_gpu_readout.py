"""emc_get_model's pieces: one slot for both arrays, pieces that straddle the two, several rounds of the slots, and
the sizes that several threads copy; with either array left out; two threads reading one context."""
import ctypes as C
import threading

import numpy as np
import pytest

import emc_amd
from emc_amd._lib import check, lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [4, 41, 51, 64, 81, 101, 130])
def test_model_reads_back(L):
    print(f"[read out] side {L}", flush=True)
    rng = np.random.default_rng(L)
    M, W = rng.random(L ** 3, dtype=np.float32), rng.random(L ** 3, dtype=np.float32)
    with emc_amd.Engine(L, 4, 4) as e:
        e.set_mstep_sums(M, W)
        e.set_model(M)
        a, b = e.get_model()
        assert np.array_equal(a, M) and np.array_equal(b, W)
        p = lambda x: x.ctypes.data_as(C.c_void_p)  # noqa: E731
        a[:], b[:] = 0.0, 0.0
        check(lib().emc_get_model(e._h, p(a), None))
        check(lib().emc_get_model(e._h, None, p(b)))
        check(lib().emc_get_model(e._h, None, None))
        assert np.array_equal(a, M) and np.array_equal(b, W)
        out = [None, None]

        def read(k):
            for _ in range(3):
                out[k] = e.get_model()

        ts = [threading.Thread(target=read, args=(k,)) for k in range(2)]
        [t.start() for t in ts]
        [t.join() for t in ts]
        for x, y in out:
            assert np.array_equal(x, M) and np.array_equal(y, W)
