"""emc_get_model into pinned memory, which the device copies into directly, into one pinned and one pageable array, and
into a single array of at most and of more than one slot."""
import ctypes as C

import numpy as np
import pytest

import emc_amd
from emc_amd._lib import check, lib

pytestmark = pytest.mark.gpu


def hip_runtime():
    """The HIP runtime libemc.so is linked against (already mapped into this process)."""
    lib()
    with open("/proc/self/maps") as f:
        paths = {ln.split()[-1] for ln in f if "libamdhip64" in ln}
    h = C.CDLL(sorted(paths)[0])
    h.hipHostMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t, C.c_uint]
    h.hipHostFree.argtypes = [C.c_void_p]
    return h


@pytest.mark.parametrize("L", [4, 40, 41, 50, 51, 64, 102])  # both arrays, then one, of at most a slot of 131,072 floats and above
def test_model_reads_back_into_any_memory(L):
    print(f"[read out] side {L}, pinned", flush=True)
    hip, n = hip_runtime(), L ** 3
    rng = np.random.default_rng(L)
    M, W = rng.random(n, dtype=np.float32), rng.random(n, dtype=np.float32)
    pinned = []
    try:
        for _ in range(2):
            p = C.c_void_p()
            assert hip.hipHostMalloc(C.byref(p), 4 * n, 0) == 0
            pinned.append((p, np.ctypeslib.as_array(C.cast(p, C.POINTER(C.c_float)), (n,))))
        pageable = [(lambda a: (a.ctypes.data_as(C.c_void_p), a))(np.empty(n, np.float32)) for _ in range(2)]
        none = (None, None)
        with emc_amd.Engine(L, 4, 4) as e:
            e.set_mstep_sums(M, W)
            e.set_model(M)
            for a, b in ((pinned[0], pinned[1]), (pinned[0], pageable[1]), (pageable[0], pinned[1]), (pinned[0], none),
                         (none, pinned[1]), (pageable[0], none), (none, pageable[1]), (pageable[0], pageable[1])):
                for x in (a[1], b[1]):
                    if x is not None:
                        x[:] = 0.0
                check(lib().emc_get_model(e._h, a[0], b[0]))
                assert a[1] is None or np.array_equal(a[1], M)
                assert b[1] is None or np.array_equal(b[1], W)
    finally:
        for p, _ in pinned:
            hip.hipHostFree(p)
