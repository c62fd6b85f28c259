"""A voxel keeps its value through the blur where the scaled value is negative: a negative quotient that the scale takes to
zero is blurred like the others (odd side; side of a multiple of 4, whose stores are 16 bytes wide)."""
import numpy as np
import pytest

import emc_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [20, 21])
def test_scaled_sign_decides(L):
    print(f"[compress signs] side {L}", flush=True)
    sigma, v = 0.6, (L // 2 * L + 3) * L + 5
    Wt = np.ones(L ** 3, np.float32)
    Mnum = np.full(L ** 3, 1.0e9, np.float32)
    Mnum[v] = -1.0e-37  # a normal float; over the average of 1e9 it is -1e-46: minus zero as a float
    Mnum[v + 7] = -1.0e9  # stays negative: kept
    with emc_amd.Engine(L, 4, 4, blur_sigma=sigma) as e:
        e.set_mstep_sums(Mnum, Wt)
        avg = e.compress()
        M = e.get_model()[0].astype(np.float64)
    n = L ** 3
    assert abs(avg - 1.0e9 * (n - 3) / n) < 1e3
    k = np.minimum(np.arange(L), L - np.arange(L))
    h = np.exp(-2 * np.pi ** 2 * sigma ** 2 * k ** 2 / L ** 2)
    f = np.where(Mnum < 0, 0.0, 1.0e9 / avg).reshape(L, L, L)
    b = np.fft.ifftn(np.fft.fftn(f) * h[:, None, None] * h[None, :, None] * h[None, None, :]).real.reshape(-1)
    b[v + 7] = -1.0e9 / avg
    assert b[v] > 0.1
    # float taps and products of sums of order 1: three axes of L terms
    assert np.abs(M - b).max() < 3 * L * 2.0 ** -23
