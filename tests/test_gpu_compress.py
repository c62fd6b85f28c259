"""The compress's axis passes at sides that are not a multiple of the tile (odd, smaller than a quad of lines,
16-byte stores or not) against the FP64 oracle, and on the eight-line tiles of large sides against the
separable form of the blur."""
import numpy as np
import pytest

import emc_amd

pytestmark = pytest.mark.gpu


def compress(L, Mnum, Wt, sigma):
    with emc_amd.Engine(L, 4, 4, blur_sigma=sigma) as e:
        e.set_mstep_sums(Mnum, Wt)
        avg = e.compress()
        return e.get_model()[0], avg


@pytest.mark.parametrize("sigma", [0.0, 0.6])
@pytest.mark.parametrize("L", [4, 5, 7, 18, 33, 64, 66])
def test_compress_sides_match_oracle(orc, L, sigma):
    print(f"[compress] side {L} sigma {sigma}", flush=True)
    rng = np.random.default_rng(L)
    Wt = rng.uniform(0.5, 3.0, L ** 3).astype(np.float32)
    Wt[rng.random(L ** 3) < 0.2] = 0.0
    Mnum = (rng.uniform(0.0, 2.0, L ** 3) * Wt).astype(np.float32)
    M, avg = compress(L, Mnum, Wt, sigma)
    Mo, avgo, _ = orc.normalize_support(orc.compress(Mnum.astype(np.float64), Wt.astype(np.float64)), Wt.astype(np.float64))
    if sigma > 0:
        Mo = orc.blur(Mo, L, sigma)
    assert abs(avg - avgo) <= 1e-6 * avgo
    assert np.array_equal(M < 0, Mo < 0)
    # float inputs and taps, L products per axis in float: 3 (L / 2 + 2) half-ulps at most, far fewer in the mean
    assert float(np.linalg.norm(M - Mo) / np.linalg.norm(Mo)) < 1e-6


def test_compress_large_side_is_the_separable_blur():
    L, sigma = 516, 0.7
    print(f"[compress] side {L}, separable model", flush=True)
    rng = np.random.default_rng(1)
    f = [rng.uniform(0.5, 1.5, L) for _ in range(3)]
    k = np.minimum(np.arange(L), L - np.arange(L))
    h = np.exp(-2 * np.pi ** 2 * sigma ** 2 * k ** 2 / L ** 2)
    outer = lambda a: (a[0][:, None, None].astype(np.float32) * a[1][None, :, None].astype(np.float32) *  # noqa: E731
                       a[2][None, None, :].astype(np.float32)).reshape(-1)
    M, avg = compress(L, outer(f), np.ones(L ** 3, np.float32), sigma)
    mean = np.prod([v.mean() for v in f])
    b = [np.fft.ifft(np.fft.fft(v) * h).real for v in f]
    b[0] = b[0] / mean
    assert abs(avg - mean) < 1e-5 * mean
    ref = outer(b)
    assert float(np.linalg.norm(M - ref) / np.linalg.norm(ref)) < 2e-6
