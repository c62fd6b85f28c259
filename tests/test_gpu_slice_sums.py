"""Slice sums T under rotation chunks of a size that is no multiple of 8, where eight rows of the responsibilities pass
may lie in two of the 64-row bands of the small tiles: each responsibility is added in FP64 there too, as in the pass
over one chunk.  Every voxel is 1 or 1e-30 (nearest voxel) and every pattern's photons lie in one pixel, so its
logits take two values 207 apart and its n rotations of the larger one have responsibility 1/n each, whatever
the chunks: the sums agree to FP64 rounding."""
import numpy as np
import pytest

import emc_amd
from tile_route import logl_tile

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chunk", [459, 581, 701])
@pytest.mark.parametrize("prec", ["bf16x2", "bf16x3"])
def test_rows_across_small_bands(chunk, prec):
    print(f"[slice sums] chunk {chunk} {prec}", flush=True)
    L, I = 16, 200
    q, _ = emc_amd.rotations(3)  # 1,380
    S = len(q)
    assert logl_tile(S, I, prec, False, chunk) == logl_tile(S, I, prec, False) == "64x64"
    coords, mask = emc_amd.coords_flat(L), emc_amd.mask_annulus(L, 1.0, 6.5)  # within the model at any orientation
    model = np.where(np.random.default_rng(5).random(L ** 3) < 0.5, 1.0, 1e-30).astype(np.float32)
    pix = np.flatnonzero(mask)
    K = np.zeros((I, L * L), np.int32)
    K[np.arange(I), pix[np.arange(I) % len(pix)]] = 3  # neighbouring patterns have different n
    T = []
    for c in (0, chunk):
        with emc_amd.Engine(L, S, I, precision=prec, interp="nearest", slice_chunk=c, fluence=1e-30) as e:
            e.setup(q, np.ones(S, np.float32), coords, mask, K, model)
            e.logl()
            e.normalize_resp()
            T.append(e.get_slice_weights())
    r0 = np.arange(S) // 8 * 8
    rl = np.minimum(r0 + 7, S - 1)
    inside = (r0 // chunk == rl // chunk) & (r0 % chunk // 256 == rl % chunk // 256)
    assert (inside & (r0 % chunk // 64 != rl % chunk // 64)).sum() >= 8
    # sums of 200 terms in FP64: below 200 x 2^-53; float sums of four neighbours' are off by 1e-9 and more
    assert np.abs(T[1] - T[0])[inside].max() / T[0].max() < 1e-13
