"""Log-sum-exps with two-term counts: every term of a pattern's sum over rotations is added in FP64, whatever the tile
of the contraction.  A flat model of ones (nearest voxel, fluence 1) makes every logit the logarithm of its
rotation's weight, so the sum is known: in each 64 rotations two weigh 1 and the others 2^-24.5, which an FP32 sum
that holds a 1 drops (together 1.3e-6 of the sum)."""
import numpy as np
import pytest

import emc_amd
from tile_route import logl_tile

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S,I,prec,tile", [
    (1380, 500, "bf16x2", "64x64"), (3240, 2560, "bf16x2", "128x128"), (1380, 2560, "bf16x2", "256x128"),
    (6300, 2001, "bf16x2", "256x256"), (6300, 2700, "bf16x2", "256x320"),
    (1380, 500, "bf16x3", "64x64"), (3240, 2560, "bf16x3", "128x128"), (6300, 2700, "bf16x3", "256x128"),
    (6300, 2001, "bf16x3", "256x256")])
def test_every_term_counts(S, I, prec, tile):
    print(f"[split sums] {S} x {I} {prec} {tile}", flush=True)
    assert logl_tile(S, I, prec, True) == tile
    L = 24
    coords, mask = emc_amd.coords_flat(L), emc_amd.mask_annulus(L, 2.0, 10.0)  # within the model at any orientation
    K = np.random.default_rng(2).integers(0, 4, (I, L * L)).astype(np.int32)
    K[:, np.flatnonzero(mask)[0]] = 300  # above 256: two BF16 terms
    q, _ = emc_amd.rotations(5)
    w = np.full(S, 2.0 ** -24.5, np.float32)
    w[0::64] = 1.0  # rows of the first accumulator register of the two half-wavefronts
    w[4::64] = 1.0
    with emc_amd.Engine(L, S, I, precision=prec, interp="nearest", fluence=1.0) as e:
        e.setup(q[:S], w, coords, mask, K, np.ones(L ** 3, np.float32))
        e.logl()
        e.normalize_resp()
        lse = e.get_lse()
    logw = np.log(w.astype(np.float64)).astype(np.float32).astype(np.float64)
    want = np.log(np.exp(logw).sum()) - float(mask.sum())
    # the small terms, 1.3e-6 of the sum, carry the float logarithm's 2^-20 and the float exponential's 2^-22; an lse near
    # 300 in FP64 6e-14
    assert np.abs(lse - want).max() < 1e-11
