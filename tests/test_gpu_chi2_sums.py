"""chi^2 sums on the larger tiles against those on 64 x 64 tiles, bit for bit: the products with the high and with the low
half of the squared counts are summed apart and added once, whatever the tile (in one chain the low products' roundings
would fall on the high sum).  A pattern's logits do not depend on the other patterns, so a small set gives the bits of
the same patterns in a large one."""
import numpy as np
import pytest

import emc_amd
from tile_route import logl_tile, pad, tile

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("diff,scaling,normalized", [("poisson", 1, False), ("poisson", 1, True), ("absolute", 0, True),
                                                     ("relative", 0, True)])
@pytest.mark.parametrize("prec", ["bf16x2", "bf16x3"])
def test_large_tiles_give_the_bits_of_the_small_ones(diff, scaling, normalized, prec):
    L, few = 24, 500
    truth = emc_amd.synth_model(L, 60, 4.5, 3)
    coords, mask = emc_amd.coords_flat(L), emc_amd.mask_annulus(L, 2.0, 12.0)
    q, w = emc_amd.rotations(5)  # 6,300
    S = len(q)
    K, _ = emc_amd.synth_patterns(truth, L, coords, mask, 2700, 900.0, 4)
    Kp = emc_amd.normalize_patterns(K, mask) if normalized else np.minimum(K, 255)
    model = truth if scaling else truth * np.float32(Kp[:, mask != 0].mean() / truth[truth > 0].mean())
    assert tile(pad(S, 256), pad(few, 256), 2, 2) == "64x64"
    out = {}
    for I in (few, 1000, 2001, 2700):
        print(f"[chi2 sums] {diff} scaling {scaling} {prec} {S} x {I}", flush=True)
        assert I == few or logl_tile(S, I, prec, True) != "64x64"
        with emc_amd.Engine(L, S, I, diff=diff, scaling=scaling, precision=prec) as e:
            e.setup(q, w, coords, mask, Kp[:I], model)
            e.logl(0.3)
            R = e.get_logl_block(0, S, 0, few)
            e.normalize_resp()
            out[I] = (R, e.get_resp_block(0, S, 0, few))
    for I in (1000, 2001, 2700):
        assert np.array_equal(out[I][0], out[few][0]), I
        assert np.array_equal(out[I][1], out[few][1]), I
