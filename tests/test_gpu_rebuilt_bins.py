"""Insertion after the mask was replaced: the unit sums' memory is kept from one build of the bins to the next, grows
where the new build has more units and is given up where it has too many to be split; the model and its weights
are bit for bit those of an engine that has had no other mask."""
import numpy as np
import pytest

import emc_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("interp", ["trilinear", "nearest"])
def test_insertion_after_a_new_mask(interp):
    L, I = 32, 16
    q, w = emc_amd.rotations(5)
    S = len(q)
    coords = emc_amd.coords_flat(L)
    truth = emc_amd.synth_model(L, 100, 0.19 * L, 11)
    # units of 4,096 pairs: about 200 (split), 650 (split, more memory), 1,270 (not split), 200 (split anew), 80 (fits)
    masks = [emc_amd.mask_annulus(L, 1.0, r) for r in (6.0, 11.0, 16.0, 6.0, 3.0)]
    assert S * masks[1].sum() < 1000 * 4096 and S * masks[2].sum() > 1024 * 4096
    K, _ = emc_amd.synth_patterns(truth, L, coords, masks[2], I, 500.0, 12)

    def one(e, m):
        e.set_mask(m)
        e.set_patterns(K)
        e.set_model(truth)
        e.iterate(5)
        return e.get_model()

    with emc_amd.Engine(L, S, I, blur_sigma=0.0, interp=interp) as e:
        e.setup(q, w, coords, masks[0], K, truth)
        for k, m in enumerate(masks):
            print(f"[rebuilt bins] {interp} mask {k}", flush=True)
            got = one(e, m)
            with emc_amd.Engine(L, S, I, blur_sigma=0.0, interp=interp) as f:
                f.setup(q, w, coords, m, K, truth)
                want = one(f, m)
            for a, b in zip(got, want):
                assert np.array_equal(a, b)
