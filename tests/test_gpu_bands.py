"""Softmax partials of the 64 x 64 contraction tiles (formed from the stored logits) against those of the 256-row
tiles' epilogue.  With a fixed fluence a pattern's logits, log-sum-exp and responsibilities do not depend on the
other patterns, so a small pattern set (64-row tiles) gives the bits of the same patterns in a large one (256-row
tiles): the partials' order is the same, and what a left-out group of logits would add is below exp(-128)."""
import numpy as np
import pytest

import emc_amd

pytestmark = pytest.mark.gpu


# a ragged last band and columns; rotation chunks (ragged last one); every logit kept
@pytest.mark.parametrize("I,chunk,keep", [(500, 0, 0), (33, 0, 0), (257, 1248, 0), (500, 1248, 1)])
def test_small_tiles_give_the_bits_of_the_large_ones(I, chunk, keep):
    print(f"[bands] {I} patterns chunk {chunk} keep {keep}", flush=True)
    L = 24
    truth = emc_amd.synth_model(L, 60, 4.5, 3)
    coords, mask = emc_amd.coords_flat(L), emc_amd.mask_annulus(L, 2.0, 12.0)
    K, _ = emc_amd.synth_patterns(truth, L, coords, mask, 3000, 900.0, 4)
    K = np.minimum(K, 255)
    q, w = emc_amd.rotations(5)  # 6,300
    out = []
    for n in (I, 3000):
        with emc_amd.Engine(L, q.shape[0], n, slice_chunk=chunk, fluence=900.0 / 400, keep_logits=keep) as e:
            e.setup(q, w, coords, mask, K[:n], truth)
            e.iterate(0)
            out.append((e.get_lse()[:I], e.get_resp_block(0, q.shape[0], 0, I)))
    assert np.array_equal(out[0][0], out[1][0])
    assert np.array_equal(out[0][1], out[1][1])
