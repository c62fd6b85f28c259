"""Binned insertion with one unit a workgroup and with blocks of four, with and without the grouping pass, against the
atomic insertion of the same slice sums."""
import numpy as np
import pytest

import emc_amd

pytestmark = pytest.mark.gpu

# L, rotations, chunk: one unit a workgroup without and with a grouping pass and with a ragged last chunk, then blocks of
# four units
CASES = [(6, 3, 0), (12, 60, 0), (24, 420, 0), (17, 420, 100), (32, 3240, 0), (45, 3240, 1300), (64, 12000, 0)]


@pytest.mark.parametrize("interp", ["trilinear", "nearest"])
@pytest.mark.parametrize("L,S,chunk", CASES)
def test_binned_insertion_matches_atomic(L, S, chunk, interp):
    print(f"[insert] side {L} rotations {S} chunk {chunk} {interp}", flush=True)
    rng = np.random.default_rng(L + S)
    q = rng.standard_normal((S, 4))
    q = (q / np.linalg.norm(q, axis=1, keepdims=True)).astype(np.float32)
    w = np.full(S, 1.0 / S, np.float32)
    truth = emc_amd.synth_model(L, max(8, L), 3.0, 3)
    coords, mask = emc_amd.coords_flat(L), emc_amd.mask_annulus(L, 1.0, L / 2)
    I = 16
    K, _ = emc_amd.synth_patterns(truth, L, coords, mask, I, 300.0, 4)
    P = rng.random((S, I)).astype(np.float32)
    P[rng.random(S) < 0.1] = 0.0  # rotations without weight are left out (T_s <= 1e-10)
    sums = []
    for insert in ("atomic", "binned", "binned"):
        with emc_amd.Engine(L, S, I, interp=interp, insert=insert, slice_chunk=chunk) as e:
            e.setup(q, w, coords, mask, K, truth)
            e.set_resp(P)
            e.maximize()
            e.compress()
            sums.append(e.get_model())
    # about n positive float terms a voxel, added in another order: a random walk of n half-ulps of the partial sums
    # in the weights, two of them and the quotient's own rounding in the model
    n = 8.0 * S * int((np.asarray(mask) > 0).sum()) / L ** 3
    for (a, b, c), k in zip(zip(*sums), (2, 1)):
        assert np.array_equal(b, c)
        assert np.array_equal(a > 0, b > 0)
        assert float(np.linalg.norm(a.astype(np.float64) - b) / np.linalg.norm(a)) < 2 * k * np.sqrt(n + 16) * 2.0 ** -24
