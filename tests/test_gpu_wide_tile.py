"""The 256 x 320 tile (two-term slices or responsibilities) at ragged column counts, with one-term and two-term counts,
in the logits and in the dense M-step, against the 128 x 128 register-staged kernel (mfma_tile = 1), bit for bit."""
import numpy as np
import pytest

import emc_amd

pytestmark = pytest.mark.gpu


def problem(L, I):
    truth = emc_amd.synth_model(L, 60, 0.19 * L, 3)
    coords, mask = emc_amd.coords_flat(L), emc_amd.mask_annulus(L, 2.0, L / 2)
    K, _ = emc_amd.synth_patterns(truth, L, coords, mask, I, 400.0, 4)
    return truth, coords, mask, np.minimum(K, 255)


# 2,561 columns: one valid column in the last tile; 2,700: a partial one; 3,200: ten whole tiles
@pytest.mark.parametrize("I", [2561, 2700, 3200])
@pytest.mark.parametrize("split,count_bytes", [(False, 0), (False, 2), (True, 0)])
def test_wide_tile_logits(I, split, count_bytes):
    L, S = 24, 6300
    print(f"[wide tile] logits {S} x {I} split={split} count_bytes={count_bytes}", flush=True)
    truth, coords, mask, K = problem(L, I)
    Kp = emc_amd.normalize_patterns(K, mask) if split else K
    q, w = emc_amd.rotations(5)
    out = []
    for tile in (0, 1):
        with emc_amd.Engine(L, S, I, precision="bf16x2", mfma_tile=tile, count_bytes=count_bytes) as e:
            e.setup(q, w, coords, mask, Kp, truth)
            e.logl()
            R = e.get_logl()
            e.normalize_resp()
            out.append((R, e.get_lse()))
    assert np.array_equal(out[0][0], out[1][0])
    assert np.allclose(out[0][1], out[1][1], rtol=2e-6, atol=0)  # band sums on exp2 in FP32 lanes against expf


@pytest.mark.parametrize("split", [False, True])
def test_wide_tile_mstep(split):
    L, S, I = 64, 6300, 96  # 3,200 padded pixels: ten tiles
    print(f"[wide tile] M-step {S} x {I} split={split}", flush=True)
    truth, coords, mask, K = problem(L, I)
    Kp = emc_amd.normalize_patterns(K, mask) if split else K
    q, w = emc_amd.rotations(5)
    P = np.random.default_rng(1).random((S, I)).astype(np.float32)
    out = []
    for tile in (0, 1):
        with emc_amd.Engine(L, S, I, precision="bf16x2", mfma_tile=tile, mstep="dense", insert="binned") as e:
            e.setup(q, w, coords, mask, Kp, truth)
            e.set_resp(P)
            e.maximize()
            e.compress()
            out.append(e.get_model())
    for a, b in zip(*out):
        assert np.array_equal(a, b)
