"""More patterns than a launch's second dimension has workgroups for (65,535, at four patterns each), on a detector of
less than 1,024 pixels.  A flat model of ones (nearest voxel) leaves each pattern's log-sum-exp to its constant: the
logarithm of the total weight, plus its counts times log fluence, less the expected counts."""
import numpy as np
import pytest

import emc_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("I,split", [(1001, False), (262201, False), (262201, True)])
def test_every_pattern_gets_its_constant(I, split):
    print(f"[many patterns] {I} split={split}", flush=True)
    L, S, phi = 8, 6, 2.0
    coords, mask = emc_amd.coords_flat(L), emc_amd.mask_annulus(L, 0.5, 3.0)  # within the model at any orientation
    K = np.random.default_rng(3).integers(0, 9, (I, L * L)).astype(np.int32)
    K[:, np.flatnonzero(mask)[0]] = 300 if split else 7
    q, _ = emc_amd.rotations(1)
    w = np.arange(1, S + 1, dtype=np.float32)
    with emc_amd.Engine(L, S, I, interp="nearest", fluence=phi) as e:
        e.setup(q[:S], w, coords, mask, K, np.ones(L ** 3, np.float32))
        e.logl()
        e.normalize_resp()
        lse = e.get_lse()
    Pa = int(mask.sum())
    # the column means are log phi as a float; the logits are the weights' logarithms as floats
    cm = float(np.float32(np.log(phi)))
    logw = np.log(w.astype(np.float64)).astype(np.float32).astype(np.float64)
    want = np.log(np.exp(logw).sum()) + K[:, mask != 0].sum(1) * cm - phi * Pa
    # float logarithms and exponentials of the S weights (2^-22 each, the largest logarithm 1.8); FP32 sums of the S terms
    assert np.abs(lse - want).max() < 2e-6


def test_many_rotations_get_their_bias():
    """More rotations than one step of the bias pass's workgroups (512 x 256) covers."""
    L, S, I, phi = 8, 131073 + 700, 3, 2.0
    print(f"[many rotations] {S}", flush=True)
    coords, mask = emc_amd.coords_flat(L), emc_amd.mask_annulus(L, 0.5, 3.0)
    K = np.random.default_rng(3).integers(0, 9, (I, L * L)).astype(np.int32)
    q0, _ = emc_amd.rotations(2)
    q = q0[np.arange(S) % len(q0)]
    w = (0.5 + np.random.default_rng(4).random(S)).astype(np.float32)
    with emc_amd.Engine(L, S, I, interp="nearest", fluence=phi, keep_logits=1) as e:
        e.setup(q, w, coords, mask, K, np.ones(L ** 3, np.float32))
        e.logl()
        R = e.get_logl()
        e.normalize_resp()
        lse = e.get_lse()
    cst = K[:, mask != 0].sum(1) * float(np.float32(np.log(phi))) - phi * int(mask.sum())
    want = np.log(w.astype(np.float64))[:, None] + cst[None, :]
    assert np.abs(R - want).max() < 2e-5  # logits of up to 200 as floats (2^-17 each), and the float logarithm
    logw = np.log(w.astype(np.float64)).astype(np.float32).astype(np.float64)
    assert np.abs(lse - (np.log(np.exp(logw).sum()) + cst)).max() < 2e-6  # float exponentials, FP32 sums of 32 terms
