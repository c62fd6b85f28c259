"""The slices that the statistics pass keeps: FP32 logits from them (one chunk covers the rotations) against those from
slices gathered chunk by chunk, bit for bit, also after the mask of the same engine shrinks; the chi^2 operands at
odd pixel counts and the pattern constants of each count form against the oracle."""
import numpy as np
import pytest

import emc_amd

pytestmark = pytest.mark.gpu


def problem(L, n, I, seed=5):
    truth = emc_amd.synth_model(L, 40, 3.0, 3)
    coords = emc_amd.coords_flat(L)
    masks = [emc_amd.mask_annulus(L, 1.0, L / 2), emc_amd.mask_annulus(L, 1.5, L / 3)]
    masks[1][np.flatnonzero(masks[1])[3]] = 0  # an odd pixel count
    K, _ = emc_amd.synth_patterns(truth, L, coords, masks[0], I, 300.0, seed)
    q, w = emc_amd.rotations(n)
    return truth, coords, masks, K, q, w


@pytest.mark.parametrize("interp", ["trilinear", "nearest"])
@pytest.mark.parametrize("diff,scaling", [("true_poisson", 0), ("poisson", 1), ("absolute", 0), ("relative", 0)])
@pytest.mark.parametrize("L,S", [(17, 61), (24, 420)])
def test_fp32_kept_slices_equal_gathered_ones(L, S, diff, scaling, interp):
    print(f"[kept slices] side {L} rotations {S} {diff} scaling={scaling} {interp}", flush=True)
    truth, coords, masks, K, q, w = problem(L, 2, 33)
    out = []
    for chunk in (0, 60):
        with emc_amd.Engine(L, S, 33, precision="fp32", diff=diff, scaling=scaling, interp=interp,
                            slice_chunk=chunk) as e:
            e.setup(q[:S], w[:S], coords, masks[0], K, truth)
            e.logl(0.3)
            a = e.get_logl()
            e.set_mask(masks[1])
            e.set_patterns(K)
            e.logl(0.3)
            out.append((a, e.get_logl()))
    for a, b in zip(*out):
        assert np.isfinite(a).all() and np.array_equal(a, b)


@pytest.mark.parametrize("diff,scaling", [("poisson", 1), ("absolute", 0), ("relative", 0)])
def test_chi2_operands_match_oracle(orc, diff, scaling):
    L, S, I = 17, 61, 40
    print(f"[chi2 operands] {diff} scaling={scaling}", flush=True)
    truth, coords, masks, K, q, w = problem(L, 2, I)
    assert int((masks[1] > 0).sum()) % 2 == 1
    for mask in masks:
        with emc_amd.Engine(L, S, I, precision="bf16x3", diff=diff, scaling=scaling) as e:
            e.setup(q[:S], w[:S], coords, mask, K, truth)
            e.logl(0.3)
            R = e.get_logl()
        W = orc.slices(truth.astype(np.float64), L, q[:S], coords, "trilinear")
        Kd = K.astype(np.float64)
        phi = orc.scaling(W, Kd, mask) if scaling else None
        Ro, _ = orc.logl(W, Kd, mask, w[:S].astype(np.float64), diff, sigma=0.3, phi0=1.0,
                         **({"phi": phi} if scaling else {}))
        # the expanded square of three-term operands: FP32 sums of a pattern's pixels, 1e-4 of its largest logit as
        # the other chi^2 tests on the matrix cores
        assert float(np.max(np.abs(R - Ro) / np.maximum(np.abs(Ro).max(0, keepdims=True), 1.0))) < 1e-4


@pytest.mark.parametrize("patterns,count_bytes", [("counts", 0), ("counts", 2), ("normalized", 0)])
@pytest.mark.parametrize("I", [1, 37, 300])
def test_pattern_constants_match_fp32(patterns, count_bytes, I):
    """lse_i carries the constant, which FP32 (no centring) does not need."""
    L, S = 24, 420
    print(f"[pattern constants] {patterns} count_bytes={count_bytes} {I} patterns", flush=True)
    truth, coords, masks, K, q, w = problem(L, 2, 300)
    Kp = (emc_amd.normalize_patterns(K, masks[0]) if patterns == "normalized" else K)[:I]
    out = []
    for prec in ("fp32", "bf16x3"):
        with emc_amd.Engine(L, S, I, precision=prec, count_bytes=count_bytes) as e:
            e.setup(q, w, coords, masks[0], Kp, truth)
            e.logl()
            tot = e.normalize_resp()
            out.append((e.get_lse(), tot))
    (a, ta), (b, tb) = out
    scale = np.maximum(np.abs(a), 1.0)
    assert float(np.max(np.abs(a - b) / scale)) < 1e-5  # FP32 logits of about 300 counts: 256-term FP32 sums
    assert abs(tb - b.sum()) <= 1e-12 * np.abs(b).sum()
