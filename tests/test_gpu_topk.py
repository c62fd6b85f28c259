"""The cells a prediction keeps and the mass they hold, against numpy: a network whose last layer is its bias alone gives
every pattern the same known probabilities (ties among them); cell counts below and above one wavefront's registers."""
import numpy as np
import pytest

import emc_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("coarse,k,recall", [(1, 1, 0), (1, 60, 3), (2, 8, 8), (2, 64, 1), (3, 8, 8)])  # 60, 420, 1,380 cells
def test_predicted_cells_and_mass(coarse, k, recall):
    print(f"[topk] coarse {coarse} k {k} recall {recall}", flush=True)
    L, I = 24, 97
    truth = emc_amd.synth_model(L, 60, 4.5, 3)
    coords, mask = emc_amd.coords_flat(L), emc_amd.mask_annulus(L, 2.0, 12.0)
    K, _ = emc_amd.synth_patterns(truth, L, coords, mask, I, 400.0, 4)
    q, w = emc_amd.rotations(4)  # 3,240
    cq = emc_amd.rotations(coarse)[0]
    rng = np.random.default_rng(coarse * 100 + k)
    with emc_amd.Engine(L, q.shape[0], I) as e:
        e.setup(q, w, coords, mask, np.minimum(K, 255), truth)
        e.enable_proposal(cq, top_k=k, recall=recall, warmup_full=1, epochs=1, hidden=64, batch=64)
        e.iterate(0)
        W1, b1, W2, b2, W3, b3 = e.mlp_params()
        b3 = rng.integers(-6, 7, b3.shape).astype(np.float32)  # many ties
        e.set_mlp_params(W1, b1, W2, b2, np.zeros_like(W3), b3)
        p = e.mlp_forward(np.zeros((1, 1024), np.float32))[0]
        cells, mass = e.proposal_predict()
        rec = e.proposal_recall() if recall else np.zeros((I, 0), np.int32)
    order = np.argsort(-p, kind="stable")[:k]
    assert np.array_equal(cells, np.tile(np.sort(order), (I, 1)))
    if recall:
        assert (rec >= 0).any()
    for i in range(I):
        want = np.float32(0.0)
        for c in list(order) + [c for c in rec[i] if c >= 0 and c not in order]:
            want += p[c]
        assert mass[i] == want  # the same float32 sums, in the same order
