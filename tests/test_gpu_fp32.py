"""Precision FP32: the f32 matrix-core tiles and the chi^2 tiles against FP64, and the sparse M-step, which leaves
the zeros out of the dense contraction's chain of fused multiply-adds, against the dense one, bit for bit."""
import numpy as np
import pytest

import emc_amd

pytestmark = pytest.mark.gpu
L = 16


@pytest.fixture(scope="module")
def data():
    truth = emc_amd.synth_model(L, 40, 3.0, 3)
    coords, mask = emc_amd.coords_flat(L), emc_amd.mask_annulus(L, 1.0, 8.0)
    K, _ = emc_amd.synth_patterns(truth, L, coords, mask, 1600, 200.0, 4)
    q, w = emc_amd.rotations(4)
    return dict(truth=truth, coords=coords, mask=mask, K=K, Kn=emc_amd.normalize_patterns(K, mask), q=q, w=w)


def engine(d, S, I, K, **kw):
    e = emc_amd.Engine(L, S, I, precision="fp32", **kw)
    e.setup(d["q"][:S], d["w"][:S], d["coords"], d["mask"], K[:I], d["truth"])
    return e


# one partial tile, ragged edges; 700 x 1,500 and 3,240 x 1,264 take the wide tile, the others the 64 x 64 one
@pytest.mark.parametrize("S,I", [(60, 33), (420, 300), (700, 1500), (3240, 1264)])
@pytest.mark.parametrize("diff,scaling", [("true_poisson", 0), ("poisson", 0), ("poisson", 1)])
def test_fp32_logits_match_fp64(orc, data, S, I, diff, scaling):
    print(f"[fp32] logits {S} x {I} {diff} scaling={scaling}", flush=True)
    d, sigma = data, 0.3
    K = d["K"][:I].astype(np.float64)
    with engine(d, S, I, d["K"], diff=diff, scaling=scaling) as e:
        e.logl(sigma)
        R = e.get_logl()
    W = orc.slices(d["truth"].astype(np.float64), L, d["q"][:S], d["coords"], "trilinear")
    phi = orc.scaling(W, K, d["mask"]) if scaling else None
    phi0 = orc.fluence(W, K, d["mask"]) if diff == "true_poisson" else 1.0
    Ro, _ = orc.logl(W, K, d["mask"], d["w"][:S].astype(np.float64), diff, sigma=sigma, phi0=phi0,
                     **({"phi": phi} if scaling else {}))
    # a chain of 256 FP32 additions, its inputs and the FP32 slices: 1e-5 of a pattern's largest logit, as the other
    # FP32 logit tests
    assert float(np.max(np.abs(R - Ro) / np.maximum(np.abs(Ro).max(0, keepdims=True), 1.0))) < 1e-5


@pytest.mark.parametrize("S,I", [(60, 33), (420, 257), (3240, 1000)])
@pytest.mark.parametrize("patterns", ["K", "Kn"])
@pytest.mark.parametrize("share", [0.0005, 0.3])
def test_fp32_sparse_mstep_is_the_dense_one(data, S, I, patterns, share):
    print(f"[fp32] sparse M-step {S} x {I} {patterns} share={share}", flush=True)
    d = data
    rng = np.random.default_rng(S + I)
    P = (rng.random((S, I)) * (rng.random((S, I)) < share)).astype(np.float32)
    P[0, 0] = 1.0
    P[S - 1, I - 1] = 1e-30
    out = []
    for mstep in ("dense", "sparse", "auto"):
        with engine(d, S, I, d[patterns], mstep=mstep) as e:
            e.set_resp(P)
            e.maximize()
            e.compress()
            out.append(e.get_model())
    for M, W in out[1:]:
        assert np.array_equal(M, out[0][0]) and np.array_equal(W, out[0][1])
