"""The contraction's tiles (64 x 64, 128 x 128, 256 x 128, 256 x 256, chosen by the shape) against the
128 x 128 register-staged kernel (mfma_tile = 1): every tile adds an element's products in the same order,
so logits and the dense M-step are equal bit for bit; only the two-launch form of three-term slices with
two-term counts adds the low counts' products last."""
import numpy as np
import pytest

import emc_amd

pytestmark = pytest.mark.gpu
L = 24


@pytest.fixture(scope="module")
def data():
    truth = emc_amd.synth_model(L, 60, 4.5, 3)
    coords, mask = emc_amd.coords_flat(L), emc_amd.mask_annulus(L, 2.0, 12.0)
    K, _ = emc_amd.synth_patterns(truth, L, coords, mask, 3000, 400.0, 4)
    K = np.minimum(K, 255)
    q, w = emc_amd.rotations(5)  # 6,300
    return dict(truth=truth, coords=coords, mask=mask, K=K, Kn=emc_amd.normalize_patterns(K, mask), q=q, w=w)


def run(d, S, I, prec, split, **kw):
    with emc_amd.Engine(L, S, I, precision=prec, mstep="dense", **kw) as e:
        e.setup(d["q"][:S], d["w"][:S], d["coords"], d["mask"], (d["Kn"] if split else d["K"])[:I], d["truth"])
        e.logl()
        R = e.get_logl()
        e.normalize_resp()
        lse = e.get_lse()
        e.maximize()
        e.compress()
        return R, lse, e.get_model()[0]


# edges of the tiles: one partial 64 x 64 tile, ragged rows and columns, then shapes for each larger tile
@pytest.mark.parametrize("S,I", [(70, 65), (1000, 300), (3240, 700), (6300, 1000), (6300, 2001), (6300, 3000)])
@pytest.mark.parametrize("prec,split", [("bf16x2", False), ("bf16x2", True), ("bf16x3", False), ("bf16x3", True)])
def test_tiles_equal_the_register_staged_kernel(data, S, I, prec, split):
    print(f"[tiles] {S} x {I} {prec} split={split}", flush=True)
    a = run(data, S, I, prec, split)
    b = run(data, S, I, prec, split, mfma_tile=1)
    if prec == "bf16x3" and split:
        # the low counts' products, at most 2^-8 of the others, are added last: a few FP32 roundings apart
        scale = np.abs(b[0]).max(0, keepdims=True)
        assert float(np.max(np.abs(a[0] - b[0]) / scale)) < 2e-6
    else:
        assert np.array_equal(a[0], b[0])
    assert np.allclose(a[1], b[1], rtol=2e-6, atol=0)  # band sums on exp2 in FP32 lanes against expf
    assert np.allclose(a[2], b[2], rtol=1e-4, atol=1e-6)
