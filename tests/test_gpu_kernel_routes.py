"""Forms of the contraction kernels that only larger shapes reach, each named by the tile its shape is given: the
register-staged kernels (mfma_staging = 1), the left-out and packed logit stores of the 256 x 256 tile and the left-out ones
of the others, and the 256 x 320 tile over a whole number of its columns."""
import numpy as np
import pytest

import emc_amd
from tile_route import logl_tile, pad, tile

pytestmark = pytest.mark.gpu
L = 24


@pytest.fixture(scope="module")
def data():
    truth = emc_amd.synth_model(L, 60, 4.5, 3)
    coords, mask = emc_amd.coords_flat(L), emc_amd.mask_annulus(L, 2.0, 12.0)
    K, _ = emc_amd.synth_patterns(truth, L, coords, mask, 4000, 900.0, 4)
    K = np.minimum(K, 255)
    rng = np.random.default_rng(7)
    model = (truth * rng.uniform(0.7, 1.3, truth.shape)).astype(np.float32)
    q, w = emc_amd.rotations(6)  # 10,860
    return dict(truth=truth, model=model, coords=coords, mask=mask, K=K, Kn=emc_amd.normalize_patterns(K, mask), q=q, w=w)


def setup(e, d, S, I, Kp, model):
    e.setup(d["q"][:S], d["w"][:S], d["coords"], d["mask"], Kp[:I], model)


@pytest.mark.parametrize("S,I,prec,route", [(6300, 1000, "bf16x2", "256x128"), (6300, 2001, "bf16x2", "256x256"),
                                            (6300, 3000, "bf16x2", "256x320"), (6300, 2001, "bf16x3", "256x256")])
@pytest.mark.parametrize("count_bytes", [0, 2])
def test_register_staging_equals_dma_staging_logits(data, S, I, prec, route, count_bytes):
    print(f"[staging] logits {S} x {I} {prec} count_bytes={count_bytes}", flush=True)
    assert logl_tile(S, I, prec, False) == route
    out = []
    for st in (0, 1):
        with emc_amd.Engine(L, S, I, precision=prec, mfma_staging=st, count_bytes=count_bytes) as e:
            setup(e, data, S, I, data["K"], data["model"])
            e.logl()
            R = e.get_logl()
            e.normalize_resp()
            out.append((R, e.get_lse(), e.get_slice_weights()))
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("chunk", [0, 4000])
@pytest.mark.parametrize("top", [16, 255])  # counts to 16: their squares are one term, so sum K^2 has one term each side
@pytest.mark.parametrize("prec", ["bf16x2", "bf16x3"])
def test_register_staging_equals_dma_staging_chi2(data, prec, top, chunk):
    S, I = 6300, 2001
    print(f"[staging] chi^2 {S} x {I} {prec} counts to {top} chunk {chunk}", flush=True)
    na = 3 if prec == "bf16x3" else 2
    for n in (na, 1):  # the register-staged kernels take the place of 256-row tiles alone
        assert tile(pad(chunk or S, 256), pad(I, 256), n, 1) == ("256x128" if chunk else "256x256")
    out = []
    for st in (0, 1):
        with emc_amd.Engine(L, S, I, precision=prec, diff="poisson", scaling=1, mfma_staging=st, slice_chunk=chunk) as e:
            setup(e, data, S, I, np.minimum(data["K"], top), data["model"])
            e.logl(0.3)
            R = e.get_logl()
            e.normalize_resp()
            out.append((R, e.get_lse()))
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("count_bytes", [0, 2])
@pytest.mark.parametrize("side,columns,route", [(58, 2688, "256x320"), (52, 2176, "256x256")])
def test_register_staging_equals_dma_staging_mstep(side, columns, route, count_bytes):
    S, I = 6300, 96  # both column counts end with half a 256-wide tile
    print(f"[staging] M-step {S} x {columns} pixels, count_bytes={count_bytes}", flush=True)
    truth = emc_amd.synth_model(side, 60, 0.19 * side, 3)
    coords, mask = emc_amd.coords_flat(side), emc_amd.mask_annulus(side, 2.0, side / 2)
    assert pad(int(mask.sum()), 128) == columns and columns % 256 == 128
    assert tile(pad(S, 256), columns, 2, 1) == route
    K, _ = emc_amd.synth_patterns(truth, side, coords, mask, I, 400.0, 4)
    q, w = emc_amd.rotations(5)
    P = np.random.default_rng(1).random((S, I)).astype(np.float32)
    out = []
    for st in (0, 1):
        with emc_amd.Engine(side, S, I, mfma_staging=st, mstep="dense", count_bytes=count_bytes) as e:
            e.setup(q, w, coords, mask, np.minimum(K, 255), truth)
            e.set_resp(P)
            e.maximize()
            e.compress()
            out.append(e.get_model())
    for a, b in zip(*out):
        assert np.array_equal(a, b)


# chunks, so that the later ones meet the earlier ones' maxima; ragged rows and columns, and whole columns
@pytest.mark.parametrize("I,chunk,route", [(2300, 5000, "256x256"), (2304, 5000, "256x256"), (2301, 6000, "256x256"),
                                           (1500, 5000, "256x128"), (3700, 5000, "256x320"), (2500, 3240, "128x128")])
def test_left_out_stores_leave_the_iteration_unchanged(data, I, chunk, route):
    S = 10860
    print(f"[left-out stores] {S} x {I} chunk {chunk} {route}", flush=True)
    assert logl_tile(S, I, "bf16x2", False, chunk) == route
    out, skipped = [], []
    for keep in (1, 0):
        with emc_amd.Engine(L, S, I, blur_sigma=0.5, slice_chunk=chunk, keep_logits=keep) as e:
            setup(e, data, S, I, data["K"], data["model"])
            st = [e.iterate(it) for it in range(3)]
            out.append((np.array([s["total_logl"] for s in st]), *e.get_model(), e.get_lse(), e.get_resp(),
                        e.get_slice_weights()))
            skipped.append([s["logits_skipped"] for s in st])
    print(f"   left out per iteration: {skipped[1]}", flush=True)
    assert skipped[0] == [0.0] * 3 and min(skipped[1]) > 0.0
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("inner,columns", [(6.0, 3200), (2.0, 2688)])  # ten tiles of 320 columns; a ragged last one
def test_wide_tile_mstep(split, inner, columns):
    side = 64 if columns == 3200 else 58
    S, I = 6300, 96
    print(f"[wide tile] M-step {S} x {columns} split={split}", flush=True)
    truth = emc_amd.synth_model(side, 60, 0.19 * side, 3)
    coords, mask = emc_amd.coords_flat(side), emc_amd.mask_annulus(side, inner, side / 2)
    assert pad(int(mask.sum()), 128) == columns and tile(pad(S, 256), columns, 2, 2 if split else 1) == "256x320"
    K, _ = emc_amd.synth_patterns(truth, side, coords, mask, I, 400.0, 4)
    K = np.minimum(K, 255)
    q, w = emc_amd.rotations(5)
    P = np.random.default_rng(1).random((S, I)).astype(np.float32)
    out = []
    for t in (0, 1):
        with emc_amd.Engine(side, S, I, mfma_tile=t, mstep="dense") as e:
            e.setup(q, w, coords, mask, emc_amd.normalize_patterns(K, mask) if split else K, truth)
            e.set_resp(P)
            e.maximize()
            e.compress()
            out.append(e.get_model())
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("split", [False, True])
def test_wide_tile_over_whole_columns(data, split):
    S, I = 5000, 3840  # twelve tiles of 320 columns
    print(f"[wide tile] {S} x {I} split={split}", flush=True)
    assert logl_tile(S, I, "bf16x2", split) == "256x320" and pad(I, 256) % 320 == 0
    out = []
    for t in (0, 1):
        with emc_amd.Engine(L, S, I, mfma_tile=t) as e:
            setup(e, data, S, I, data["Kn" if split else "K"], data["model"])
            e.logl()
            out.append(e.get_logl())
    assert np.array_equal(*out)
