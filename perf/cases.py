"""Performance cases of the EMC engine: what a reconstruction program has it do, over the range of its use.

A case is a dict of plain values.  Kinds:

  iterate   a context that holds its rotations, detector, patterns and a formed model runs one EMC
            iteration and reads the model back (the loop of a reconstruction; likelihood, precision,
            interpolation and pattern type as given);
  stages    the same iteration through the stage calls (likelihood, responsibilities, maximize,
            compress), as a program drives them that does something of its own between the stages;
  proposal  an iteration whose search is restricted by the learned orientation proposal (prediction,
            grouped search, refresh training of the network);
  compress  the allocation-free compress on device buffers of a caller (divide by weight, normalise, blur).

Data are synthetic, made from the seed: Gaussian atoms, flat- or Ewald-detector slices at random
orientations, Poisson counts.  The starting model is the true one with every voxel off by up to 20 %, which is
what an iteration sees for most of a reconstruction (sharp posteriors), and it keeps the outputs of
an iteration a smooth function of its inputs.
"""
import math

import numpy as np
import torch

import emc_amd
from emc_amd import _lib

ITERATION = 30          # the iteration index of every pass: late in the annealing schedule
SIGMA = (0.4, 0.12, 25)  # start, final, half life (the engine's defaults)

_BASE = dict(kind="iterate", diff="true_poisson", interp="trilinear", precision="bf16x2", insert="binned",
             scaling=0, chunk=0, blur=0.5, detector="flat", patterns="counts")


def _case(name, **kw):
    c = dict(_BASE, **kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # a quick look at a few patterns on a coarse grid: launches and latency are all there is
        _case("poisson_24_tiny", L=24, n=2, I=64, photons=800.0),
        # the small complete workload (32^3, 3,240 rotations, 1,000 patterns)
        _case("poisson_32", L=32, n=4, I=1000, photons=2000.0),
        # the benchmark's workload (64^3, 25,680 rotations, 20,000 patterns of 5,000 photons)
        _case("poisson_64_full", L=64, n=8, I=20000, photons=5000.0),
        # a large model with few photons per pattern, an odd pattern count
        _case("poisson_128_sparse", L=128, n=5, I=3001, photons=300.0),
        # the reference's own likelihood (chi^2 with per-pattern scaling) on the matrix cores
        _case("chi2_scaled_64", L=64, n=5, I=4000, photons=5000.0, diff="poisson", scaling=1),
        # the same in plain FP32, as the reference computes it
        _case("chi2_scaled_48_fp32", L=48, n=4, I=1500, photons=3000.0, diff="poisson", scaling=1, precision="fp32"),
        # plain FP32 Poisson likelihood, the setting to check the other precisions with
        _case("poisson_64_fp32", L=64, n=5, I=4001, photons=5000.0, precision="fp32"),
        # normalised (non-integer) patterns, which the matrix cores take as two terms
        _case("normalized_64", L=64, n=5, I=3000, photons=5000.0, patterns="normalized"),
        # stage calls, nearest-voxel slicing, three-term split, Ewald detector, rotations in chunks, odd sizes
        _case("stages_45_nearest", kind="stages", L=45, n=4, I=777, photons=2500.0, precision="bf16x3",
              interp="nearest", detector="ewald", chunk=1000),
        # learned proposal: 10,860 rotations in 420 cells
        _case("proposal_64", kind="proposal", L=64, n=6, I=4000, photons=5000.0, coarse_n=2),
        # compress alone on a caller's device buffers: a large model, and a small odd one in a serving loop
        dict(name="compress_128", kind="compress", L=128, blur=0.5),
        dict(name="compress_41", kind="compress", L=41, blur=0.7),
    ]


def _loguniform(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    kind = rng.choice(["iterate"] * 7 + ["stages", "proposal", "compress"])
    if kind == "compress":
        return dict(kind="compress", L=_loguniform(rng, 20, 128), blur=round(rng.uniform(0.4, 1.0), 2))
    L = _loguniform(rng, 20, 100)
    n = rng.randint(2, 6)
    I = _loguniform(rng, 48, max(96, min(5000, 2.4e7 / (L * L))))
    c = _case(None, kind=kind, L=L, n=n, I=I, photons=round(math.exp(rng.uniform(math.log(300.0), math.log(5000.0)))),
              blur=rng.choice([0.0, 0.5]), interp=rng.choice(["trilinear", "trilinear", "nearest"]),
              detector=rng.choice(["flat", "ewald"]))
    if kind == "proposal":
        c.update(n=max(4, n), I=max(256, I), interp="trilinear", coarse_n=rng.choice([1, 2]))
        return c
    c["precision"] = rng.choice(["bf16x2", "bf16x2", "bf16x3", "fp32"])
    c["patterns"] = rng.choice(["counts", "counts", "normalized"])
    c["diff"] = rng.choice(["true_poisson", "true_poisson", "poisson", "absolute"])
    if c["diff"] != "true_poisson":
        c["scaling"] = rng.choice([0, 1])
        if not c["scaling"]:  # a known intensity: the patterns are normalised
            c["patterns"] = "normalized"
    if rng.random() < 0.25:
        c["chunk"] = rng.randint(200, 2500)
    return c


# ---- inputs -------------------------------------------------------------------------------------

def _inputs(case, seed):
    """Host arrays of a case: rotations, detector, mask, patterns and the starting model."""
    L, I = case["L"], case["I"]
    truth = emc_amd.synth_model(L, 3 * L, 0.19 * L, 10 * seed + 1)
    if case["detector"] == "ewald":
        coords = emc_amd.coords_ewald(L, 75.0e-6 * 64 / L, 0.74, 1.03e-9)
    else:
        coords = emc_amd.coords_flat(L)
    mask = emc_amd.mask_annulus(L, L / 16.0, L / 2.0)
    K, _ = emc_amd.synth_patterns(truth, L, coords, mask, I, case["photons"], 10 * seed + 2)
    if case["patterns"] == "normalized":
        K = emc_amd.normalize_patterns(K, mask)
    q, w = emc_amd.rotations(case["n"])
    rng = np.random.default_rng(seed)
    model = truth * rng.uniform(0.8, 1.2, truth.shape).astype(np.float32)
    if case["diff"] != "true_poisson" and not case["scaling"]:  # these kinds compare the model with the counts
        model *= np.float32(K[:, mask != 0].mean() / truth[truth > 0].mean())
    else:
        model /= np.float32(model[model > 0].mean(dtype=np.float64))
    return q, w, coords, mask, K, model


def _sums(case, seed, device):
    """Insertion sums of a compress: voxels in the corners never hit, some hit without counts."""
    L = case["L"]
    g = torch.Generator(device="cpu").manual_seed(seed)
    ax = torch.arange(L) - (L - 1) / 2
    r2 = (ax[:, None, None] ** 2 + ax[None, :, None] ** 2 + ax[None, None, :] ** 2).reshape(-1)
    weight = torch.rand(L ** 3, generator=g) * 3.0 * (r2 <= (L / 2) ** 2)
    numerator = torch.rand(L ** 3, generator=g) * 2.0 * weight * (torch.rand(L ** 3, generator=g) > 0.05)
    return numerator.to(device), weight.to(device)


def _sigma(it):
    return float(np.float32(SIGMA[1] + (SIGMA[0] - SIGMA[1]) * math.exp(-it / SIGMA[2] * math.log(2.0))))


def prepare(case, seed):
    if case["kind"] == "compress":
        numerator, weight = _sums(case, seed, "cuda")
        return dict(case=case, numerator=numerator, weight=weight, model=torch.empty_like(weight),
                    avg=torch.zeros(1, dtype=torch.float64, device="cuda"))
    q, w, coords, mask, K, model = _inputs(case, seed)
    eng = emc_amd.Engine(case["L"], q.shape[0], case["I"], slice_chunk=case["chunk"], diff=case["diff"],
                         interp=case["interp"], precision=case["precision"], insert=case["insert"],
                         scaling=case["scaling"], blur_sigma=case["blur"])
    eng.setup(q, w, coords, mask, K, model)
    if case["kind"] == "proposal":
        # one full search trains the network; every pass after it is a proposal iteration
        eng.enable_proposal(emc_amd.rotations(case["coarse_n"])[0], warmup_full=1, full_every=1 << 30, min_mass=0.0)
        eng.iterate(0)
    return dict(case=case, eng=eng)


def run(state):
    case = state["case"]
    if case["kind"] == "compress":
        _lib.check(_lib.lib().emc_compress_device(case["L"], case["blur"], state["numerator"].data_ptr(),
                                                  state["weight"].data_ptr(), state["model"].data_ptr(),
                                                  state["avg"].data_ptr(), torch.cuda.current_stream().cuda_stream))
        return {"model": state["model"], "avg": state["avg"]}
    eng = state["eng"]
    if case["kind"] == "stages":
        eng.logl(_sigma(ITERATION))
        total = eng.normalize_resp()
        eng.maximize()
        avg = eng.compress()
    else:
        st = eng.iterate(ITERATION)
        total, avg = st["total_logl"], st["model_avg"]
    model, weight = eng.get_model()
    return {"model": model, "weight": weight, "total_logl": total, "model_avg": avg}


def work(case):
    L = case["L"]
    if case["kind"] == "compress":  # two sums read, the model written; three axes of L taps per voxel
        return {"bytes": 12.0 * L ** 3, "flops": 6.0 * L ** 4}
    S, I = 10.0 * (5 * case["n"] ** 3 + case["n"]), float(case["I"])
    Pa = math.pi * L * L * (1 / 4 - 1 / 256)
    # every (rotation, pattern) pair is scored once over the pixels (the proposal scores the patterns'
    # own cells alone: 16 of the coarse grid's, of which there are 60 or 420)
    share = 1.0
    if case["kind"] == "proposal":
        share = min(1.0, 16.0 / (10.0 * (5 * case["coarse_n"] ** 3 + case["coarse_n"])))
    sums = 1.0
    if case["diff"] != "true_poisson":  # sum a W K and sum a K^2; with scaling also sum K^2 and sum W K
        sums = 4.0 if case["scaling"] else 2.0
    count_bytes = 4.0 if case["precision"] == "fp32" or case["patterns"] != "counts" else 1.0
    # the counts, the pairs of insertion (voxel and fractions follow from the rotation) and the model
    return {"bytes": I * Pa * count_bytes + 12.0 * L ** 3, "flops": share * sums * 2.0 * S * I * Pa + 60.0 * S * Pa}


# ---- the same outputs in 64 bits ----------------------------------------------------------------

def _fma(a, b, c):
    """float32 fma(a, b, c) of float32 values held in float64 (the product is exact there)."""
    return (a * b + c).float().double()


def _rotmats(q):
    q0, q1, q2, q3 = (q[:, k] for k in range(4))
    f = lambda x: x.float().double()  # noqa: E731
    m = [_fma(q0, q0, _fma(q1, q1, _fma(-q2, q2, -f(q3 * q3)))), 2 * _fma(q1, q2, -f(q0 * q3)), 2 * _fma(q1, q3, f(q0 * q2)),
         2 * _fma(q1, q2, f(q0 * q3)), _fma(q0, q0, _fma(-q1, q1, _fma(q2, q2, -f(q3 * q3)))), 2 * _fma(q2, q3, -f(q0 * q1)),
         2 * _fma(q1, q3, -f(q0 * q2)), 2 * _fma(q2, q3, f(q0 * q1)), _fma(q0, q0, _fma(-q1, q1, _fma(-q2, q2, f(q3 * q3))))]
    return [x[:, None] for x in m]


def _points(m, xyz, L):
    """Grid coordinates of the detector points under the rotations m, in the float32 steps that fix every voxel index."""
    X, Y, Z = (a[None, :] for a in xyz)
    c = 0.5 * L - 0.5
    return [(c + _fma(m[3 * r], X, _fma(m[3 * r + 1], Y, (m[3 * r + 2] * Z).float().double()))).float().double() for r in range(3)]


def _corners(u, L, interp, slicing):
    """(valid, [(voxel index, weight)]) of the points; the nearest voxel's lower bound is open when slicing."""
    if interp == "nearest":
        v = [torch.sign(a) * torch.floor(a.abs() + 0.5) for a in u]
        lo = 1 if slicing else 0
        ok = torch.ones_like(u[0], dtype=torch.bool)
        for a in v:
            ok &= (a >= lo) & (a < L)
        x, y, z = (torch.where(ok, a, 0.0).long() for a in v)
        return ok, [((z * L + y) * L + x, torch.ones_like(u[0]))]
    ok = torch.ones_like(u[0], dtype=torch.bool)
    for a in u:
        ok &= (a >= 0) & (a <= L - 1)
    b = [torch.where(ok, torch.clamp(torch.floor(a), max=L - 2), 0.0) for a in u]
    f = [torch.where(ok, a - i, 0.0) for a, i in zip(u, b)]
    x, y, z = (a.long() for a in b)
    out = []
    for dz in (0, 1):
        for dy in (0, 1):
            for dx in (0, 1):
                wgt = (f[0] if dx else 1 - f[0]) * (f[1] if dy else 1 - f[1]) * (f[2] if dz else 1 - f[2])
                out.append((((z + dz) * L + y + dy) * L + x + dx, wgt))
    return ok, out


def _blur(model, L, sigma):
    k = torch.arange(L, dtype=torch.float64, device=model.device)
    h = torch.exp(-2.0 * math.pi ** 2 * sigma ** 2 * torch.minimum(k, L - k) ** 2 / L ** 2)
    field = torch.fft.fftn(torch.clamp(model, min=0.0).reshape(L, L, L))
    out = torch.fft.ifftn(field * h[:, None, None] * h[None, :, None] * h[None, None, :]).real.reshape(-1)
    return torch.where(model < 0, model, out)


def _compress(num, weight, L, blur):
    hit = weight > 0
    model = torch.where(hit, num / torch.where(hit, weight, 1.0), -1.0)
    avg = model[hit].mean()
    model = model / avg
    return (_blur(model, L, blur) if blur > 0 else model), avg


def exact(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    f64 = dict(dtype=torch.float64, device=dev)
    if case["kind"] == "compress":
        num, weight = _sums(case, seed, dev)
        model, avg = _compress(num.double(), weight.double(), case["L"], case["blur"])
        return {"model": model, "avg": avg.reshape(1)}
    q, w, coords, mask, K, model = _inputs(case, seed)
    L, S, I = case["L"], q.shape[0], case["I"]
    act = torch.as_tensor(np.flatnonzero(mask), device=dev)
    xyz = [torch.as_tensor(c, **f64)[act] for c in coords]
    K = torch.as_tensor(K.reshape(I, -1), device=dev)[:, act].double()
    q, logw = torch.as_tensor(q, **f64), torch.log(torch.as_tensor(w, **f64))
    model = torch.as_tensor(model, **f64)
    step = max(1, int(4e6 // act.numel()))
    poisson, scaled = case["diff"] == "true_poisson", bool(case["scaling"])
    for it in ([0] if case["kind"] == "proposal" else []) + [ITERATION]:
        R = torch.empty(S, I, **f64)
        ip = torch.ones(S, I, **f64) if scaled else None
        sumW = torch.zeros(S, **f64)
        sigma = _sigma(it)
        for s0 in range(0, S, step):
            s = slice(s0, min(S, s0 + step))
            ok, corners = _corners(_points(_rotmats(q[s]), xyz, L), L, case["interp"], True)
            W = torch.zeros_like(corners[0][1])
            for v, wgt in corners:
                W += wgt * model[v]
                ok &= model[v] >= 0
            ok &= W > 0
            W = torch.where(ok, W, 0.0)
            sumW[s] = W.sum(1)
            if poisson:  # without the fluence, which follows from all rotations
                R[s] = torch.log(torch.where(ok, W, 1.0)) @ K.T
                if s0 == 0:
                    valid = torch.empty(S, I, **f64)
                valid[s] = ok.double() @ K.T
                continue
            a = {"poisson": 1.0 / (W + 0.02), "absolute": torch.ones_like(W)}[case["diff"]] * ok
            D2 = a @ (K * K).T
            D1 = (a * W) @ K.T
            D0 = (a * W * W).sum(1, keepdim=True)
            if scaled:
                inn = (W > 1e-10).double()
                kk, kw = inn @ (K * K).T, (W * inn) @ K.T
                ip[s] = torch.where((kk > 0) & (kw > 0), kw / torch.where(kk > 0, kk, 1.0), 1.0)
                D = D0 - 2 * ip[s] * D1 + ip[s] ** 2 * D2
            else:
                D = D0 - 2 * D1 + D2
            n = ok.sum(1, keepdim=True).double()
            R[s] = logw[s, None] - torch.where(n > 0, D / (2 * sigma ** 2 * torch.clamp(n, min=1.0)), 0.0)
        if poisson:
            phi = (K.sum() / I) / (sumW.sum() / S)
            R += logw[:, None] + math.log(float(phi)) * valid - phi * sumW[:, None]
        lse = torch.logsumexp(R, 0)
        P = torch.exp(R - lse[None, :])
        T = P.sum(1)
        if scaled:
            P = P * ip
        del R, ip
        num, weight = torch.zeros(L ** 3, **f64), torch.zeros(L ** 3, **f64)
        for s0 in range(0, S, step):
            s = slice(s0, min(S, s0 + step))
            U = P[s] @ K
            ok, corners = _corners(_points(_rotmats(q[s]), xyz, L), L, case["interp"], False)
            ok &= (T[s] > 1e-10)[:, None]
            Ts = T[s][:, None].expand_as(U)
            for v, wgt in corners:
                wgt = torch.where(ok, wgt, 0.0)
                num.index_add_(0, v.reshape(-1), (wgt * U).reshape(-1))
                weight.index_add_(0, v.reshape(-1), (wgt * Ts).reshape(-1))
        del P
        model, avg = _compress(num, weight, L, case["blur"])
    return {"model": model, "weight": weight, "total_logl": float(lse.sum()), "model_avg": float(avg)}
