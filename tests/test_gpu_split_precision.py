"""The split kernels (k_pop_split, k_lat_split: 32-bit operands in 16-bit parts) against the 32-bit matrix kernels they stand
in for (NTC_HIP_POP_PAIR=0): each side's error from 64-bit sums over the same 32-bit weights, latents and features, on
ordinary models and on ones where 16-bit parts could lose bits: small latents, weights far larger than their layer's
others, layers of very different sizes."""
import numpy as np
import pytest

from gpu_common import LAYOUTS, data, say, trainer
from neural_block_textures_amd.trainer import PK_UV, Layout
from test_gpu_split import check, latent

pytestmark = pytest.mark.gpu

MODELS = {
    "rgb_16x2": LAYOUTS["rgb_16x2"], "two_level": LAYOUTS["two_level"], "material": LAYOUTS["material"], "large": LAYOUTS["large"],
    "mat_qat_36": LAYOUTS["mat_qat_36"], "chief1_36": LAYOUTS["chief1_36"], "dct_17": LAYOUTS["dct_17"], "run8x3": LAYOUTS["run8x3"],
    "jit_mfma_28": LAYOUTS["jit_mfma_28"],
    # five hidden values a lane and 9 inputs; one hidden layer
    "rgb_20": Layout(64, 48, [(16, 12, 4, False), (8, 6, 3, False)], [20, 20], leak=0.01),
    "one_24": Layout(40, 24, [(10, 6, 4, False)], [24], T=3, pos=[PK_UV], leak=0.1),
}


def model(name, regime, seed):
    lay = MODELS[name]
    z, p, tgt = data(lay, seed, zscale=0.01 if regime == "small" else 0.4)
    nin, h, o, cuts = lay.nin, lay.hidden[0], 0, []
    for n in (*lay.hidden, lay.nout):
        k = nin if not cuts else h
        cuts.append((o, o + n * k, o + n * k + n))
        o += n * k + n
    p = p.copy()
    if regime == "small":      # latents of 0.01 whose first-layer weights are as much larger
        p[:h * nin].reshape(h, nin)[:, :nin - 2 * len(lay.pos)] *= np.float32(16.0)
    elif regime == "outlier":  # one weight a layer far above the others
        for a, b, _ in cuts:
            p[a + 1 + (b - a) // 3] = np.float32(12.0)
    elif regime == "outlier_dead":   # ... and far more so, into a unit that is off (leak 0)
        a, b, c = cuts[0]
        p[a:a + nin] = np.float32(3e4)
        p[b] = np.float32(-1e6)
    elif regime == "wide":
        for a, b, _ in cuts[:-1]:
            p[a:b] *= np.float32(3.0)
    return lay, z, p, tgt


def losses64(lay, f, t, sets):
    """[members, slots] losses in 64 bits of the weight sets (64-bit values) over the slots' features f [nin, n] and targets"""
    cw, wsum = lay.loss_weights()
    leak, out = float(np.float32(lay.leak)), []
    for s in np.array_split(sets, max(1, len(sets) * max(lay.hidden) * f.shape[1] >> 24)):
        x, o, k = f, 0, lay.nin
        for l, n in enumerate([*lay.hidden, lay.nout]):
            x = s[:, o:o + n * k].reshape(-1, n, k) @ x + s[:, o + n * k:o + n * k + n, None]
            o, k = o + n * k + n, n
            x = 1.0 / (1.0 + np.exp(-x)) if l == len(lay.hidden) else np.where(x > 0, x, x * leak)
        out.append((((x - t) ** 2) * np.array(cw[:lay.nout])[:, None]).sum(1))
    return np.concatenate(out) / (3.0 * wsum)


def population_errors(orc, monkeypatch, name, regime, path, seeds, batch):
    """[split, 32-bit]: the loss differences' relative error from 64 bits (2-norm, RMS over the seeds)"""
    pairs, sigma, h = 48, np.float32(0.02), np.float32(1e-3)
    sq = np.zeros(2)
    for seed in range(seeds):
        lay, z, p, tgt = model(name, regime, 70 + seed)
        got = []
        for env in (None, "0"):
            (monkeypatch.delenv("NTC_HIP_POP_PAIR", raising=False) if env is None else monkeypatch.setenv("NTC_HIP_POP_PAIR", env))
            tr = trainer(lay, z, p, tgt, max_pairs=pairs, max_batch=batch, seed=seed)
            assert tr.on_matrix_cores("pop_split") == (env is None)
            if path == "es":
                tr.mlp_step(1, sigma, 0.0, pairs, batch)
            else:
                tr.mlp_step_fd(1, h, 0.0, batch)
            got.append(tr.debug_last_dl())
            idx = tr.debug_last_batch()
            tr.close()
        f = np.stack([orc.features(lay, z, int(i) % lay.W, int(i) // lay.W) for i in idx], 1).astype(np.float64)
        t, w = tgt.reshape(-1, lay.nout)[idx].T.astype(np.float64), p.astype(np.float64)
        if path == "es":
            eps = np.stack([orc.gauss_fill(seed, 2, 1, i, 0, p.size) for i in range(pairs)]).astype(np.float64)
            plus, minus = w + float(sigma) * eps, w - float(sigma) * eps
        else:   # the weights a step takes are 32-bit
            plus, minus = (w + np.diag(a.astype(np.float64) - w) for a in (p + h, p - h))
        want = losses64(lay, f, t, plus).mean(1) - losses64(lay, f, t, minus).mean(1)
        for k in range(2):
            sq[k] += np.sum((got[k] - want) ** 2) / np.sum(want ** 2)
    e = np.sqrt(sq / seeds)
    say(path, name, regime, "batch", batch, "error split %.3e 32-bit %.3e ratio %.3f" % (e[0], e[1], e[0] / e[1]))
    return e


REGIMES = ["plain", "small", "outlier", "wide", "outlier_dead"]


def cases(names):
    return [(n, r) for n in sorted(names) for r in REGIMES if r != "outlier_dead" or MODELS[n].leak == 0.0]


# The members' roundings are independent: 192 loss differences give each error to 5% and the ratio of two to 7%. Measured 0.38 to
# 0.97 (with the weights in two parts up to 1.75).
@pytest.mark.parametrize("name,regime", cases(MODELS))
def test_population_no_further_from_64_bits(orc, monkeypatch, name, regime):
    split, full = population_errors(orc, monkeypatch, name, regime, "es", 4, 1500)
    assert split <= 1.1 * full


# Thousands of differences each. Measured 0.81 to 1.02.
@pytest.mark.parametrize("name,regime", cases(["rgb_16x2", "two_level", "material", "chief1_36", "jit_mfma_28", "one_24"]))
def test_central_differences_no_further_from_64_bits(orc, monkeypatch, name, regime):
    split, full = population_errors(orc, monkeypatch, name, regime, "fd", 2, 1500)
    assert split <= 1.1 * full


def latent_errors(orc, monkeypatch, name, regime, seeds, K=4):
    sq = np.zeros(2)
    for seed in range(seeds):
        lay, z, p, tgt = model(name, regime, 80 + seed)
        sigma = np.float32(0.001 if regime == "small" else 0.05)
        got = []
        for env in (None, "0"):
            (monkeypatch.delenv("NTC_HIP_POP_PAIR", raising=False) if env is None else monkeypatch.setenv("NTC_HIP_POP_PAIR", env))
            tr = trainer(lay, z, p, tgt, max_pairs=1, max_batch=16, seed=seed)
            tr.lat_step(1, sigma, 0.0, K)
            got.append(tr.debug_last_dpix().reshape(K, -1))
            tr.close()
        t, w = tgt.reshape(-1, lay.nout).T.astype(np.float64), p.astype(np.float64)[None]
        for k in range(K):
            eps = orc.gauss_fill(seed, 1, 0, k, 0, lay.nz).astype(np.float64)
            e = []
            for s in (float(sigma), -float(sigma)):
                zz = (z + s * eps).astype(np.float32)   # one rounding, as a fused operation
                f = np.stack([orc.features(lay, zz, x, y) for y in range(lay.H) for x in range(lay.W)], 1).astype(np.float64)
                e.append(losses64(lay, f, t, w)[0])
            want = (e[0] - e[1]) / (lay.W * lay.H)
            for q in range(2):
                sq[q] += np.sum((got[q][k] - want) ** 2) / np.sum(want ** 2)
    e = np.sqrt(sq / (seeds * K))
    say("latent", name, regime, "error split %.3e 32-bit %.3e ratio %.3f" % (e[0], e[1], e[0] / e[1]))
    return e


# Measured 0.68 to 1.0; 1.13 for the 16-wide model of large weights, whose 32-bit sums round few times where its hidden values
# have 22 bits. (A shape compiled at init has no 32-bit latent pair kernel beside the split one.)
@pytest.mark.parametrize("name,regime", cases(n for n in MODELS if n not in ("jit_mfma_28", "rgb_20", "one_24")))
def test_latent_pairs_no_further_from_64_bits(orc, monkeypatch, name, regime):
    split, full = latent_errors(orc, monkeypatch, name, regime, 1)
    assert split <= (1.2 if regime == "wide" else 1.1) * full


@pytest.mark.parametrize("name", ["rgb_16x2", "material", "material_clamp", "large", "chief1_36"])
@pytest.mark.parametrize("e1,e2", [(50, 0), (-50, 0), (40, -60), (-70, 45)])
def test_layers_of_very_different_sizes(orc, name, e1, e2):
    """hidden layers times 2^e1 and 2^e2 and the output layer back: no power of two in the kernels' range fits such a layer, so
    they evaluate in 32 bits, from the 32-bit weights; the outputs and the bounds are an ordinary model's"""
    lay = LAYOUTS[name]
    z, p, tgt = data(lay, 29)
    nin, h = lay.nin, lay.hidden[0]
    n1, n2 = h * nin + h, h * nin + h + h * h + h
    p = p.copy()
    p[:n1] *= np.float32(2.0 ** e1)
    p[n1:n1 + h * h] *= np.float32(2.0 ** e2)
    p[n1 + h * h:n2] *= np.float32(2.0 ** (e1 + e2))
    p[n2:n2 + lay.nout * h] *= np.float32(2.0 ** -(e1 + e2))
    say("far layers", name, e1, e2)
    check(orc, lay, z, p, tgt, 3, 200, sigma=0.02 * 2.0 ** min(e1, e2, e1 + e2, -(e1 + e2)))
    for batch in (40, 700):     # one chunk, which draws the Gaussians itself, and two
        check(orc, lay, z, p, tgt, 2100, batch, sigma=0.02 * 2.0 ** min(e1, e2, e1 + e2, -(e1 + e2)))
    latent(orc, lay, z, p, tgt, 2)
