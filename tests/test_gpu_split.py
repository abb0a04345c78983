"""The ES population on the 16-bit matrix instructions with two-part operands (k_pop_split), at the sizes and values where
it can go wrong: minibatches around its 16-slot tiles and its 32- and 64-slot passes, every operand layout of a hidden
layer (7 to 64 units, one and two hidden layers), and models whose values leave the 16-bit range."""
import numpy as np
import pytest

from gpu_common import LAYOUTS, data, rel, say, trainer
from neural_block_textures_amd.trainer import Layout

pytestmark = pytest.mark.gpu

# Outputs are within 2e-6 of the reference's (the bar of the decode; a 32-bit pre-activation of size up to 8 is itself
# within 5e-7). A member's loss is the mean of squared differences d, so it moves by at most 2 sqrt(loss) 2e-6 + (2e-6)^2.
DELTA = 2e-6


def check(orc, lay, z, p, tgt, pairs, batch, sigma=0.02, seed=5):
    tr = trainer(lay, z, p, tgt, max_pairs=pairs, max_batch=batch, seed=seed)
    tr.mlp_step(3, sigma, 0.005, pairs, batch)
    idx = tr.debug_last_batch()
    lp, lm = tr.debug_last_losses()
    _, _, lp_o, lm_o = orc.mlp_es_eval(lay, p, z, tgt, seed, 3, sigma, pairs, idx)
    worst = 0.0
    for got, want in ((lp, lp_o), (lm, lm_o)):
        bound = 2 * np.sqrt(want) * DELTA + DELTA ** 2
        worst = max(worst, float((np.abs(got - want) / bound).max()))
    say("pairs", pairs, "batch", batch, "largest error over its bound", worst)
    assert worst <= 1.0
    tr.close()


@pytest.mark.parametrize("name", ["rgb_16x2", "rgb_24x2", "two_level", "material", "material_clamp", "dct_plane", "large",
                                  "chief1_36", "mat_qat_36", "image3_27", "dct_17", "dct_11", "run8x3", "jit_mfma_28",
                                  "jit_own_13"])
def test_split_population_edges(orc, name):
    lay = LAYOUTS[name]
    z, p, tgt = data(lay, 21)
    say("split edges", name)
    for pairs, batch in ((1, 1), (2, 15), (1, 16), (3, 17), (2, 33), (2, 63), (1, 64), (2, 65), (5, 257), (2, 1000), (40, 300)):
        check(orc, lay, z, p, tgt, pairs, batch)


@pytest.mark.parametrize("hidden,nout", [(16, 1), (48, 1), (24, 3)])
def test_split_population_one_hidden_layer(orc, hidden, nout):
    lay = Layout(40, 24, [(10, 6, 4, False)], [hidden], T=nout, leak=0.1)
    z, p, tgt = data(lay, 22)
    say("split one hidden layer", hidden, nout)
    check(orc, lay, z, p, tgt, 3, 100)


@pytest.mark.parametrize("name", ["rgb_16x2", "material", "material_clamp", "large", "chief1_36", "two_level"])
@pytest.mark.parametrize("scale", [2.0 ** 14, 2.0 ** -14])
def test_split_population_range(orc, name, scale):
    """Latents whose hidden values pass 65504 (the kernel then evaluates its slots in 32 bits), and layers whose sizes are far
    from one another: the first layer's weights and biases scaled, the output layer scaled back, so the outputs are those of
    an ordinary model and the bound is the same."""
    lay = LAYOUTS[name]
    z, p, tgt = data(lay, 23)
    nin, h = lay.nin, lay.hidden[0]
    p = p.copy()
    n1, n2 = h * nin + h, h * nin + h + h * h + h
    p[:n1] *= np.float32(scale)
    p[n1 + h * h:n2] *= np.float32(scale)
    p[n2:n2 + lay.nout * h] *= np.float32(1.0 / scale)
    say("split range", name, scale)
    # sigma follows the smallest layer's scale
    check(orc, lay, z, p, tgt, 3, 200, sigma=0.02 * min(scale, 1.0 / scale))
    if scale > 1:   # large features in place of large weights: the layers' scales cannot take them
        z2, p2 = z * np.float32(scale), data(lay, 23)[1].copy()
        p2[h * nin:n1] *= np.float32(scale)
        p2[n1 + h * h:n2] *= np.float32(scale)
        p2[n2:n2 + lay.nout * h] /= np.float32(scale)
        check(orc, lay, z2, p2, tgt, 3, 200, sigma=0.02 / scale)


def test_split_population_infinite_bias(orc):
    """an infinite output bias saturates its output (main.cpp:624): a finite loss, as the oracle's"""
    lay = LAYOUTS["material"]
    z, p, tgt = data(lay, 24)
    p = p.copy()
    p[-1] = np.inf
    tr = trainer(lay, z, p, tgt, max_pairs=2, max_batch=100)
    tr.mlp_step(1, 0.02, 0.005, 2, 100)
    lp, lm = tr.debug_last_losses()
    _, _, lp_o, lm_o = orc.mlp_es_eval(lay, p, z, tgt, 5, 1, 0.02, 2, tr.debug_last_batch())
    assert np.isfinite(lp_o).all() and rel(lp, lp_o).max() < 1e-5 and rel(lm, lm_o).max() < 1e-5
    tr.close()


@pytest.mark.parametrize("name", ["rgb_16x2", "dct_11", "material", "chief1_36", "jit_mfma_28"])
def test_split_central_differences_edges(orc, name):
    """The central-difference population on the split kernel, which forms its members from the weights itself. A loss
    difference carries the rounding of both losses: as in the full-size check, at most 1e-3 of the differences' RMS, or
    where the minibatch is small (few roundings average out) twice the bound of one loss."""
    lay = LAYOUTS[name]
    z, p, tgt = data(lay, 25)
    h = np.float32(1e-3)
    for batch in (1, 17, 65, 1000):
        tr = trainer(lay, z, p, tgt, max_pairs=4, max_batch=batch)
        tr.mlp_step_fd(2, h, 0.005, batch)
        dl = tr.debug_last_dl()
        dl_o, hh, l0 = orc.mlp_fd_eval(lay, p, z, tgt, h, tr.debug_last_batch())
        rms = np.sqrt((dl_o ** 2).mean())
        worst = np.abs(dl - dl_o).max()
        say("fd", name, "batch", batch, "largest error over the RMS", worst / rms)
        assert worst <= max(1e-3 * rms, 2 * (2 * np.sqrt(l0) * DELTA / np.sqrt(batch) + DELTA ** 2))
        g = tr.debug_last_wgrad()
        assert np.array_equal(g, orc.fd_grad(dl, hh))          # the realized 32-bit steps
        w, m, v = p.copy(), np.zeros_like(p), np.zeros_like(p)
        orc.adam(w, g, m, v, 0.005, 1)
        assert np.array_equal(tr.download_model()[1], w)
        tr.close()


def latent(orc, lay, z, p, tgt, K, sigma=0.05, seed=6):
    """the per-pixel differences of a latent step against the oracle's, at the reference's bar (1e-3 of their RMS)"""
    tr = trainer(lay, z, p, tgt, max_pairs=1, max_batch=16, seed=seed)
    tr.lat_step(1, np.float32(sigma), 0.0, K)
    dpix = tr.debug_last_dpix()
    mask = (1 << len(lay.levels)) - 1
    _, want, _, _ = orc.lat_grad(lay, p, z, z, tgt, seed, 0, np.float32(sigma), K, mask, want_dpix=True)
    rms = np.sqrt((want.astype(np.float64) ** 2).mean())
    say("latent", lay.W, lay.H, "pairs", K, "largest error over the RMS", np.abs(dpix.ravel() - want).max() / rms)
    assert np.abs(dpix.ravel() - want).max() < 1e-3 * rms
    tr.close()


@pytest.mark.parametrize("name", ["rgb_16x2", "two_level", "material", "material_clamp", "dct_17", "chief1_36", "large", "run8x3",
                                  "jit_own_13"])
def test_split_latent_edges(orc, name):
    """image sizes around a wave's 64 pixels and a block's four rounds, one pair and several"""
    base = LAYOUTS[name]
    for W, H, K in ((1, 1, 1), (7, 9, 3), (64, 1, 2), (65, 1, 1), (50, 41, 5), (128, 2, 1)):
        lay = Layout(**{k: getattr(base, k) for k in base.__dataclass_fields__})
        lay.W, lay.H = W, H
        lay.levels = [(max(1, W * w // base.W), max(1, H * h // base.H), c, near) for w, h, c, near in base.levels]
        z, p, tgt = data(lay, 26)
        latent(orc, lay, z, p, tgt, K)


@pytest.mark.parametrize("name", ["rgb_16x2", "material", "material_clamp", "large"])
def test_split_latent_range(orc, name):
    """hidden values past the 16-bit range: the kernel's rounds in 32 bits, on an image of several rounds a wave"""
    lay = LAYOUTS[name]
    z, p, tgt = data(lay, 27)
    nin, h, s = lay.nin, lay.hidden[0], np.float32(2.0 ** 14)
    p = p.copy()
    n1, n2 = h * nin + h, h * nin + h + h * h + h
    p[h * nin:n1] *= s
    p[n1 + h * h:n2] *= s
    p[n2:n2 + lay.nout * h] /= s
    latent(orc, lay, z * s, p, tgt, 3, sigma=0.05 * 2.0 ** 14)


@pytest.mark.parametrize("name", ["material", "material_clamp", "chief1_36", "mat_qat_36", "image3_27", "jit_mfma_28", "dct_plane"])
@pytest.mark.parametrize("scale", [1.0, 2.0 ** 14])
def test_split_selector_search(orc, name, scale):
    """the selector search on the split kernel against the oracle's, over image sizes around a wave's 64 pixels, on ordinary
    models and on ones whose hidden values pass the 16-bit range (large features of the other level): the same choices, but for
    texels whose candidates' losses agree to 1e-6 (main.cpp:3143-3144)"""
    from neural_block_textures_amd import synth
    base = LAYOUTS[name]
    for W, H in ((1, 1), (63, 1), (65, 3), (52, 41)):
        lay = Layout(**{k: getattr(base, k) for k in base.__dataclass_fields__})
        lay.W, lay.H = W, H
        lay.levels = [(W, H, base.levels[0][2], True)] + [(max(1, W * w // base.W), max(1, H * h // base.H), c, near)
                                                          for w, h, c, near in base.levels[1:]]
        z, p, tgt = data(lay, 28)
        grid, C0 = synth.qat_grid(), lay.levels[0][2]
        bits = [2 + (c % 2) for c in range(C0)]
        n0 = W * H * C0
        lv0 = z[:n0].reshape(-1, C0)
        for c in range(C0):
            lv0[:, c] = synth.qat_snap(lv0[:, c], bits[c], grid)
        if scale != 1.0:
            nin, h, s = lay.nin, lay.hidden[0], np.float32(scale)
            z[n0:] *= s
            n1, n2 = h * nin + h, h * nin + h + h * h + h
            w1 = p[:h * nin].reshape(h, nin)
            w1[:, :C0] *= s                      # the searched inputs keep their share of the first layer
            p[h * nin:n1] *= s
            p[n1 + h * h:n2] *= s
            p[n2:n2 + lay.nout * h] /= s
        tr = trainer(lay, z, p, tgt, qat_bits=bits, qat_grid=grid)
        tr.qat_search()
        zg, zc = tr.download_model()[0], z.copy()
        orc.qat_search(lay, p, zc, tgt, bits, grid)
        assert np.array_equal(zg[n0:], z[n0:])
        diff = np.nonzero((zg[:n0] != zc[:n0]).reshape(-1, C0).any(1))[0]
        say("selectors", name, W, H, "scale", scale, "differ", diff.size, "of", W * H)
        if diff.size:
            ec, eg = orc.decode_err(lay, p, zc, tgt), orc.decode_err(lay, p, zg, tgt)
            assert (np.abs(ec[diff] - eg[diff]) <= 1e-6 * np.maximum(ec[diff], eg[diff]) + 1e-12).all()
        tr.close()


@pytest.mark.parametrize("name", ["rgb_16x2", "two_level", "material", "material_clamp", "chief1_36", "large"])
def test_latent_pairs_on_the_32_bit_instructions(orc, monkeypatch, name):
    """the same latent steps with NTC_HIP_POP_PAIR=0 (k_lat_pair_mfma on the listed shapes), at the same bar"""
    monkeypatch.setenv("NTC_HIP_POP_PAIR", "0")
    base = LAYOUTS[name]
    for W, H, K in ((1, 1, 1), (65, 1, 1), (50, 41, 5)):
        lay = Layout(**{k: getattr(base, k) for k in base.__dataclass_fields__})
        lay.W, lay.H = W, H
        lay.levels = [(max(1, W * w // base.W), max(1, H * h // base.H), c, near) for w, h, c, near in base.levels]
        z, p, tgt = data(lay, 26)
        latent(orc, lay, z, p, tgt, K)


@pytest.mark.parametrize("T", [1, 4])
def test_selector_search_one_hidden_layer(orc, T):
    """one hidden layer: at most 4 outputs on k_qat_mfma, more on k_qat_split; the oracle's choices but for ties"""
    from neural_block_textures_amd import synth
    lay = Layout(65, 21, [(65, 21, 2, True), (17, 6, 4, False)], [32], T=T, leak=0.01)
    z, p, tgt = data(lay, 30)
    grid, bits, n0 = synth.qat_grid(), [2, 3], 65 * 21 * 2
    for c in range(2):
        z[:n0].reshape(-1, 2)[:, c] = synth.qat_snap(z[:n0].reshape(-1, 2)[:, c], bits[c], grid)
    tr = trainer(lay, z, p, tgt, qat_bits=bits, qat_grid=grid)
    tr.qat_search()
    zg, zc = tr.download_model()[0], z.copy()
    tr.close()
    orc.qat_search(lay, p, zc, tgt, bits, grid)
    assert np.array_equal(zg[n0:], z[n0:])
    diff = np.nonzero((zg[:n0] != zc[:n0]).reshape(-1, 2).any(1))[0]
    say("selectors, one hidden layer", T, "differ", diff.size)
    ec, eg = orc.decode_err(lay, p, zc, tgt), orc.decode_err(lay, p, zg, tgt)
    assert (np.abs(ec[diff] - eg[diff]) <= 1e-6 * np.maximum(ec[diff], eg[diff]) + 1e-12).all()


def test_split_population_past_32_bit_offsets():
    """a minibatch whose split arrays pass 4 GiB (9 to 12 inputs: 67 million slots) evaluates on the 32-bit kernel, whose rows
    still fit. The oracle would take minutes over its slots: the members are the weights themselves (sigma 0), and their loss is
    the mean of the pixels' losses within five of its standard deviations."""
    lay = Layout(16, 16, [(4, 4, 4, False), (2, 2, 4, False)], [36, 36], T=4, leak=0.01)
    z, p, tgt = data(lay, 31)
    for M, split in ((1 << 20, True), (68 << 20, False)):
        tr = trainer(lay, z, p, tgt, max_pairs=1, max_batch=M)
        assert tr.on_matrix_cores("pop_eval") and tr.on_matrix_cores("pop_split") == split
        say("split sizes", M)
        d = (tr.decode_full().astype(np.float64) - tgt).reshape(-1, lay.nout)
        tr.mlp_step(1, 0.0, 0.0, 1, M)
        loss = tr.mlp_stats()[0]
        tr.close()
        e = (d * d).sum(1) / (3.0 * lay.T)
        assert abs(loss - e.mean()) <= 5 * e.std() / np.sqrt(M) + 1e-6 * e.mean()


@pytest.mark.parametrize("hidden,leak", [([23, 23], 0.03), ([29], 0.0)])
def test_specialised_shapes_compile_one_population(orc, monkeypatch, tmp_path, hidden, leak):
    """a shape compiled at init holds the population kernels its trainer launches and no others: k_pop_split's, or with
    NTC_HIP_POP_PAIR=0 k_pop_mfma's (the three of both take a third longer to compile); one process runs both"""
    monkeypatch.setenv("NTC_HIP_JIT_CACHE", str(tmp_path))
    lay = Layout(40, 24, [(10, 6, 4, False)], hidden, T=4, leak=leak)
    z, p, tgt = data(lay, 32)
    for env, kernel, other in ((None, "k_pop_split", "k_pop_mfma"), ("0", "k_pop_mfma", "k_pop_split")):
        if env:
            monkeypatch.setenv("NTC_HIP_POP_PAIR", env)
        old = set(tmp_path.glob("*.names"))
        for pairs, batch in ((3, 100), (2, 1200)):
            check(orc, lay, z, p, tgt, pairs, batch)
        names = "".join(f.read_text() for f in set(tmp_path.glob("*.names")) - old)
        assert names.count(kernel) == 3 and other not in names
        tr = trainer(lay, z, p, tgt, max_pairs=4, max_batch=100)
        tr.mlp_step_fd(1, 1e-3, 0.0, 100)
        tr.close()
