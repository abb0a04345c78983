"""The latent gradient's footprint gather in its three forms (a thread per texel, runs from memory, rows through LDS) against
the oracle's scatter of the device's own differences: the same sums bit for bit, over footprints up to the whole image,
texels that no pixel reads, and numbers of pairs around its waves of four."""
import numpy as np
import pytest

from gpu_common import data, say, trainer
from neural_block_textures_amd.trainer import Layout

pytestmark = pytest.mark.gpu

CASES = {
    # rectangles of several LDS steps a row (700 columns), and of every column
    "wide_700": Layout(700, 21, [(2, 3, 8, False), (1, 1, 4, False)], [32, 32], leak=0.0),
    # 16 and 64 pixels a texel, texels of a row over several tiles
    "wide_512": Layout(512, 40, [(32, 3, 8, False), (8, 2, 4, False)], [32, 32], leak=0.0),
    # ragged ratios on either side of 16 columns, nearest
    "ragged": Layout(331, 37, [(37, 5, 8, False), (19, 7, 4, True)], [32, 32], leak=0.0),
    # levels finer than the image: texels that no pixel reads
    "fine": Layout(33, 27, [(90, 70, 8, False), (40, 80, 4, True)], [32, 32], leak=0.0),
    # one pixel per texel, beside a bilinear level
    "unit": Layout(70, 45, [(70, 45, 1, True), (18, 12, 4, False)], [32, 32], leak=0.01),
    "unit2": Layout(61, 33, [(61, 33, 2, True), (4, 3, 4, False)], [32, 32], T=4, leak=0.01),
}


@pytest.mark.parametrize("name", sorted(CASES))
@pytest.mark.parametrize("K,group", [(1, 0), (4, 0), (5, 0), (15, 0), (17, 0), (9, 4)])
def test_gather_same_sums(orc, name, K, group):
    lay = CASES[name]
    z, p, tgt = data(lay, 41)
    seed, sigma, lr = 8, np.float32(0.05), 0.02
    tr = trainer(lay, z, p, tgt, max_pairs=1, max_batch=16, seed=seed)
    mask = (1 << len(lay.levels)) - 1
    zz, m, v = z.copy(), np.zeros_like(z), np.zeros_like(z)
    for step in (0, 1):   # the second step's Gaussians are drawn by the first one's gather
        tr.lat_step(step + 1, sigma, lr, K)
        g = tr.debug_last_zgrad()
        dpix = tr.debug_last_dpix()
        if group == 0:
            eps = np.concatenate([orc.gauss_fill(seed, 1, step, k, 0, lay.nz) for k in range(K)])
            assert np.array_equal(g, orc.lat_scatter(lay, eps, dpix, K, mask, sigma))
        orc.adam(zz, g, m, v, lr, step + 1)
        assert np.array_equal(tr.download_model()[0], zz)
    say("gather", name, K)
    if group:   # in groups of pairs, the same gradient
        got = []
        for n in (0, group):
            t2 = trainer(lay, z, p, tgt, max_pairs=1, max_batch=16, seed=seed)
            t2.set_lat_group(n)
            t2.lat_step(1, sigma, lr, K)
            got.append(t2.debug_last_zgrad())
            t2.close()
        assert np.array_equal(got[0], got[1])
    tr.close()
